"""The fp32 matrix-core kernels: k_gemm_f32's two tilings at ragged rows,
columns and K tails, every epilogue of fc_gemm, against float64. The error must
not exceed what sequential fp32 sums would show."""
import pytest

torch = pytest.importorskip("torch")
from flaxchat_amd._lib import check, lib  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(9, 40, 8), (33, 100, 24), (9, 96, 72), (100, 768, 256), (64, 33, 1024),
                                   (200, 768, 3072), (65, 768, 3072), (1000, 8192, 256), (1543, 1600, 104)])
@pytest.mark.parametrize("epi", [0, 1, 2, 4])
def test_fp32_gemm(M, N, K, epi):
    print(f"M={M} N={N} K={K} epi={epi}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, device="cuda", generator=g)
    w = torch.randn(N, K, device="cuda", generator=g) * 0.1
    z = x.double() @ w.double().t()
    out = torch.full((M + 1, N), 7.0, device="cuda")
    base = torch.randn(M, N, device="cuda", generator=g)
    if epi == 1:
        out[:M] = base
    check(lib().fc_gemm(x.data_ptr(), w.data_ptr(), out.data_ptr(), M, N, K, 0, epi,
                        torch.cuda.current_stream().cuda_stream), "fc_gemm")
    want = {0: z, 1: z + base, 2: torch.relu(z) ** 2, 4: 15 * torch.tanh(z / 15)}[epi]
    assert bool((out[M] == 7.0).all())
    err = float((out[:M] - want).norm() / want.norm())
    # eight-product chains, two levels of pairs, compensated after that, and the
    # epilogue's own roundings: below 4 roundings of 2^-24 in the 2-norm
    assert err <= 4 * 2.0 ** -24, err


@pytest.mark.parametrize("M,N,K", [(33, 100, 24), (1000, 8192, 256)])
def test_fp32_gemm_infinities(M, N, K):
    """An overflowing or infinite sum is infinite, as a plain sum is; other outputs are untouched."""
    print(f"M={M} N={N} K={K}", flush=True)
    x = torch.ones(M, K, device="cuda")
    w = torch.ones(N, K, device="cuda")
    x[1, 3] = float("inf")
    x[2, 5] = float("nan")
    x[3] = 3e38
    w[N - 1, 3] = -1.0
    out = torch.empty(M, N, device="cuda")
    check(lib().fc_gemm(x.data_ptr(), w.data_ptr(), out.data_ptr(), M, N, K, 0, 0,
                        torch.cuda.current_stream().cuda_stream), "fc_gemm")
    want = torch.full((M, N), float(K), device="cuda")
    want[:, N - 1] -= 2
    want[1], want[2], want[3] = float("inf"), float("nan"), float("inf")
    want[1, N - 1] = -float("inf")
    assert bool(torch.equal(torch.nan_to_num(out, 1e4, 2e4, -2e4), torch.nan_to_num(want, 1e4, 2e4, -2e4)))
