"""The fp32 matrix-core kernels: k_gemm_f32's three tilings (64 x 64; 32 x 32 with
K over four or eight waves) at ragged rows, columns and K tails, and k_gemv on
either side of them, every epilogue of fc_gemm, against float64; and fp32
attention over ragged rows, GQA, windows and key counts around its 32-key
tiles. Their error must not exceed what sequential fp32 sums would show."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")
import flaxchat_amd.torch_ops  # noqa: E402,F401
from flaxchat_amd._lib import check, lib  # noqa: E402

pytestmark = pytest.mark.gpu


# k_gemv: 9 rows. Four waves: up to 9 chunks of 32 k, whose last one has 8. Eight waves (K of 512
# and more, up to 256 tiles): 17, 24 and 25 chunks, where some waves have one fewer, an odd number
# of rounds and a last chunk of 8 among them. 64 x 64: an even and an odd number of chunks.
@pytest.mark.parametrize("M,N,K", [(9, 40, 8), (33, 100, 24), (9, 96, 72), (100, 768, 256), (64, 33, 1024),
                                   (200, 768, 3072), (65, 768, 3072), (1000, 8192, 256), (1543, 1600, 104),
                                   (17, 40, 8), (40, 96, 72), (100, 768, 264), (33, 300, 520), (100, 768, 768),
                                   (100, 768, 776), (1543, 1600, 72)])
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


@pytest.mark.parametrize("H,G,n,start,window", [
    (2, 2, [1, 1, 1], [0, 31, 500], 0), (2, 2, [33, 0, 7], [0, 0, 300], 100), (6, 2, [5, 64], [63, 10], 0),
    (12, 4, [1, 9], [1000, 0], 0), (2, 2, [500, 499], [0, 0], 256), (4, 1, [3], [40], 8)])
def test_fp32_attention(H, G, n, start, window):
    print(f"H={H} G={G} n={n} start={start} window={window}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(len(n) + H)
    B, cap = len(n), (max(a + b for a, b in zip(n, start)) + 31) // 32 * 32
    off = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    q = torch.randn(int(off[-1]), H, 128, device="cuda", generator=g) * 2
    k = torch.randn(B, G, cap, 128, device="cuda", generator=g)
    v = torch.randn(B, G, cap, 128, device="cuda", generator=g)
    vb = v.view(B, G, cap // 32, 32, 128).transpose(3, 4).contiguous()
    got = torch.ops.flaxchat_mi355x.attention(q, k, vb, torch.from_numpy(off).cuda(),
                                              torch.tensor(start, dtype=torch.int32, device="cuda"), max(n), window)
    rep = H // G
    for b in range(B):
        if n[b] == 0:
            continue
        end = start[b] + n[b]
        qb = q[off[b]:off[b + 1]].double().transpose(0, 1)
        kb, vv = (t[b, :, :end].double().repeat_interleave(rep, 0) for t in (k, v))
        pos = torch.arange(start[b], end, device="cuda")[:, None]
        key = torch.arange(end, device="cuda")[None]
        see = (key <= pos) & ((pos - key <= window) if window > 0 else True)
        s = (torch.matmul(qb, kb.transpose(1, 2).contiguous()) / np.sqrt(128)).masked_fill(~see, -np.inf)
        want = torch.matmul(torch.softmax(s, -1), vv).transpose(0, 1).reshape(n[b], -1)
        # scores of up to ~12 from 128 products (two chains of 64 / 2): ~8 roundings, through exp
        # as a relative error; at most 64 rescalings and 32-key sums
        err = float((got[off[b]:off[b + 1]] - want).abs().max())
        assert err <= 100 * 2.0 ** -24 * 4, err


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


def test_fp32_attention_unseen_keys():
    """Keys a query does not see, past the row's end, after it or left of its window, do not
    reach it even where their K and V are infinite or NaN; the queries that see one do get it."""
    g = torch.Generator(device="cuda").manual_seed(1)
    n, start, window, cap = 40, 50, 20, 128
    q = torch.randn(n, 2, 128, device="cuda", generator=g)
    k = torch.randn(1, 2, cap, 128, device="cuda", generator=g)
    v = torch.randn(1, 2, cap, 128, device="cuda", generator=g)
    off, st = torch.tensor([0, n], dtype=torch.int32).cuda(), torch.tensor([start], dtype=torch.int32).cuda()

    def run():
        vb = v.view(1, 2, cap // 32, 32, 128).transpose(3, 4).contiguous()
        return torch.ops.flaxchat_mi355x.attention(q, k, vb, off, st, n, window)

    clean = run().clone()
    k[:, :, start + n:], v[:, :, start + n:] = float("nan"), float("nan")
    k[:, :, :start - window], v[:, :, :start - window] = float("nan"), float("inf")
    v[:, 1, start + 20] = float("inf")  # seen by queries 20 .. 39 of head 1 (window 20: up to 40)
    got = run()
    seen = torch.zeros(n, 2, 128, dtype=torch.bool, device="cuda")
    seen[20:, 1] = True
    seen = seen.view(n, -1)
    assert bool(torch.isinf(got[seen]).all())
    # the same terms by FMA instead of by the matrix cores: a few roundings
    assert float((got - clean)[~seen].abs().max()) <= 64 * 2.0 ** -24


@pytest.mark.parametrize("n,start", [([5, 4], [-3, -50]), ([40], [-20])])
def test_fp32_attention_without_a_key(n, start):
    """A query before position 0 sees no key: it gives 0, and the others of its row what they see."""
    print(f"n={n} start={start}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(2)
    B, tot = len(n), sum(n)
    q = torch.randn(tot, 2, 128, device="cuda", generator=g)
    k = torch.randn(B, 2, 64, 128, device="cuda", generator=g)
    v = torch.randn(B, 2, 64, 128, device="cuda", generator=g)
    off = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    got = torch.ops.flaxchat_mi355x.attention(q, k, v.view(B, 2, 2, 32, 128).transpose(3, 4).contiguous(),
                                              torch.from_numpy(off).cuda(),
                                              torch.tensor(start, dtype=torch.int32, device="cuda"), max(n), 0)
    for b in range(B):
        for j in range(n[b]):
            end, out = max(0, start[b] + j + 1), got[off[b] + j].view(2, 128)
            if end == 0:
                assert bool((out == 0).all())
                continue
            s = (k[b, :, :end].double() * q[off[b] + j][:, None].double()).sum(-1) / np.sqrt(128)
            want = (torch.softmax(s, -1)[..., None] * v[b, :, :end].double()).sum(1)
            # scores of up to ~6 from 128 products, through exp; at most 20 keys
            assert float((out - want).abs().max()) <= 50 * 2.0 ** -24 * 4


@pytest.mark.parametrize("n,start,window,cap", [([40], [40], 0, 64), ([5, 70], [64, 30], 0, 96), ([64], [50], 20, 96)])
def test_fp32_attention_past_the_cache(n, start, window, cap):
    """A position past the cache's end sees what the cache's last position sees."""
    print(f"n={n} start={start} window={window} cap={cap}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    B, tot = len(n), sum(n)
    q = torch.randn(tot, 2, 128, device="cuda", generator=g)
    k = torch.randn(B, 2, cap, 128, device="cuda", generator=g)
    v = torch.randn(B, 2, cap, 128, device="cuda", generator=g)
    off = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    got = torch.ops.flaxchat_mi355x.attention(q, k, v.view(B, 2, cap // 32, 32, 128).transpose(3, 4).contiguous(),
                                              torch.from_numpy(off).cuda(),
                                              torch.tensor(start, dtype=torch.int32, device="cuda"), max(n), window)
    for b in range(B):
        pos = torch.arange(start[b], start[b] + n[b], device="cuda").clamp(max=cap - 1)[:, None]
        key = torch.arange(cap, device="cuda")[None]
        see = (key <= pos) & ((pos - key <= window) if window > 0 else True)
        qb = q[off[b]:off[b + 1]].double().transpose(0, 1)
        s = (torch.matmul(qb, k[b].double().transpose(1, 2).contiguous()) / np.sqrt(128)).masked_fill(~see, -np.inf)
        want = torch.matmul(torch.softmax(s, -1), v[b].double()).transpose(0, 1).reshape(n[b], -1)
        # as above: scores of up to ~6, through exp; three tiles
        assert float((got[off[b]:off[b + 1]] - want).abs().max()) <= 100 * 2.0 ** -24 * 4
