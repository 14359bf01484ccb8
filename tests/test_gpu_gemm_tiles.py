"""k_gemm_big's four tiles (128 x 128, 128 x 192, 256 x 192, 256 x 256) at
ragged row counts and k-step counts that are not a multiple of its ring, each
epilogue fc_gemm offers, and the QKV projection on its 128 x 128 tile."""

import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
from flaxchat_amd._lib import check, lib  # noqa: E402

pytestmark = pytest.mark.gpu


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _pack(t):
    R, K = t.shape
    out = torch.empty((R + 15) // 16 * 16, K, dtype=t.dtype, device="cuda")
    check(lib().fc_pack_operand(t.data_ptr(), out.data_ptr(), R, K, _stream()), "pack")
    return out


# the smallest row counts past 512 tiles of 64 x 64 and ragged ones; K / 32 = 2,
# 6, 10 (ring remainders 2), 24 and 192; K = 4 N from 48 tiles of 64 x 64 an XCD; and a
# wide output with 1, 33 and 129 rows in the second 256-row tile
@pytest.mark.parametrize("M,N,K", [(2753, 768, 64), (2753, 768, 192), (3000, 768, 320), (4111, 1152, 768),
                                   (16385, 128, 64), (3056, 1536, 768), (6000, 1536, 3072), (8191, 2048, 1536),
                                   (1025, 16384, 128), (961, 1536, 6144), (1473, 768, 3072), (257, 32768, 64),
                                   (289, 32768, 64), (385, 32768, 64)])
@pytest.mark.parametrize("epi", [0, 1, 2, 4])
def test_large_tiles(M, N, K, epi):
    print(f"M={M} N={N} K={K} epi={epi}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda", generator=g) * 0.05).to(torch.bfloat16)
    a, b = _pack(x), _pack(w)
    ref = x.double() @ w.double().t()
    # fp32 accumulation of K products: 2^-24 per add on a sum of size |x||w| sqrt(K)
    tol = 2.0 ** -24 * K * 0.05 * 3
    if epi == 2:
        out = torch.zeros((M + 15) // 16 * 16, N, device="cuda", dtype=torch.bfloat16)
    elif epi == 1:
        base = torch.randn(M, N, device="cuda", generator=g)
        out = base.clone()
    else:
        out = torch.full((M + 1, N), 7.0, device="cuda")
    check(lib().fc_gemm(a.data_ptr(), b.data_ptr(), out.data_ptr(), M, N, K, 1, epi, _stream()), "fc_gemm")
    if epi == 0:
        assert float((out[:M] - ref).abs().max()) <= tol and bool((out[M] == 7.0).all())
    elif epi == 1:
        assert float((out - (ref + base)).abs().max()) <= tol + 2.0 ** -21
    elif epi == 4:
        # the bf16 kernels' softcap is within 5e-6 of 15 tanh(z / 15)
        assert float((out[:M] - 15 * torch.tanh(ref / 15)).abs().max()) <= tol + 1e-5 and bool((out[M] == 7.0).all())
    else:
        from flaxchat_amd.torch_ops import frag_to_rows
        got, want = frag_to_rows(out, M).double(), torch.relu(ref) ** 2
        assert bool(((got - want).abs() <= want * 2.0 ** -8 + 2 * tol * ref.abs() + 1e-6).all())


@pytest.mark.parametrize("M,D,kv", [(1000, 1536, 12), (1301, 1536, 4), (2050, 768, 6)])
def test_qkv_tile_matches_the_separate_prologue(M, D, kv):
    """fc_attn_qkv's fused tile against the plain GEMM and fc_attn_prologue:
    the same q and cache to one bf16 ulp (different order of the sums)."""
    import flaxchat_amd.torch_ops  # noqa: F401
    from flaxchat_amd.config import GPTConfig
    from flaxchat_amd.runtime import DeviceCache, DeviceModel
    ops = torch.ops.flaxchat_mi355x
    print(f"M={M} D={D} kv={kv}", flush=True)
    cfg = GPTConfig(sequence_len=512, vocab_size=1000, n_layer=2, n_head=D // 128, n_kv_head=kv, n_embd=D)
    dm = DeviceModel.random_init(cfg, seed=1, dtype="bf16")
    B, per = 4, (M + 3) // 4
    g = torch.Generator(device="cuda").manual_seed(M)
    tok = torch.randint(0, 1000, (M,), device="cuda", dtype=torch.int32, generator=g)
    i = torch.arange(M, device="cuda")
    row, pos = (i // per).int(), (i % per).int()
    row[5] = -1                                   # skipped token
    h = torch.randn((M + 15) // 16 * 16, D, device="cuda", generator=g).to(torch.bfloat16)
    addr = ctypes.addressof(dm.desc)
    got, want = DeviceCache(dm, B, per + 32), DeviceCache(dm, B, per + 32)
    for layer in (0, 1):                          # without and with a value embedding
        assert lib().fc_attn_qkv_workspace_bytes(ctypes.byref(dm.desc), M, 0) == 0
        q = ops.attn_qkv(addr, layer, got.k, got.v, h, tok, row, pos)
        qkv = torch.empty(M, (dm.H + 2 * dm.G) * 128, device="cuda")
        check(lib().fc_gemm(h.data_ptr(), dm.t["layers"][layer]["wqkv"].data_ptr(), qkv.data_ptr(), M, qkv.shape[1],
                            D, 1, 0, _stream()), "fc_gemm")
        q2 = ops.attn_prologue(addr, layer, want.k, want.v, qkv, h, tok, row, pos)
        keep = np.arange(M) != 5
        np.testing.assert_allclose(q.float().cpu().numpy()[keep], q2.float().cpu().numpy()[keep], rtol=2.0 ** -7,
                                   atol=2.0 ** -9)
    for a, b in ((got.k, want.k), (got.v, want.v)):
        np.testing.assert_allclose(a.float().cpu().numpy(), b.float().cpu().numpy(), rtol=2.0 ** -7, atol=2.0 ** -9)


# rows past 832 with an n_embd whose MLP c_proj (K 3072, 6144) splits K on the large tiles; 720 rows,
# where c_fc keeps the folded norm (n_embd 768) or takes the large tiles without it (1536)
@pytest.mark.parametrize("B,q,D,kv", [(93, 9, 768, 6), (119, 7, 768, 6), (128, 9, 1536, 4), (80, 9, 768, 6),
                                      (80, 9, 1536, 4)])
def test_split_residual_gemm_in_a_chunk(B, q, D, kv):
    """A chunk against its rows in batches below those row counts (other GEMM
    kernels): the same logits up to bf16 operand rounding."""
    import flaxchat_amd.torch_ops  # noqa: F401
    from flaxchat_amd.config import GPTConfig
    from flaxchat_amd.runtime import DeviceCache, DeviceModel
    print(f"B={B} q={q} D={D}", flush=True)
    cfg = GPTConfig(sequence_len=512, vocab_size=1000, n_layer=2, n_head=D // 128, n_kv_head=kv, n_embd=D)
    dm = DeviceModel.random_init(cfg, seed=2, dtype="bf16")
    rng = np.random.default_rng(B)
    tok = rng.integers(0, 1000, (B, q)).astype(np.int32)

    def forward(t):
        n = len(t)
        cache = DeviceCache(dm, n, 64)
        off = torch.arange(0, n * q + 1, q, dtype=torch.int32, device="cuda")
        logits = torch.zeros(n, q, dm.V, device="cuda")
        nb = lib().fc_forward_workspace_bytes(ctypes.byref(dm.desc), n, n * q, q, 0)
        ws = torch.zeros(nb, device="cuda", dtype=torch.uint8)
        torch.ops.flaxchat_mi355x.forward(ctypes.addressof(dm.desc), cache.k, cache.v, cache.hist,
                                          torch.from_numpy(t.reshape(-1).copy()).cuda(), off,
                                          torch.zeros(n, dtype=torch.int32, device="cuda"), q, q, logits, ws)
        return logits.double()

    got = forward(tok)
    want = torch.cat([forward(tok[i:i + 32]) for i in range(0, B, 32)])
    # bf16 operands (2^-9 each) through 2 layers: each side is within about 0.3% of float64
    assert float((got - want).norm() / want.norm()) <= 0.012


# the lm_head's kernels: K-split (5 rows), LDS-shared (32, 150), large tiles (256; 1100)
@pytest.mark.parametrize("M", [5, 32, 150, 256, 1100])
def test_softcap_is_odd_and_as_exact_on_both_sides(M):
    """15 tanh(z / 15) of the bf16 kernels against float64 on the same sums z: the same
    error for negative logits as for positive ones."""
    N, K = 16384, 64
    print(f"M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    w = torch.randn(N, K, device="cuda", generator=g).to(torch.bfloat16)
    b = _pack(w)

    def logits(rows, epi):
        out = torch.empty(M, N, device="cuda")
        check(lib().fc_gemm(_pack(rows).data_ptr(), b.data_ptr(), out.data_ptr(), M, N, K, 1, epi, _stream()), "fc_gemm")
        return out

    z, y = logits(x, 0), logits(x, 4)
    same = logits(-x, 0) == -z  # all but a few: the matrix cores' own rounding is not the same on both sides
    assert float(same.float().mean()) > 0.9 and torch.equal(logits(-x, 4)[same], -y[same])
    err = (y.double() - 15 * torch.tanh(z.double() / 15))[z < -1]
    # 15 - 30 r, r in (0, 0.47), e = exp2(t), t in (0.19, 7): the last rounding 2^-21, the
    # reciprocal's ulp 30 x 2^-25, e + 1 and e to 2^-24 and 2^-23 of themselves (30 r 2^-24, 30 r (1 - r) 2^-23),
    # t to 2 x 2^-24 (30 r (1 - r) t ln 2 2^-23): 3.9e-6 at most, 0.6e-6 as uniform errors at r = 0.2
    assert float(err.square().mean().sqrt()) <= 0.7e-6 and float(err.abs().max()) <= 4e-6
