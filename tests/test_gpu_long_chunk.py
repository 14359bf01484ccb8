"""Chunks longer than 32 tokens per row take the token-parallel embedding;
the same tokens fed in pieces of at most 32 take the one-workgroup-per-row
embedding. Both must leave the same smear history and the same first-layer keys
and values (one layer), and, where the second layer mixes x0 in again, the same
second-layer keys and values and the same logits of every row's last token."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,dtype", [(128, "fp32"), (24, "fp32"), (256, "bf16"), (1536, "bf16")])
@pytest.mark.parametrize("full", [0, 1])
def test_long_chunk_embedding_matches_short_pieces(D, dtype, full):
    from flaxchat_amd import _lib
    from flaxchat_amd.config import GPTConfig
    from flaxchat_amd.runtime import DeviceCache, DeviceModel, Workspace, forward_packed, pack_rows
    print(f"D={D} {dtype} full={full}", flush=True)
    H = max(1, D // 128)
    cfg = GPTConfig(sequence_len=512, vocab_size=300, n_layer=1, n_head=H, n_kv_head=H, n_embd=D, window_pattern="L")
    dm = DeviceModel.random_init(cfg, seed=3, dtype=dtype, std=0.3)
    dm.desc.smear_lambda = 0.7
    rng = np.random.default_rng(D)
    lens, first = [200, 0, 33, 1, 65, 64], [0, 0, 5, 0, 2, 0]
    rows = [rng.integers(0, 300, f + n).tolist() for n, f in zip(lens, first)]
    B = len(rows)
    ws = Workspace(dm.device)

    def feed(cache, pieces, starts, logits=None):
        tok, off, mpr = pack_rows(pieces)
        up = lambda a: torch.from_numpy(np.asarray(a, np.int32)).to(dm.device)  # noqa: E731
        forward_packed(dm, cache, up(tok), up(off), up(starts), mpr, 1 if logits is not None else 0, logits, ws,
                       flags=_lib.FC_CHUNK_FULL_SMEAR if full else 0)

    caches = []
    for step in (1024, 32):
        cache = DeviceCache(dm, B, 256)
        feed(cache, [r[:f] for r, f in zip(rows, first)], [0] * B)   # rows that start past position 0
        for c0 in range(0, 200, step):
            feed(cache, [r[f:][c0:c0 + step] for r, f in zip(rows, first)], [f + c0 for f in first])
        caches.append(cache)
    torch.cuda.synchronize()
    long, short = caches
    # the same fp32 operations per element in the same order (the compiler may
    # contract them differently): a chain of 200 with |gate| < 0.7 keeps
    # 1 / (1 - 0.7) roundings of 2^-24 of values below 8
    np.testing.assert_allclose(long.hist.cpu().numpy(), short.hist.cpu().numpy(), rtol=0, atol=4 * 3.4 * 8 * 2.0 ** -24)
    # K and V: the projection of h. fp32: the same sums. bf16: one ulp (2^-7) of
    # the value, and where a value of h rounds the other way (one ulp, at most
    # 2^-6 below 4) that times a weight (below 5 sigma = 1.5), a few times over
    rtol, atol = (1e-5, 1e-4) if dtype == "fp32" else (2.0 ** -7, 3 * 1.5 * 2.0 ** -6)
    for a, b in ((long.k, short.k), (long.v, short.v)):
        np.testing.assert_allclose(a.float().cpu().numpy(), b.float().cpu().numpy(), rtol=rtol, atol=atol)


@pytest.mark.parametrize("D,dtype", [(128, "fp32"), (24, "fp32"), (256, "bf16"), (1536, "bf16")])
@pytest.mark.parametrize("full", [0, 1])
def test_long_chunk_x0_and_logits_match_short_pieces(D, dtype, full):
    from flaxchat_amd import _lib
    from flaxchat_amd.config import GPTConfig
    from flaxchat_amd.runtime import DeviceCache, DeviceModel, Workspace, forward_packed, pack_rows
    print(f"D={D} {dtype} full={full}", flush=True)
    H = max(1, D // 128)
    cfg = GPTConfig(sequence_len=512, vocab_size=300, n_layer=2, n_head=H, n_kv_head=H, n_embd=D, window_pattern="L")
    dm = DeviceModel.random_init(cfg, seed=4, dtype=dtype, std=D ** -0.5)  # every product of the size of its input
    dm.desc.smear_lambda = 0.7
    dm.desc.layers[1].x0_lambda = 0.9  # x0, which nothing else reads, is half of the second layer's input
    rng = np.random.default_rng(D)
    lens = [200, 33, 1, 65, 64]
    rows = [rng.integers(0, 300, n).tolist() for n in lens]
    B = len(rows)
    ws = Workspace(dm.device)
    up = lambda a: torch.from_numpy(np.asarray(a, np.int32)).to(dm.device)  # noqa: E731
    sides = []
    for step in (1024, 32):
        cache = DeviceCache(dm, B, 256)
        last = torch.zeros(B, dm.V, device=dm.device)
        for c0 in range(0, 200, step):
            tok, off, mpr = pack_rows([r[c0:c0 + step] for r in rows])
            logits = torch.zeros(B, 1, dm.V, device=dm.device)
            forward_packed(dm, cache, up(tok), up(off), up([c0] * B), mpr, 1, logits, ws,
                           flags=_lib.FC_CHUNK_FULL_SMEAR if full else 0)
            ended = [b for b in range(B) if c0 < lens[b] <= c0 + step]
            last[ended] = logits[ended, 0]
        sides.append([t.double() for t in (last, cache.k[1], cache.v[1])])
    torch.cuda.synchronize()
    for name, a, b in zip(("logits", "K", "V"), *sides):
        err = float((a - b).norm() / b.norm())
        print(f"{name}: {err:.2e}", flush=True)
        # fp32: sums of up to 512 products in another order, a few layers deep (some 2^-24 each);
        # bf16: each side is within about 0.3% of float64 after two layers
        assert err <= (1e-5 if dtype == "fp32" else 0.012), name
