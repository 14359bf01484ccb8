"""Prefill-width attention: the one- and two-group kernels at ragged rows
(empty and one-token rows among them), GQA groups whose columns straddle
tokens, windows, key counts around its 64-key steps, and row-major against
operand-order output. And the merge of the decode kernels' key splits."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")
import flaxchat_amd.torch_ops as tops  # noqa: E402
from flaxchat_amd import _lib  # noqa: E402
from flaxchat_amd._lib import check, lib  # noqa: E402

pytestmark = pytest.mark.gpu


def _reference(q, k, v, n, start, off, window):
    """float64 attention of packed rows over plain [B][G][cap][128] keys / values; a query past
    the cache's end sees what its window leaves of the cache, and one that sees no key gives 0."""
    out = torch.zeros(q.shape[0], q.shape[1] * 128, dtype=torch.float64, device=q.device)
    rep = q.shape[1] // k.shape[1]
    for b in range(len(n)):
        if n[b] == 0:
            continue
        end = start[b] + n[b]
        qb = q[off[b]:off[b + 1]].double().transpose(0, 1)                     # [H][n][128]
        kb = k[b, :, :end].double().repeat_interleave(rep, 0)
        vb = v[b, :, :end].double().repeat_interleave(rep, 0)
        pos = torch.arange(start[b], end, device=q.device)[:, None]
        key = torch.arange(kb.shape[1], device=q.device)[None]
        see = (key <= pos) & ((pos - key <= window) if window > 0 else True)
        s = (torch.matmul(qb, kb.transpose(1, 2).contiguous()) / np.sqrt(128)).masked_fill(~see, -np.inf)
        p = torch.softmax(s, -1).masked_fill(~see, 0.0)
        out[off[b]:off[b + 1]] = torch.matmul(p, vb).transpose(0, 1).reshape(n[b], -1)
    return out


def _layouts(k, v):
    """The caches' layouts: K blocks of 32 keys in K.Q^T fragment order, V blocks transposed."""
    B, G, cap = k.shape[:3]
    kb = torch.empty_like(k)
    kk, d = torch.arange(32, device="cuda")[:, None], torch.arange(128, device="cuda")[None]
    e = ((2 * (d // 32) + (kk // 4) % 2) * 64 + 4 * (kk // 8) + kk % 4 + 16 * ((d // 8) % 4)) * 8 + d % 8
    kb.view(B, G, cap // 32, 4096)[..., e.reshape(-1)] = k.view(B, G, cap // 32, 4096)
    return kb, v.view(B, G, cap // 32, 32, 128).transpose(3, 4).contiguous()


# (heads, groups, tokens per row, first positions, window): up to 256 workgroups
# take two groups of waves, more one
CASES = [(2, 2, [128], [0], 0), (2, 2, [129, 0, 1, 200], [0, 0, 700, 63], 0), (12, 4, [43, 100, 7], [500, 0, 64], 100),
         (6, 6, [300], [1000], 256), (6, 2, [64, 63], [1, 130], 0), (12, 12, [256] * 12, [0, 1, 31, 32, 63, 64, 65, 127,
                                                                                         300, 512, 600, 20], 300),
         (12, 4, [180] * 17, list(range(0, 340, 20)), 0)]


@pytest.mark.parametrize("H,G,n,start,window", CASES)
def test_prefill_attention(H, G, n, start, window):
    print(f"H={H} G={G} n={n} start={start} window={window}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(len(n) + H)
    B, cap = len(n), (max(a + b for a, b in zip(n, start)) + 31) // 32 * 32
    off = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    tot = int(off[-1])
    # keys with a few large scores, so that maxima rise late in the walk too
    q = (torch.randn(tot, H, 128, device="cuda", generator=gen) * 2).to(torch.bfloat16)
    k = (torch.randn(B, G, cap, 128, device="cuda", generator=gen) * 1.5).to(torch.bfloat16)
    v = torch.randn(B, G, cap, 128, device="cuda", generator=gen).to(torch.bfloat16)
    kb, vb = _layouts(k, v)
    ro, st = torch.from_numpy(off).cuda(), torch.tensor(start, dtype=torch.int32, device="cuda")
    mpr = max(max(n), -(-128 * G // H))  # prefill width: at least 128 columns per row and group
    got = torch.ops.flaxchat_mi355x.attention(q, kb, vb, ro, st, mpr, window)
    want = _reference(q, k, v, n, start, off, window)
    # P and the output are rounded to bf16 (2^-9 relative each), P against values below ~4.5
    assert float((got.double() - want).abs().max()) <= 2 * 2.0 ** -9 * 4.5 + 2.0 ** -9
    # operand order: the same numbers elsewhere
    y = torch.zeros((tot + 15) // 16 * 16, H * 128, dtype=torch.bfloat16, device="cuda")
    max_keys = min(cap, window + mpr) if window > 0 else cap
    ws = torch.empty(max(1, lib().fc_attention_workspace_bytes(B, mpr, H, G, 128, max_keys)), dtype=torch.uint8,
                     device="cuda")
    check(lib().fc_attention(q.data_ptr(), kb.data_ptr(), vb.data_ptr(), y.data_ptr(), B, tot, mpr, H, G, 128, cap,
                             ro.data_ptr(), st.data_ptr(), window, max_keys, _lib.FC_BF16, ws.data_ptr(), ws.numel(),
                             torch.cuda.current_stream().cuda_stream), "fc_attention")
    assert torch.equal(tops.frag_to_rows(y, tot), got)


# rows that run past the cache's end: an odd number of 32-key tiles (3, 9, 5) and of 64-key
# steps (5, 3), one and two groups of waves (two: 256 keys or more and few workgroups), a
# first position behind the end, queries whose window lies behind it, GQA
@pytest.mark.parametrize("H,G,n,start,window,cap", [
    (2, 2, [130], [0], 0, 96), (2, 2, [300, 130], [0, 200], 0, 288), (2, 2, [400], [100], 100, 288),
    (6, 2, [200, 64], [150, 288], 0, 288), (2, 2, [128], [300], 20, 288), (12, 4, [180] * 17, list(range(0, 340, 20)), 0,
                                                                          160)])
def test_prefill_attention_past_the_cache(H, G, n, start, window, cap):
    """Every cached key counts once for a query at a position past the cache."""
    print(f"H={H} G={G} n={n} start={start} window={window} cap={cap}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(len(n) + H)
    B = len(n)
    off = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    q = torch.randn(int(off[-1]), H, 128, device="cuda", generator=gen).to(torch.bfloat16)
    k = torch.randn(B, G, cap, 128, device="cuda", generator=gen).to(torch.bfloat16)
    v = torch.randn(B, G, cap, 128, device="cuda", generator=gen).to(torch.bfloat16)
    kb, vb = _layouts(k, v)
    ro, st = torch.from_numpy(off).cuda(), torch.tensor(start, dtype=torch.int32, device="cuda")
    got = torch.ops.flaxchat_mi355x.attention(q, kb, vb, ro, st, max(n), window)
    want = _reference(q, k, v, n, start, off, window)
    # P and the output are rounded to bf16 (2^-9 relative each), P against values below ~4.5
    assert float((got.double() - want).abs().max()) <= 2 * 2.0 ** -9 * 4.5 + 2.0 ** -9


# key splits of 128 keys: 1, 2, 3, 4, 5, 8, 9, 16, 17 and 43 (merged 2, 4 or 8 at a time); splits past a short row's end and before a
# window hold nothing; empty rows; 21 columns of a GQA group
@pytest.mark.parametrize("H,G,n,start,window", [
    (6, 6, [1], [100], 0), (6, 6, [1], [254], 0), (6, 6, [1], [300], 0), (6, 6, [1, 1], [500, 3], 0),
    (6, 6, [3], [600], 0), (6, 6, [1], [1022], 0), (6, 6, [1], [1024], 0),
    (6, 6, [1], [2047], 0), (6, 6, [1], [2048], 0), (6, 6, [1, 0, 1], [2048, 5, 10], 0), (6, 6, [1], [5600], 0),
    (12, 4, [7, 3], [5400, 900], 0), (6, 6, [5], [3000], 1024)])
def test_key_split_merge(H, G, n, start, window):
    print(f"H={H} G={G} n={n} start={start} window={window}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(start[0] + H)
    B, cap = len(n), (max(a + b for a, b in zip(n, start)) + 31) // 32 * 32
    off = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    q = (torch.randn(int(off[-1]), H, 128, device="cuda", generator=gen) * 2).to(torch.bfloat16)
    k = (torch.randn(B, G, cap, 128, device="cuda", generator=gen) * 1.5).to(torch.bfloat16)
    v = torch.randn(B, G, cap, 128, device="cuda", generator=gen).to(torch.bfloat16)
    kb, vb = _layouts(k, v)
    ro, st = torch.from_numpy(off).cuda(), torch.tensor(start, dtype=torch.int32, device="cuda")
    got = torch.ops.flaxchat_mi355x.attention(q, kb, vb, ro, st, max(n), window)
    want = _reference(q, k, v, n, start, off, window)
    # P and the output are rounded to bf16 (2^-9 relative each), P against values below ~4.5
    assert float((got.double() - want).abs().max()) <= 2 * 2.0 ** -9 * 4.5 + 2.0 ** -9


# NaN in the V of keys 96-127 reaches no query before them, of keys 64-95 no wave (32 queries)
# whose windows start at key 96 or behind, though they lie in one 64-key step with keys it sees
@pytest.mark.parametrize("bad,window,clean", [(range(96, 128), 0, range(0, 96)),
                                              (range(64, 96), 40, [*range(0, 64), *range(160, 300)])])
@pytest.mark.parametrize("cap", [320, 1024])
@pytest.mark.parametrize("B", [1, 80])  # two groups of waves, one group
def test_prefill_attention_unseen_tiles(bad, window, clean, cap, B):
    """A 32-key tile that none of a wave's queries sees does not reach them, whatever its V holds."""
    print(f"bad={bad} window={window} cap={cap} B={B}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(7)
    n, G = 300, 2
    q = torch.randn(B * n, G, 128, device="cuda", generator=gen).to(torch.bfloat16)
    k = torch.randn(B, G, cap, 128, device="cuda", generator=gen).to(torch.bfloat16)
    v = torch.randn(B, G, cap, 128, device="cuda", generator=gen).to(torch.bfloat16)
    ro = torch.arange(0, B * n + 1, n, dtype=torch.int32, device="cuda")
    st = torch.zeros(B, dtype=torch.int32, device="cuda")

    def run():
        return torch.ops.flaxchat_mi355x.attention(q, *_layouts(k, v), ro, st, n, window).view(B, n, -1)

    before = run()
    v[:, :, list(bad)] = float("nan")
    after = run()
    assert torch.equal(after[:, list(clean)], before[:, list(clean)])
    assert bool(after[:, bad[0]:bad[-1] + 1].isnan().all())
