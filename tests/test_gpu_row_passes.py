"""The one-pass row kernels at the edges of their ranges: row statistics and
the sampling step with the row in registers (rows of up to 65536 entries,
longer ones on the general path) and the cross-entropy, on rows with ties,
masked (-inf) entries, infinities and NaN, aligned and not."""

import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
import flaxchat_amd.torch_ops  # noqa: E402,F401
from flaxchat_amd import _lib  # noqa: E402
from flaxchat_amd._lib import FcRowstat, check, lib  # noqa: E402

pytestmark = pytest.mark.gpu


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _rows(V, seed):
    rng = np.random.default_rng(seed)
    z = (rng.standard_normal((8, V)) * 2.5).astype(np.float32)
    z[1] = np.round(z[1])                      # many equal values
    z[2] = 0.5                                 # all equal
    z[3, rng.random(V) < 0.9] = -np.inf        # masked vocabulary
    z[4] = -np.inf
    z[4, V // 2] = 1.0                         # a single finite entry
    z[5] = -np.inf
    z[6, V // 3] = np.inf
    z[7, V - 1] = z[7].max() + 1               # the last entry is the largest
    return z


def _upload(z, off):
    """z on the device with its first row `off` floats past a 16-byte boundary."""
    buf = torch.empty(z.size + off, dtype=torch.float32, device="cuda")
    t = buf[off:].view(z.shape)
    t.copy_(torch.from_numpy(z))
    return t


@pytest.mark.parametrize("V", [1, 3, 1000, 4098, 4099, 16384, 16385, 32768, 65535, 65536, 65540])
@pytest.mark.parametrize("top_k,T", [(40, 0.8), (1, 1.0), (130, 0.8), (1024, 1.0), (1500, 0.7), (0, 0.8), (40, 0.0)])
def test_row_stats_and_sample(V, top_k, T):
    from oracle.sampling import fast_sample, topk_keep
    print(f"V={V} top_k={top_k} T={T}", flush=True)
    z = _rows(V, V + top_k)
    B = len(z)
    zt = _upload(z, 1 if V % 2 else 0)
    stats = torch.zeros(B, 8, dtype=torch.int32, device="cuda")
    check(lib().fc_row_stats(zt.data_ptr(), B, V, T, top_k, stats.data_ptr(), _stream()), "row_stats")
    mx, sm, tau, tie, am = torch.ops.flaxchat_mi355x.row_stats(zt, T, top_k)
    i32 = dict(dtype=torch.int32, device="cuda")
    gen, pos, step, tok = torch.zeros(B, 8, **i32), torch.zeros(B, **i32), torch.full((B,), 3, **i32), torch.zeros(B, **i32)
    forced = torch.full((B,), -1, **i32)
    forced[0] = V - 1
    st2 = torch.zeros(B, 8, dtype=torch.int32, device="cuda")
    check(lib().fc_engine_sample(zt.data_ptr(), B, V, T, top_k, 9, forced.data_ptr(), gen.data_ptr(), 8, pos.data_ptr(),
                                 step.data_ptr(), tok.data_ptr(), st2.data_ptr(), _stream()), "engine_sample")
    torch.cuda.synchronize()
    raw = stats.cpu().numpy().tobytes()
    # the operator's fields are the records'
    f = stats.view(torch.float32)
    for got, want in ((mx, f[:, 0]), (sm, f[:, 1]), (tau, f[:, 2]), (tie, stats[:, 3]), (am, stats[:, 4])):
        assert torch.equal(got.view(torch.int32), want.contiguous().view(torch.int32))
    assert torch.equal(st2[1:].cpu(), stats[1:].cpu())
    assert int(tok[0]) == V - 1 and pos.cpu().tolist() == [1] * B and step.cpu().tolist() == [4] * B
    assert gen.cpu()[:, 1].tolist() == tok.cpu().tolist()
    for r in range(B):
        rs = FcRowstat.from_buffer_copy(raw[r * 32:(r + 1) * 32])
        assert rs.argmax == int(np.argmax(z[r])), r
        if not T > 0:
            assert (rs.mx, rs.sum, rs.tau, rs.tie_idx) == (0.0, 1.0, -np.inf, V)
            assert r == 0 or int(tok[r]) == rs.argmax
            continue
        keep = topk_keep(z[r], top_k)
        tv = np.float32(rs.tau)
        assert np.array_equal((z[r] > tv) | ((z[r] == tv) & (np.arange(V) <= rs.tie_idx)), keep), r
        if not (keep & (z[r] == tv))[~keep].any() and not (~keep & (z[r] == tv)).any():
            assert rs.tie_idx == V, r                 # no equal entry left out
        with np.errstate(invalid="ignore"):
            x = (z[r][keep] / np.float32(T)).astype(np.float32)
            want = np.exp(x.astype(np.float64) - x.max()).sum()
        assert np.float32(rs.mx) == x.max(), r
        # fp32 sum of at most 65540 terms over 1024 threads: 64 sequential adds and
        # a tree of 10, each within 2^-24, and expf within 2 ulp
        np.testing.assert_allclose(rs.sum, want, rtol=(64 + 10 + 4) * 2.0 ** -24)
        if r > 0 and np.isfinite(x.max()):
            assert int(tok[r]) == fast_sample(z[r], T, top_k, 9, r, 3), r


@pytest.mark.parametrize("V,top_k", [(5000, 7), (65536, 0)])
def test_row_stats_with_nan_takes_the_general_path(V, top_k):
    """A NaN outranks every number: it is kept first and makes the sum NaN."""
    z = _rows(V, 1)[:2]
    z[1, 17] = np.nan
    zt = torch.from_numpy(z).cuda()
    mx, sm, tau, tie, am = torch.ops.flaxchat_mi355x.row_stats(zt, 1.0, top_k)
    assert int(am[1]) == int(np.nanargmax(z[1])) and bool(torch.isnan(sm[1])) and not bool(torch.isnan(sm[0]))
    assert float(mx[1]) == np.nanmax(z[1])


@pytest.mark.parametrize("V,stride", [(1, 1), (3, 5), (1000, 1000), (4099, 4100), (65535, 65535), (65536, 65540)])
@pytest.mark.parametrize("rows", [3, 600])
def test_cross_entropy_rows(V, stride, rows):
    print(f"V={V} stride={stride} rows={rows}", flush=True)
    if rows * stride > 1 << 25:
        rows = 520
    rng = np.random.default_rng(V)
    z = (rng.standard_normal((rows, stride)) * 3).astype(np.float32)
    t = rng.integers(0, V, rows).astype(np.int32)
    t[0] = -1
    if V > 3:
        z[1, :V - 1] = -np.inf                 # whole threads see masked entries alone
        t[1] = V - 1
        z[2, :V // 2] = -np.inf
        t[2] = V - 1
    zt = _upload(z, 1)
    tt = torch.from_numpy(t).cuda()
    loss = torch.empty(rows, dtype=torch.float32, device="cuda")
    check(lib().fc_cross_entropy(zt.data_ptr(), stride, tt.data_ptr(), rows, V, loss.data_ptr(), _stream()), "xent")
    zd = z[:, :V].astype(np.float64)
    m = zd.max(1, keepdims=True)
    want = np.log(np.exp(zd - m).sum(1)) + m[:, 0] - zd[np.arange(rows), np.maximum(t, 0)]
    want[t < 0] = 0.0
    # lse within 2^-24 (|lse| + the sum's relative error), and one subtraction
    np.testing.assert_allclose(loss.cpu().numpy(), want, rtol=1e-6, atol=40 * 2.0 ** -24 * 16)


def test_cross_entropy_nan_and_inf():
    z = np.zeros((3, 5000), np.float32)
    z[0, 77] = np.nan
    z[1] = -np.inf
    z[1, 4000] = np.nan
    z[2, 9] = np.inf
    loss = torch.ops.flaxchat_mi355x.cross_entropy(torch.from_numpy(z).cuda(), torch.zeros(3, dtype=torch.int32).cuda())
    assert torch.isnan(loss).all()
