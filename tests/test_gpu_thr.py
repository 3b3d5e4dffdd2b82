"""Rows that take the threshold statistics (csrc/sdx_thr.hip) against the oracle, bit
for bit: every shape of row at which the region, its list, the refinement over the
row or the compaction can go wrong, at vocabularies on the edges of the parts and
records, and rows that do not start 16-byte aligned."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import sampling as O
from specdec import _lib
from specdec import sampling as S

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rows(V, seed, dtype=np.float32):
    """Rows [n, V]: spread, narrow and nearly equal logits, tie groups from a few
    members to the whole row (past the list of 2,048, so the row is refined), rows of
    -inf but one or a tenth, and extremes of the range."""
    rng = np.random.RandomState(seed)
    masked = rng.randn(V) * 3
    masked[rng.rand(V) < 0.9] = -np.inf
    one = np.full(V, -np.inf)
    one[V // 2] = 1.0
    peak = rng.randn(V) * 2
    peak[7] = 60.0
    half = rng.randn(V) * 2
    half[: V // 2] = 1.25
    rows = [rng.randn(V) * 3, rng.randn(V) * 0.3, rng.randn(V) * 0.01, np.zeros(V),
            np.where(np.arange(V) % 3 == 0, 2.0, -1.0), np.round(rng.randn(V) * 12) / 4,
            np.round(rng.randn(V) * 2) / 4, masked, one, np.linspace(-40, 10, V),
            rng.randn(V) * 30, peak, half,
            torch.tensor(rng.randn(V) * 3).bfloat16().float().numpy()]
    if dtype == np.float32:
        rows += [rng.randn(V) * 1e-30, -np.abs(rng.randn(V)) * 1e30]
    return np.stack(rows).astype(dtype)


TRANSFORMS = [(1.0, 1.0, 0), (0.8, 0.95, 0), (0.7, 0.9, 50), (1.0, 0.5, 0), (1.3, 1.0, 20),
              (0.6, 0.999999, 0), (1.0, 0.99999994, 0), (2.0, 0.95, 3000), (0.9, 0.3, 5000),
              (1e-3, 0.9, 0), (4e6, 0.9, 0)]


def _same(got, ref):
    bad = np.argwhere(got.view(np.uint32) != ref.view(np.uint32))
    assert bad.size == 0, f"{len(bad)} elements differ, first at {bad[0]}"


# one workgroup per row: a few ids, and both sides of the workgroup sizes
@pytest.mark.parametrize("V", [9, 1000, 2048, 2049, 4096, 4097, 8192])
@pytest.mark.parametrize("T,tp,tk", TRANSFORMS)
def test_to_probs_short_rows(V, T, tp, tk):
    x = _rows(V, V)
    got = S.to_probs(torch.tensor(x, device=DEV), T, tp, tk).cpu().numpy()
    _same(got, O.to_probs(x, T, tp, tk))
    if V % 8 == 0 and T > 1e-2:
        h = _rows(V, V, np.float16)
        got = S.to_probs(torch.tensor(h, device=DEV), T, tp, tk).cpu().numpy()
        _same(got, O.to_probs(h.astype(np.float32), T, tp, tk))


# 8193: the shortest row, one part; 12291: three parts' worth of 4,096 and 3 ids more;
# 33000: several parts
@pytest.mark.parametrize("V", [8193, 12291, 33000])
@pytest.mark.parametrize("T,tp,tk", TRANSFORMS)
def test_to_probs_rows(V, T, tp, tk):
    x = _rows(V, V)
    got = S.to_probs(torch.tensor(x, device=DEV), T, tp, tk).cpu().numpy()
    _same(got, O.to_probs(x, T, tp, tk))


@pytest.mark.parametrize("V", [8200, 33000])
@pytest.mark.parametrize("T,tp,tk", [t for t in TRANSFORMS if t[0] > 1e-2])
def test_to_probs_fp16_rows(V, T, tp, tk):
    x = _rows(V, V, np.float16)
    got = S.to_probs(torch.tensor(x, device=DEV), T, tp, tk).cpu().numpy()
    _same(got, O.to_probs(x.astype(np.float32), T, tp, tk))


# odd lengths, the maximum (or an infinity) among the ids after the last whole 16 bytes
@pytest.mark.parametrize("V", [9, 1001, 8191, 8193, 8199, 33001, 50257])
def test_to_probs_fp16_odd_rows(V):
    x = _rows(V, V, np.float16)
    x[:4, V - 1] = 40.0
    x[4:8, V - 1 - V % 8 // 2] = 35.0
    for T, tp, tk in ((0.8, 0.95, 0), (1.0, 1.0, 0), (1.0, 0.9, 50)):
        got = S.to_probs(torch.tensor(x, device=DEV), T, tp, tk).cpu().numpy()
        _same(got, O.to_probs(x.astype(np.float32), T, tp, tk))


@pytest.mark.parametrize("V", [1000, 4097, 9000, 33000])
def test_top_k_among_subnormal_probabilities(V):
    """The k-th largest probability is subnormal: its tie group spans up to a unit of the
    logits over T, far below the group's largest logit, and all of it is kept."""
    rng = np.random.RandomState(V)
    x = np.full((4, V), -200.0, np.float32)
    x[0, [10, 20, 30]] = 0.0, -103.0, -103.5
    for r in (1, 2):  # 70 logits where p runs from normal to 0
        x[r, rng.permutation(V)[:70]] = -rng.uniform(85.0, 104.5, 70)
        x[r, 5] = 0.0
    x[3] = rng.randn(V) * 3
    ties = 0
    for T, tp, tk in [(1.0, 1.0, k) for k in range(2, 70)] + \
            [(t, 0.9, k) for t in (0.02, 0.03, 0.05, 0.08) for k in (20, 50, 200)]:
        ref = O.to_probs(x, T, tp, tk)
        ties += int(((ref > 0).sum(-1) > tk).any())
        _same(S.to_probs(torch.tensor(x, device=DEV), T, tp, tk).cpu().numpy(), ref)
    assert ties > 5


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("V", [1001, 2048, 4001, 8192, 9001, 33000, 151936])
def test_to_probs_refined_rows(dtype, V):
    """Regions past the list (2,048, or 256 to 1,024 in short rows): flat rows whose masked ids (a finite value) widen
    the steps, tie groups within and across them, values too near for the first bins.
    The boundary ends in a short list, in a tie group (whole or in part) or nowhere."""
    rng = np.random.RandomState(V)
    x = np.stack([rng.randn(V), rng.randn(V), np.round(rng.randn(V) * 8) / 8, rng.randn(V) * 1e-3,
                  np.where(np.arange(V) % 3 == 0, 2.0, -1.0), np.full(V, 0.5),
                  np.where(rng.rand(V) < 0.5, 1.25, rng.randn(V))])
    x[1:, :: V // 100] = -1e4
    t = torch.tensor(x).to(dtype)
    x = t.float().numpy()
    for T, tp, tk in [(1.5, 0.9, 0), (4.0, 0.9, 0), (2.0, 1.0, 5000), (8.0, 1.0, V // 2),
                      (3.0, 0.6, V // 4), (8.0, 0.3, V // 4), (8.0, 0.3, V // 3 + 2),
                      (50.0, 0.5, 0), (50.0, 1.0, V - 200), (50.0, 0.999999, 0)]:
        ref = O.to_probs(x, T, tp, tk)
        _same(S.to_probs(t.to(DEV), T, tp, tk).cpu().numpy(), ref)
        if V == 9001:  # more rows than CUs: smaller workgroups
            got = S.to_probs(t.to(DEV).repeat(40, 1), T, tp, tk).view(40, *t.shape)
            assert torch.equal(got, got[:1].expand_as(got))
            _same(got[0].cpu().numpy(), ref)


def test_top_k_of_all_but_one():
    x = _rows(9000, 1)
    got = S.to_probs(torch.tensor(x, device=DEV), 1.0, 1.0, 8999).cpu().numpy()
    _same(got, O.to_probs(x, 1.0, 1.0, 8999))


@pytest.mark.parametrize("off,ld,ldo", [(0, 9001, 9003), (1, 9002, 9001), (3, 9004, 9007)])
def test_to_probs_rows_at_any_alignment(off, ld, ldo):
    """C ABI rows of logits and probabilities at every 16-byte phase, with strides that
    put them out of phase with each other."""
    V, L = 9001, _lib.lib()
    x = _rows(V, 5)
    n = x.shape[0]
    buf = torch.zeros(off + n * ld, device=DEV)
    buf[off:].view(n, ld)[:, :V].copy_(torch.tensor(x))
    out = torch.full((n * ldo + 4,), -1.0, device=DEV)
    ws = _lib.workspace(L.sdx_to_probs_workspace(n, V, _lib.F32), DEV, prepare=False)
    rc = L.sdx_to_probs(ctypes.c_void_p(buf.data_ptr() + 4 * off), _lib.F32, n, V, ld, 0.8, 0.95, 0,
                        ctypes.c_void_p(out.data_ptr()), ldo, _lib.ptr(ws), ws.numel(),
                        _lib.stream_of(out))
    _lib.check(rc, "to_probs")
    got = out[: n * ldo].view(n, ldo)[:, :V].cpu().numpy()
    _same(np.ascontiguousarray(got), O.to_probs(x, 0.8, 0.95, 0))
    # nothing past the last row is touched
    assert bool((out[(n - 1) * ldo + V:] == -1.0).all())


# 8193: the shortest row of this kernel, 32768: its longest; odd fp16 lengths
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("V", [8193, 12345, 32761, 32768])
@pytest.mark.parametrize("T", [1.0, 0.7, 0.03, 400.0])
def test_to_probs_without_a_filter(dtype, V, T):
    x = _rows(V, V, dtype)
    got = S.to_probs(torch.tensor(x, device=DEV), T).cpu().numpy()
    _same(got, O.to_probs(x.astype(np.float32), T, 1.0, 0))
    x[0], x[1, 3] = -np.inf, np.inf  # no finite maximum: 0 / 0
    got = S.to_probs(torch.tensor(x, device=DEV), T).cpu().numpy()
    assert np.isnan(got[:2]).all() and not np.isnan(got[2:]).any()


@pytest.mark.parametrize("off,ld,ldo", [(0, 9001, 9003), (1, 9002, 9001), (3, 9004, 9007)])
def test_to_probs_without_a_filter_at_any_alignment(off, ld, ldo):
    V, L = 9001, _lib.lib()
    x = _rows(V, 6)
    n = x.shape[0]
    buf = torch.zeros(off + n * ld, device=DEV)
    buf[off:].view(n, ld)[:, :V].copy_(torch.tensor(x))
    out = torch.full((n * ldo + 4,), -1.0, device=DEV)
    ws = _lib.workspace(L.sdx_to_probs_workspace(n, V, _lib.F32), DEV, prepare=False)
    rc = L.sdx_to_probs(buf.data_ptr() + 4 * off, _lib.F32, n, V, ld, 0.8, 1.0, 0, _lib.ptr(out),
                        ldo, _lib.ptr(ws), ws.numel(), _lib.stream_of(out))
    _lib.check(rc, "to_probs")
    got = out[: n * ldo].view(n, ldo)
    _same(np.ascontiguousarray(got[:, :V].cpu().numpy()), O.to_probs(x, 0.8, 1.0, 0))
    assert bool((got[:-1, V:] == -1.0).all()) and bool((out[(n - 1) * ldo + V:] == -1.0).all())


def _verify_case(B, k, V, dtype, seed):
    """Logits of the row shapes above (without those whose p is 0 / 0 in every target),
    drafted ids from the likely ones and from tie groups."""
    rng = np.random.RandomState(seed)
    base = _rows(V, seed, np.float16 if dtype == torch.float16 else np.float32)[:14]
    pick = rng.randint(0, 14, size=(B, k + 1))
    tgt = base[pick].astype(np.float32)
    drf = tgt[:, :k] + np.where(rng.rand(B, k, 1) < 0.5, 0.0,
                                np.round(rng.randn(B, k, V)) / 4).astype(np.float32)
    t = torch.tensor(tgt).to(dtype)
    d = torch.tensor(drf).to(dtype)
    ids = rng.randint(0, V, size=(B, k))
    top = np.argsort(-d.float().numpy(), axis=-1, kind="stable")[..., :40]
    near = np.take_along_axis(top, rng.randint(0, 40, size=(B, k, 1)), -1)[..., 0]
    ids = np.where(rng.rand(B, k) < 0.8, near, ids)
    return (t, d, torch.tensor(ids), torch.tensor(rng.rand(B, k).astype(np.float32)),
            torch.tensor(rng.rand(B).astype(np.float32)))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("V,T,tp,tk", [(40, 1.0, 0.9, 5), (1000, 0.8, 0.95, 0), (8200, 0.8, 0.95, 0),
                                       (9217, 1.0, 0.7, 0), (33000, 0.7, 0.9, 50),
                                       (16384, 1.0, 1.0, 0)])
@pytest.mark.parametrize("B,k", [(12, 3), (3, 40)])  # 40: more positions than half a wave
def test_verify_rows(dtype, V, T, tp, tk, B, k):
    t, d, ids, ua, uf = _verify_case(B, k, V, dtype, V)
    n, y, f = S.rejection_sample(t.to(DEV), d.to(DEV), ids.to(DEV), ua.to(DEV), uf.to(DEV),
                                 temperature=T, top_p=tp, top_k=tk)
    rn, ry, rf = O.rejection_sample(t.float().numpy(), d.float().numpy(), ids.numpy(), ua.numpy(),
                                    uf.numpy(), T, tp, tk)
    assert np.array_equal(n.cpu().numpy(), rn)
    assert np.array_equal(y.cpu().numpy(), ry)
    assert np.array_equal(f.cpu().numpy(), rf)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("V,T,tp,tk", [(8200, 0.8, 0.95, 0), (33000, 1.0, 0.7, 300)])
def test_draft_step_rows(dtype, V, T, tp, tk):
    """The draw of every row and the drawn id's probability; a row of -inf but one id
    draws it."""
    x = _rows(V, V + 1, np.float16 if dtype == torch.float16 else np.float32)[:14]
    lg = torch.tensor(x).to(dtype)
    u = torch.rand(14, generator=torch.Generator().manual_seed(V))
    conf = torch.full((14,), 0.5, device=DEV)
    xd, qx, _ = S.draft_step(lg.to(DEV), u.to(DEV), T, tp, tk, conf=conf)
    q = O.to_probs(lg.float().numpy(), T, tp, tk)
    ref = O.sample_from_probs(q, u.numpy())
    assert np.array_equal(xd.cpu().numpy(), ref)
    rq = q[np.arange(14), ref]
    assert np.array_equal(qx.cpu().numpy(), rq)
    assert np.array_equal(conf.cpu().numpy(), np.float32(0.5) * rq)


def test_fp16_verify_without_room_for_the_scratch():
    """A workspace of the register-resident kernel's size (sdx_verify_noalloc's array for
    many rows) still serves fp16 rows, with the same results where a row's values fit that
    kernel's window (it flags the others); a +inf logit flags its row in both."""
    L, B, k, V = _lib.lib(), 6, 2, 9000
    t, d, ids, ua, uf = (x.to(DEV) for x in _verify_case(B, k, V, torch.float16, 3))
    t[4, 1, 17] = float("inf")
    full = L.sdx_verify_workspace(B, k, V, _lib.F16)
    scratch = 64 + 1024 + 2048 * 8 + 1024 * 12  # per row
    small = full - (B * (2 * k + 1) * scratch + 255) // 256 * 256
    res = []
    for n in (full, small):
        ws = _lib.workspace(n, DEV)
        out = [torch.empty(B, dtype=x, device=DEV) for x in (torch.int64, torch.int64, torch.uint8)]
        rc = L.sdx_verify(_lib.ptr(t), _lib.ptr(d), _lib.F16, B, k, V, _lib.ptr(ids), _lib.ptr(ua),
                          _lib.ptr(uf), None, 0.8, 0.9, 0, *[_lib.ptr(o) for o in out],
                          _lib.ptr(ws), small if n == small else ws.numel(), _lib.stream_of(t))
        _lib.check(rc, "verify")
        res.append([o.cpu().numpy() for o in out])
    fine = (np.arange(B) != 4) & (res[1][2] & S.FLAG_UNSUPPORTED == 0)
    assert fine.sum() >= 2
    for a, b in zip(*res):
        assert np.array_equal(a[fine], b[fine])
    assert not (res[0][2] & S.FLAG_UNSUPPORTED).any()
    assert res[0][2][4] & S.FLAG_NONFINITE and res[1][2][4] & S.FLAG_NONFINITE
