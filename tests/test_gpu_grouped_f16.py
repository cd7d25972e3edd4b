"""The grouped call's 64-pair tiles on f16 MFMA, at sizes that run them
(test_grouped_plan_cpu.py checks that they do): against a float64 forward to
the precision of f32 sums, and against the oracle where the values need it."""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from grouped_f16_cases import LONG_ROWS, LONG_ROWS_QMM, MANY, Q4, Q8  # noqa: E402
from test_gpu_grouped import oracle_moe  # noqa: E402
from test_gpu_parity import ABS_TOL, _table, assert_ffn_close, make_expert, say, to_dev  # noqa: E402
from test_gpu_qmm import assert_qmm_close  # noqa: E402

pytestmark = pytest.mark.gpu

BLOCK_BYTES = {Q4: 18, Q8: 34}


def _blobs(g, dtype, n, dm, dff, gpu):
    blocks = n * 3 * dm * dff // 32
    b = torch.empty((blocks, BLOCK_BYTES[dtype]), dtype=torch.uint8, device=gpu).random_(0, 256, generator=g)
    lo, hi = (0.005, 0.02) if dtype == Q4 else (0.002, 0.01)
    b[:, :2] = torch.empty((blocks, 1), device=gpu).uniform_(lo, hi, generator=g).half().view(torch.uint8)
    blobs = b.view(n, -1)
    return blobs, blobs.data_ptr() + blobs.shape[1] * torch.arange(n, dtype=torch.int64, device=gpu)


def _weights64(blob, dtype, dm, dff):
    """(gate, up [d_ff, d_model], down [d_model, d_ff]) in float64."""
    b = blob.view(3, -1, BLOCK_BYTES[dtype])
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    q = b[:, :, 2:]
    q = torch.cat([q & 15, q >> 4], 2).double() - 8 if dtype == Q4 else q.contiguous().view(torch.int8).double()
    w = (d * q).view(3, -1)
    return w[0].view(dff, dm), w[1].view(dff, dm), w[2].view(dm, dff)


def _ffn64(weights, x):
    g, u = x @ weights[0].t(), x @ weights[1].t()
    return g * torch.sigmoid(g) * u @ weights[2].t()


def _moe64(blobs, dtype, dm, dff, ids, w, x):
    """The float64 forward, and the same with the inputs kept as one f16."""
    out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    one = torch.zeros_like(out)
    for e in ids.unique().tolist():
        t, k = (ids == e).nonzero(as_tuple=True)
        m = _weights64(blobs[e], dtype, dm, dff)
        for acc, v in ((out, x[t].double()), (one, x[t].half().double())):
            acc.index_add_(0, t, _ffn64(m, v) * w[t, k].double()[:, None])
    return out, one


def _rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


# A sum of K products in f32, summed 32 and 512 at a time as the kernel does,
# is off by sqrt(32 / 2 + 16 + K / 512) roundings of up to 2^-25 on average,
# and K is 14336 at most: 2.3e-7 of the summands' norm, which the output's norm
# is close to on random signs.  Twice for the two projections and the inputs'
# 2^-24.  An input kept as one f16 alone is off by more than 1e-4.
BAR = 5e-7


@pytest.mark.parametrize("dtype,qmm,dm,dff,n_tok,k,n_exp,parts", LONG_ROWS + MANY)
def test_f16_tiles_precision(mer, gpu, dtype, qmm, dm, dff, n_tok, k, n_exp, parts):
    say(f"f16 tiles dtype={dtype} dm={dm} dff={dff} experts={n_exp} tokens={n_tok} k={k} parts={parts}")
    g = torch.Generator(device=gpu).manual_seed(dm + dff + n_tok)
    blobs, table = _blobs(g, dtype, n_exp, dm, dff, gpu)
    ids = torch.rand((n_tok, n_exp), generator=g, device=gpu).argsort(1)[:, :k].to(torch.int32).contiguous()
    w = torch.rand((n_tok, k), generator=g, device=gpu)
    w[n_tok // 2, 0] = 0.0  # a skipped slot
    x = torch.randn((n_tok, dm), generator=g, device=gpu)
    want, one = _moe64(blobs, dtype, dm, dff, ids, w, x)
    args = (mer.WeightDtype(dtype), dm, dff, table, ids, w, x)
    got = mer.moe_grouped(*args)
    err = _rel(got, want)
    say(f"  error {err:.2e}, with one f16 an input {_rel(one, want):.2e}")
    assert err <= BAR
    assert _rel(one, want) > 100 * BAR
    worst = ((got.double() - want).norm(dim=1) / want.norm(dim=1).clamp(min=want.norm(dim=1).mean() / 4)).max().item()
    assert worst <= 4 * BAR, worst  # each token by itself
    assert torch.equal(mer.moe_grouped(*args, residual=True), got + x)
    mer.take_device_status()


@pytest.mark.parametrize("dtype,qmm,dm,dff,n_tok,k,n_exp,parts", LONG_ROWS_QMM)
@pytest.mark.parametrize("limit", [None, 0.5])
def test_f16_tiles_qmm(mer, oracle, gpu, dtype, qmm, dm, dff, n_tok, k, n_exp, parts, limit):
    """Against the oracle under its flip bound, with and without a gate clamp,
    a NaN and an infinite input element among them: the quantisation turns the
    NaN into 0, and the NaN gates that the infinite element gives likewise."""
    say(f"f16 tiles qmm dm={dm} dff={dff} experts={n_exp} tokens={n_tok} k={k} limit={limit}")
    blobs = [make_expert(oracle, Q4, dm, dff, 80 + e) for e in range(n_exp)]
    devs, table = _table(blobs, gpu)
    rng = np.random.default_rng(dm + n_tok)
    ids = np.stack([rng.choice(n_exp, k, replace=False) for _ in range(n_tok)]).astype(np.int32)
    w = (rng.random((n_tok, k)) + 0.1).astype(np.float32)
    x = rng.standard_normal((n_tok, dm)).astype(np.float32)
    x[3, 5], x[7, dm - 1] = np.nan, np.inf
    want, bound = np.zeros((n_tok, dm), np.float32), np.zeros((n_tok, dm))
    try:
        mer.set_swiglu_limit(limit)
        oracle.set_swiglu_limit(limit if limit else float("inf"))
        for t in range(n_tok):
            res = [oracle.q4_0_qmm_forward_bounded(blobs[i], x[t], dm, dff) for i in ids[t]]
            want[t] = oracle.combine_outputs(np.stack([r[0] for r in res]), w[t])
            bound[t] = sum(float(w[t, i]) * res[i][1].astype(np.float64) for i in range(k))
        got = mer.moe_grouped(mer.WeightDtype.Q4_0, dm, dff, table, to_dev(ids, gpu), to_dev(w, gpu), to_dev(x, gpu),
                              qmm=True).cpu().numpy()
    finally:
        mer.set_swiglu_limit(None)
        oracle.set_swiglu_limit(float("inf"))
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert ok.sum() >= (n_tok - 1) * dm
    assert_qmm_close(got[ok], want[ok], bound[ok], f"f16 tiles qmm limit={limit}")
    mer.take_device_status()
    del devs


@pytest.mark.parametrize("dtype,dm,dff,n_tok,k,n_exp", [(Q4, 64, 8256, 40, 2, 2), (Q8, 192, 8256, 33, 1, 1)])
def test_f16_tiles_gate_clamp(mer, oracle, gpu, dtype, dm, dff, n_tok, k, n_exp):
    say(f"f16 tiles gate clamp dtype={dtype} dm={dm} dff={dff}")
    blobs = [make_expert(oracle, dtype, dm, dff, 60 + e) for e in range(n_exp)]
    devs, table = _table(blobs, gpu)
    rng = np.random.default_rng(31)
    ids = np.stack([rng.choice(n_exp, k, replace=False) for _ in range(n_tok)]).astype(np.int32)
    w = rng.random((n_tok, k)).astype(np.float32)
    x = (rng.standard_normal((n_tok, dm)) * 3).astype(np.float32)
    run = lambda: mer.moe_grouped(mer.WeightDtype(dtype), dm, dff, table, to_dev(ids, gpu), to_dev(w, gpu),
                                  to_dev(x, gpu)).cpu().numpy()
    plain = run()
    limit = 0.5 if dtype == Q4 else 2.0
    try:
        mer.set_swiglu_limit(limit)
        oracle.set_swiglu_limit(limit)
        got, want = run(), oracle_moe(oracle, dtype, blobs, ids, w, x, dm, dff)
    finally:
        mer.set_swiglu_limit(None)
        oracle.set_swiglu_limit(float("inf"))
    assert_ffn_close(got, want, "f16 tiles clamped")
    assert np.abs(got - plain).max() > 10 * ABS_TOL, "the clamp did not bind"
    assert np.array_equal(run(), plain)
    mer.take_device_status()
    del devs


@pytest.mark.parametrize("dtype,qmm,dm,dff,n_tok,k,n_exp", [(Q8, 0, 64, 8256, 90, 2, 4), (Q4, 0, 192, 8256, 45, 3, 3),
                                                            (Q4, 1, 64, 8256, 40, 2, 3)])
def test_f16_tiles_missing_experts(mer, gpu, dtype, qmm, dm, dff, n_tok, k, n_exp):
    """Absent entries, negative ids and ids past the table are misses, slots of
    weight zero are skipped whatever their id: the rest equals, bit for bit, a
    call whose missing slots weigh nothing.  The down sums come in four parts,
    with slots that no tile writes; then a call without any tile."""
    say(f"f16 tiles missing experts dtype={dtype} qmm={qmm} dm={dm} dff={dff}")
    g = torch.Generator(device=gpu).manual_seed(dm)
    blobs, table = _blobs(g, dtype, n_exp, dm, dff, gpu)
    table[1] = 0
    rng = np.random.default_rng(n_tok)
    ids = rng.integers(-1, n_exp + 2, (n_tok, k)).astype(np.int32)
    w = (rng.random((n_tok, k)) + 0.1).astype(np.float32)
    w[rng.random((n_tok, k)) < 0.2] = 0.0
    hit = (ids >= 0) & (ids < n_exp) & (ids != 1) & (w != 0)
    x = torch.randn((n_tok, dm), generator=g, device=gpu)

    def run(ids_, w_, **kw):
        return mer.moe_grouped(mer.WeightDtype(dtype), dm, dff, table, to_dev(ids_, gpu), to_dev(w_, gpu), x,
                               qmm=bool(qmm), **kw)

    got = run(ids, w)
    with pytest.raises(mer.GpuExpertDispatchError):
        mer.take_device_status()
    assert torch.equal(got, run(np.where(hit, ids, 0).astype(np.int32), np.where(hit, w, 0).astype(np.float32)))
    mer.take_device_status()  # no miss
    if not qmm:
        keep = to_dev(np.where(hit, ids, -1).astype(np.int32), gpu)
        want = torch.zeros((n_tok, dm), dtype=torch.float64, device=gpu)
        for e in set(ids[hit].tolist()):
            t, j = (keep == e).nonzero(as_tuple=True)
            want.index_add_(0, t, _ffn64(_weights64(blobs[e], dtype, dm, dff), x[t].double()) *
                            to_dev(w, gpu)[t, j].double()[:, None])
        assert _rel(got, want) <= BAR
    none = np.full((n_tok, k), -1, np.int32)
    ones = np.ones((n_tok, k), np.float32)
    assert torch.equal(run(none, ones, residual=True), x)
    with pytest.raises(mer.GpuExpertDispatchError):
        mer.take_device_status()
    out = x.clone()
    run(none, np.zeros((n_tok, k), np.float32), out=out, accumulate=True)
    assert torch.equal(out, x)
    mer.take_device_status()


def test_f16_tiles_extreme_inputs(mer, gpu):
    """Vectors of very different sizes, elements far below their vector's
    largest one, and non-finite vectors, which make their own token's outputs
    NaN and no others."""
    dm, dff, n_tok = 256, 8256, 40
    say("f16 tiles extreme inputs")
    g = torch.Generator(device=gpu).manual_seed(4)
    blobs, table = _blobs(g, Q8, 1, dm, dff, gpu)
    rng = np.random.default_rng(4)
    x = rng.standard_normal((n_tok, dm)).astype(np.float32)
    x[:8] *= np.float32(2.0) ** np.arange(-40, -8, 4, dtype=np.float32)[:, None]
    x[8:16] *= np.float32(2.0) ** rng.integers(-30, 1, (8, dm)).astype(np.float32)
    x[16] = 0.0
    x[17, 5], x[18, 200] = np.inf, np.nan
    x = to_dev(x, gpu)
    got = mer.moe_grouped(mer.WeightDtype.Q8_0, dm, dff, table, torch.zeros((n_tok, 1), dtype=torch.int32, device=gpu),
                          torch.ones((n_tok, 1), device=gpu), x)
    mer.take_device_status()
    assert torch.isnan(got[17:19]).all() and (got[16] == 0).all()
    ok = [t for t in range(n_tok) if t not in (16, 17, 18)]
    want = _ffn64(_weights64(blobs[0], Q8, dm, dff), x[ok].double())
    err = ((got[ok].double() - want).norm(dim=1) / want.norm(dim=1)).max().item()
    assert err <= 4 * BAR, err


@pytest.mark.parametrize("outlier", [2.0**10, 2.0**16, 2.0**20])
def test_f16_tiles_small_elements_beside_an_outlier(mer, gpu, outlier):
    """An input element is held to 2^-23 of itself or 2^-39 of its vector's
    largest one, whichever is more.  The outlier's weights are 0 here, so the
    small elements alone decide the output."""
    dm, dff, n_tok = 128, 8256, 40
    say(f"f16 tiles outlier {outlier}")
    g = torch.Generator(device=gpu).manual_seed(6)
    blobs, table = _blobs(g, Q8, 1, dm, dff, gpu)
    rows = blobs.view(3, -1, 34)[:2].view(2, dff, dm // 32, 34)
    rows[:, :, 0, 2 + 7] = 0  # element 7 of every gate and up row
    x = torch.randn((n_tok, dm), generator=g, device=gpu)
    x[:, 7] = outlier
    got = mer.moe_grouped(mer.WeightDtype.Q8_0, dm, dff, table, torch.zeros((n_tok, 1), dtype=torch.int32, device=gpu),
                          torch.ones((n_tok, 1), device=gpu), x).double()
    mer.take_device_status()
    wg, wu, wd = _weights64(blobs[0], Q8, dm, dff)
    x = x.double()
    want = _ffn64((wg, wu, wd), x)
    small = x.clone()
    small[:, 7] = 0
    # the inputs' error, and 40 roundings of the f32 sums (4 blocks of K)
    dx = torch.maximum(small.abs() * 2.0**-23, torch.full_like(x, outlier * 2.0**-39))
    dx[:, 7] = 0
    a, u = small @ wg.t(), small @ wu.t()
    da, du = [dx @ m.abs().t() + 40 * 2.0**-24 * (small.abs() @ m.abs().t()) for m in (wg, wu)]
    s = a * torch.sigmoid(a)
    # |silu'| <= 1.1; h in f32 with a fast exponential, then held as the inputs are
    dh = 1.1 * da * (u.abs() + du) + s.abs() * du + 8 * 2.0**-24 * (s * u).abs()
    h = s * u
    dh += torch.maximum(h.abs() * 2.0**-23, h.abs().amax(1, keepdim=True) * 2.0**-39)
    bar = dh @ wd.abs().t() + 80 * 2.0**-24 * (h.abs() @ wd.abs().t())
    say(f"  worst error / bound {((got - want).abs() / bar).max().item():.3f}, relative {_rel(got, want):.2e}")
    assert ((got - want).abs() <= bar).all()
    # normwise: what inputs off by a random part of 2^-39 of the outlier give
    assert _rel(got, want) <= BAR + outlier * 2.0**-39
