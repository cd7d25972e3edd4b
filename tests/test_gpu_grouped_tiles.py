"""The grouped path at the ends of its tiles, against the CPU oracle: tiles
of one to several 16-pair groups, K that ends inside a stage, rows that end
inside a row tile, and the grouping of pairs.  These calls are small: most run
the int8 kernel's tiles of 16 pairs, those with 8256 inner rows the f16
kernel's tiles of 64, which test_gpu_grouped_f16.py covers."""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_grouped import oracle_moe  # noqa: E402
from test_gpu_parity import Q4, Q8, _table, assert_ffn_close, make_expert, say, to_dev  # noqa: E402
from test_gpu_qmm import assert_qmm_close  # noqa: E402

pytestmark = pytest.mark.gpu


def _routes(n_tok, k, n_exp, seed):
    rng = np.random.default_rng(seed)
    ids = np.stack([rng.choice(n_exp, k, replace=False) for _ in range(n_tok)]).astype(np.int32)
    return ids, rng.random((n_tok, k)).astype(np.float32), rng


@pytest.mark.parametrize("dtype,dm,dff,n_exp,n_tok,k", [
    (Q4, 64, 64, 1, 16, 1),      # two blocks of K, one 16-pair group
    (Q8, 64, 64, 1, 33, 1),      # two full tiles and one pair
    (Q8, 192, 320, 2, 65, 1),    # d_model that no 128-row tile divides
    (Q4, 192, 320, 3, 48, 2),    # six and ten blocks of K: stages cut short
    (Q4, 576, 192, 2, 40, 2),    # eighteen blocks
    (Q8, 1088, 64, 1, 17, 1),    # 34 blocks, one pair past a tile
    (Q4, 64, 4160, 2, 17, 2),    # down K of 130 blocks
    (Q8, 128, 8256, 1, 20, 1),   # f16 tiles: 258 blocks in four parts, the last one short
    (Q4, 64, 64, 140, 300, 7),   # 2100 pairs: 128-row gate/up workgroups
    (Q8, 64, 64, 140, 300, 7),   # 2100 pairs: 128-row gate/up workgroups
])
def test_tiles_vs_oracle(mer, oracle, gpu, dtype, dm, dff, n_exp, n_tok, k):
    say(f"grouped tiles dtype={dtype} dm={dm} dff={dff} experts={n_exp} tokens={n_tok} k={k}")
    blobs = [make_expert(oracle, dtype, dm, dff, 60 + e) for e in range(n_exp)]
    devs, table = _table(blobs, gpu)
    ids, w, rng = _routes(n_tok, k, n_exp, dm + dff)
    w[n_tok // 2, 0] = 0.0  # a skipped slot
    x = rng.standard_normal((n_tok, dm)).astype(np.float32)
    want = oracle_moe(oracle, dtype, blobs, ids, w, x, dm, dff) + x
    args = (mer.WeightDtype(dtype), dm, dff, table, to_dev(ids, gpu), to_dev(w, gpu), to_dev(x, gpu))
    got = mer.moe_grouped(*args, residual=True).cpu().numpy()
    assert_ffn_close(got, want, "grouped tiles")
    assert np.array_equal(mer.moe_grouped(*args, residual=True).cpu().numpy(), got)
    mer.take_device_status()
    del devs


@pytest.mark.parametrize("dm,dff,n_exp,n_tok,k", [
    (64, 64, 1, 16, 1), (192, 320, 2, 70, 1), (128, 4160, 2, 33, 1), (576, 192, 1, 64, 1),
    (64, 64, 140, 300, 7),  # 2100 pairs: 128-row gate/up workgroups
])
def test_tiles_qmm_vs_oracle(mer, oracle, gpu, dm, dff, n_exp, n_tok, k):
    say(f"grouped tiles qmm dm={dm} dff={dff} experts={n_exp} tokens={n_tok} k={k}")
    blobs = [make_expert(oracle, Q4, dm, dff, 80 + e) for e in range(n_exp)]
    devs, table = _table(blobs, gpu)
    ids, w, rng = _routes(n_tok, k, n_exp, dm + dff)
    x = rng.standard_normal((n_tok, dm)).astype(np.float32)
    want = np.zeros((n_tok, dm), np.float32)
    bound = np.zeros((n_tok, dm), np.float64)
    for t in range(n_tok):
        res = [oracle.q4_0_qmm_forward_bounded(blobs[i], x[t], dm, dff) for i in ids[t]]
        want[t] = oracle.combine_outputs(np.stack([r[0] for r in res]), w[t])
        bound[t] = sum(float(w[t, i]) * res[i][1].astype(np.float64) for i in range(k))
    got = mer.moe_grouped(mer.WeightDtype.Q4_0, dm, dff, table, to_dev(ids, gpu), to_dev(w, gpu), to_dev(x, gpu),
                          qmm=True).cpu().numpy()
    assert_qmm_close(got, want, bound, "grouped tiles qmm")
    mer.take_device_status()
    del devs


def test_tiles_extreme_inputs(mer, oracle, gpu):
    """Vectors of very different sizes, elements far below their vector's
    largest one, and non-finite vectors: relative to each token's largest
    output the error stays that of f32 sums (1e-5, K = 256 and 128 terms), and
    a non-finite input makes its own token's outputs NaN and no others."""
    dm, dff, n_tok = 256, 128, 40
    say("grouped tiles extreme inputs")
    blobs = [make_expert(oracle, Q8, dm, dff, 90)]
    devs, table = _table(blobs, gpu)
    rng = np.random.default_rng(4)
    x = rng.standard_normal((n_tok, dm)).astype(np.float32)
    x[:8] *= np.float32(2.0) ** np.arange(-40, -8, 4, dtype=np.float32)[:, None]
    x[8:16] *= np.float32(2.0) ** rng.integers(-30, 1, (8, dm)).astype(np.float32)
    x[16] = 0.0
    x[17, 5], x[18, 200] = np.inf, np.nan
    ids = np.zeros((n_tok, 1), np.int32)
    w = np.ones((n_tok, 1), np.float32)
    got = mer.moe_grouped(mer.WeightDtype.Q8_0, dm, dff, table, to_dev(ids, gpu), to_dev(w, gpu),
                          to_dev(x, gpu)).cpu().numpy()
    assert np.isnan(got[17:19]).all()
    assert (got[16] == 0).all()
    for t in [t for t in range(n_tok) if t not in (16, 17, 18)]:
        want = oracle.q8_0_direct_forward(blobs[0], x[t], dm, dff)[1].astype(np.float64)
        assert np.isfinite(got[t]).all(), t
        assert np.abs(got[t] - want).max() <= 1e-5 * np.abs(want).max(), t
    mer.take_device_status()
    del devs


@pytest.mark.parametrize("table_len,n_tok,k", [(1, 5, 1), (1024, 171, 6), (1025, 170, 6), (4096, 200, 7)])
def test_grouping_sparse_table(mer, oracle, gpu, table_len, n_tok, k):
    """Grouping with one and several experts and pairs per thread: absent
    entries, negative ids and ids past the table are misses, zero-weight
    slots are skipped whatever their id."""
    dm = dff = 64
    say(f"grouping table={table_len} tokens={n_tok} k={k}")
    blobs = [make_expert(oracle, Q8, dm, dff, 30 + e) for e in range(3)]
    devs, base = _table(blobs, gpu)
    rng = np.random.default_rng(table_len)
    kind = np.arange(table_len) % 4  # 3: absent
    table = torch.where(torch.from_numpy(kind == 3).to(gpu), torch.zeros(1, dtype=torch.int64, device=gpu),
                        base[torch.from_numpy(kind % 3).to(gpu)])
    ids = rng.integers(-2, table_len + 2, (n_tok, k)).astype(np.int32)
    w = rng.random((n_tok, k)).astype(np.float32) + np.float32(0.1)
    w[rng.random((n_tok, k)) < 0.2] = 0.0
    x = rng.standard_normal((n_tok, dm)).astype(np.float32)
    want = np.zeros((n_tok, dm), np.float32)
    for t in range(n_tok):
        valid = [j for j in range(k) if 0 <= ids[t, j] < table_len and kind[ids[t, j]] != 3 and w[t, j] != 0]
        if valid:
            ys = [oracle.q8_0_direct_forward(blobs[kind[ids[t, j]] % 3], x[t], dm, dff)[1] for j in valid]
            want[t] = oracle.combine_outputs(np.stack(ys), w[t, valid])
    got = mer.moe_grouped(mer.WeightDtype.Q8_0, dm, dff, table, to_dev(ids, gpu), to_dev(w, gpu), to_dev(x, gpu))
    got = got.cpu().numpy()
    missed = (w != 0) & ((ids < 0) | (ids >= table_len) | (kind[np.clip(ids, 0, table_len - 1)] == 3))
    if missed.any():
        with pytest.raises(mer.GpuExpertDispatchError):
            mer.take_device_status()
    mer.take_device_status()
    assert_ffn_close(got, want, "sparse table")
    del devs
