"""The router on batches large enough for its matrix kernel (tokens * experts
>= 40000): ends of token, expert and k tiles, d_model not a multiple of four,
and every register width of the selection."""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_router import dev, routing, say  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_experts,d_model,top_k,opts,n_tok", [
    (20, 132, 4, {}, 2049),                  # one token past a tile, experts inside one, k past a stage
    (1024, 130, 8, {}, 40),                  # d_model % 4 = 2
    (257, 3, 5, {}, 160),                    # one expert past a tile, less than one load of k
    (8, 64, 2, {}, 5003),                    # half a stage
    (128, 1031, 8, dict(sigmoid=True, n_group=8, topk_group=3, scaling=2.5), 320),  # nine stages, d_model % 4 = 3
    (200, 2048, 6, dict(sigmoid=True, normalise=False), 200),
])
def test_router_batches(mer, oracle, gpu, n_experts, d_model, top_k, opts, n_tok):
    say(f"router batch E={n_experts} dm={d_model} k={top_k} {opts} tokens={n_tok}")
    r = routing(mer)
    rng = np.random.default_rng(n_experts + d_model)
    w = (rng.standard_normal((n_experts, d_model)) * 0.05).astype(np.float32)
    x = rng.standard_normal((n_tok, d_model)).astype(np.float32)
    x[n_tok // 2] = np.nan  # its own row only: uniform or no eligible expert
    ids, ws, lg = r.route_linear_gate_gpu(dev(w, gpu), dev(x, gpu), top_k, return_logits=True, **opts)
    ids, ws, lg = ids.cpu().numpy(), ws.cpu().numpy(), lg.cpu().numpy()
    ok = np.arange(n_tok) != n_tok // 2
    want = x.astype(np.float64) @ w.astype(np.float64).T
    # at most 16 + 8 + d_model / 1024 + 8 roundings of 2^-24 on the way to a sum
    bar = (33 + d_model / 1024) * 2.0**-24 * (np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T)
    assert (np.abs(lg[ok] - want[ok]) <= bar[ok]).all()
    assert np.isnan(lg[~ok]).all()
    for t in [0, 1, 31, 32, n_tok // 2, n_tok - 2, n_tok - 1]:
        want_ids, want_ws = oracle.gate_route_ex(lg[t], top_k, **opts)
        assert list(ids[t][:len(want_ids)]) == list(want_ids), f"ids token {t}"
        assert (ids[t][len(want_ids):] == -1).all()
        assert np.allclose(ws[t][:len(want_ws)], want_ws, rtol=1e-5, atol=1e-7), f"weights token {t}"


@pytest.mark.parametrize("d_model", [64, 200, 384, 1031, 2048, 7168])
def test_equal_rows_have_equal_logits(mer, gpu, d_model):
    """A logit depends on its token and its gate row alone, not on the tile
    that they fall in: copies of a token, and experts with the same gate row,
    get the same bits, so their ties go to the lower id in every tile."""
    say(f"router equal rows dm={d_model}")
    r = routing(mer)
    rng = np.random.default_rng(d_model)
    n_tok, n_experts, period = 1030, 99, 33
    base_w = (rng.standard_normal((period, d_model)) * 0.05).astype(np.float32)
    base_x = rng.standard_normal((5, d_model)).astype(np.float32)
    w, x = np.tile(base_w, (n_experts // period, 1)), np.tile(base_x, (n_tok // 5, 1))
    ids, ws, lg = r.route_linear_gate_gpu(dev(w, gpu), dev(x, gpu), 3, return_logits=True)
    ids, ws, lg = ids.cpu().numpy(), ws.cpu().numpy(), lg.cpu().numpy()
    want = lg[:5, :period]
    assert (lg.reshape(-1, 5, n_experts // period, period) == want[None, :, None, :]).all()
    best = want.argmax(1)
    assert (ids.reshape(-1, 5, 3) == best[None, :, None] + period * np.arange(3)).all()
    assert (ws.reshape(-1, 5, 3) == ws[:5]).all()
