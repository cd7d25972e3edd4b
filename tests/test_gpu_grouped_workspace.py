"""A grouped call that is no larger than an earlier one on its stream leaves
the stream's workspace where it is, whichever kernel and number of K parts
its sizes choose, so graphs captured with the larger call stay valid."""
from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

from test_gpu_parity import say  # noqa: E402

pytestmark = pytest.mark.gpu

BLOCK_BYTES = {4: 18, 5: 34}


def _call(gpu, dtype, dm, dff, n_tok, k, table_len, blob):
    g = torch.Generator(device=gpu).manual_seed(n_tok)
    table = torch.full((table_len,), blob.data_ptr(), dtype=torch.int64, device=gpu)
    ids = torch.randint(0, table_len, (n_tok, k), generator=g, dtype=torch.int32, device=gpu)
    return dict(args=(dm, dff, table, ids, torch.rand((n_tok, k), generator=g, device=gpu),
                      torch.randn((n_tok, dm), generator=g, device=gpu)),
                out=torch.zeros((n_tok, dm), device=gpu))


@pytest.mark.parametrize("dtype,dm,dff,large,small", [
    # 256 x 8 pairs over 140 experts (tiles of 16), then 250 x 8 over 8 (tiles of 64)
    (5, 1024, 1792, (256, 8, 140), [(250, 8, 8), (256, 8, 8), (17, 1, 1)]),
    # down projection in one part, then in two
    (4, 16384, 4160, (1792, 1, 8), [(1728, 1, 8), (1024, 1, 2), (40, 1, 1)]),
])
def test_smaller_calls_keep_the_workspace(mer, gpu, dtype, dm, dff, large, small):
    say(f"workspace after smaller calls dtype={dtype} {dm}x{dff} {large} {small}")
    g = torch.Generator(device=gpu).manual_seed(dm)
    blocks = 3 * dm * dff // 32
    blob = torch.empty((blocks, BLOCK_BYTES[dtype]), dtype=torch.uint8, device=gpu).random_(0, 256, generator=g)
    blob[:, :2] = torch.empty((blocks, 1), device=gpu).uniform_(0.005, 0.01, generator=g).half().view(torch.uint8)
    calls = [_call(gpu, dtype, dm, dff, *c, blob) for c in [large, *small]]
    x = calls[0]["args"][5]
    xs = [torch.randn(x.shape, generator=g, device=gpu) for _ in range(3)]
    want = torch.empty_like(x)
    s = torch.cuda.Stream(device=gpu)
    run = lambda c, out: mer.moe_grouped(mer.WeightDtype(dtype), *c["args"], out=out)
    with torch.cuda.stream(s):
        run(calls[0], calls[0]["out"])
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info(gpu)[0]
    with torch.cuda.stream(s):
        for c in calls[1:]:
            run(c, c["out"])
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info(gpu)[0] == free, "a smaller call made the workspace grow"
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        run(calls[0], calls[0]["out"])
    for i, new in enumerate(xs):
        with torch.cuda.stream(s):
            run(calls[1 + i % len(small)], calls[1 + i % len(small)]["out"])
            x.copy_(new)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            run(calls[0], want)
        torch.cuda.synchronize()
        assert torch.isfinite(want).all() and torch.equal(calls[0]["out"], want), f"replay {i}"
    mer.take_device_status()
    del graph
    mer.stream_release(s)
