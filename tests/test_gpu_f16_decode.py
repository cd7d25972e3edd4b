"""f16 views on the decode kernel (mer_hip_expert_batch_f16): the same
products and sums as the f32 routed forward of one-slot tokens, so row i is
that forward's row rounded to f16, bit for bit.

Sizes: one block pair, odd numbers of 64-column chunks, one and several
passes of the packing items, gate/up in one slice and in two (paired
workgroups), down rows in several slices, one expert and more than a
wave's worth of rows."""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_decode_geometry import SHAPES as VARIANTS  # noqa: E402
from test_gpu_decode_geometry import _plan  # noqa: E402
from test_gpu_parity import Q4, Q8, _table, make_expert, randn, say, to_dev  # noqa: E402

pytestmark = pytest.mark.gpu

SHAPES = [(Q4, 64, 64, 1), (Q8, 64, 128, 3), (Q4, 192, 320, 5), (Q8, 576, 64, 2), (Q4, 1024, 5120, 2), (Q4, 2048, 768, 8),
          (Q8, 2048, 768, 9), (Q8, 4160, 128, 4)]
# every instance of the kernel's f16 mode, by format, lane groups and pairing
SHAPES += [(dt, dm, dff, n * k) for dt in (Q4, Q8) for dm, dff, n, k in VARIANTS]


def test_shapes_reach_every_variant():
    assert {_plan(dm, dff, n * k, 1) for dm, dff, n, k in VARIANTS} == set(VARIANTS.values())


@pytest.mark.parametrize("dtype,dm,dff,n", SHAPES)
def test_f16_rows_are_the_rounded_f32_rows(mer, oracle, gpu, dtype, dm, dff, n):
    say(f"f16 decode dtype={dtype} {dm}x{dff} n={n}")
    blobs = [make_expert(oracle, dtype, dm, dff, 11 + e) for e in range(3)]
    devs, table = _table(blobs, gpu)
    ids = torch.from_numpy(np.arange(n, dtype=np.int32) % 3).to(gpu)
    x16 = (randn(dm, 17) * 0.5).astype(np.float16)
    x32 = to_dev(np.tile(x16.astype(np.float32), (n, 1)), gpu)
    want = mer.moe_forward(mer.WeightDtype(dtype), dm, dff, table, ids.view(n, 1),
                           torch.ones((n, 1), dtype=torch.float32, device=gpu), x32).view(n, dm).half()
    # an input on an odd f16 boundary
    flat = to_dev(np.concatenate([np.zeros(1, np.float16), x16]), gpu)
    got = mer.routed_expert_matmul_batch(mer.WeightDtype(dtype), dm, dff, table, ids, flat[1:])
    # the output on the input: row n - 1 of out holds x
    out = torch.zeros((n, dm), dtype=torch.float16, device=gpu)
    out[n - 1] = flat[1:]
    mer.routed_expert_matmul_batch(mer.WeightDtype(dtype), dm, dff, table, ids, out[n - 1], out=out)
    torch.cuda.synchronize()
    mer.take_device_status()
    assert torch.equal(got, want)
    assert torch.equal(out, want)
    del devs
