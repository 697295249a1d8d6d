"""The order in which the kernels walk their tiles: whatever it is, every tile lands where it belongs.  Row-major launches
with a multiple of eight tile columns give each XCD every eighth column; one column more or less, and transposed output, take
adjacent columns.  Every kernel id that accepts the shape, integer operands, bit-exact against the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle
from venom_amd import format as F
from venom_amd import spatha

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("v,m", [(64, 8), (128, 16), (64, 12), (32, 16), (32, 8)])
@pytest.mark.parametrize("N", [2048, 4096, 2056, 1920])      # 8 / 16 columns of 256 and 16 / 32 of 128; 9 and 17; 8 and 15
@pytest.mark.parametrize("transposed", [False, True])
def test_every_kernel_places_its_tiles(gpu, v, m, N, transposed):
    rows, cols = 1536, 16 * m * 3 - 5
    vals, meta, columns = F.synthetic_vnm(rows, cols, 2, m, v, seed=4, integer_values=True)
    rng = np.random.default_rng(5)
    B = rng.integers(-4, 5, size=(cols, N)).astype(np.float16)
    bias = rng.integers(-3, 4, size=rows).astype(np.float16) if transposed else None
    want = oracle.spmm(vals, meta, columns, rows, cols, 2, m, v, B, bias=bias, transposed_out=transposed)

    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)).to(gpu)

    plan = spatha.SpmmPlan(dev(vals), dev(meta), dev(columns), rows, cols, 2, m, v)
    dB, dbias = dev(B), None if bias is None else dev(bias)
    ran = 0
    for variant in range(spatha.num_variants()):
        name = plan.kernel_name(N, 1 if transposed else 0, variant)
        if name is None:
            continue
        print(rows, cols, N, m, v, transposed, variant, name, flush=True)
        got = plan.run(dB, bias=dbias, transposed_out=transposed, variant=variant)
        assert np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16)), name
        ran += 1
    assert ran > 1
