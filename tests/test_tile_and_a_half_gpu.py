"""The tile-and-a-half kernel (id 22): k-loops of one, two, three and more steps, whose last steps stand behind the loops, on workgroups
with and without an extra half tile, ragged columns and k tails, both layouts, plain and fused; bit for bit against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from venom_amd import format as F
from venom_amd import spatha

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [128, 256, 384, 1280, 3072])
@pytest.mark.parametrize("cols,m", [(64, 8), (512, 16), (380, 8), (1000, 16), (1280, 16)])          # 1 .. 5 k-steps
@pytest.mark.parametrize("N", [136, 520])
def test_every_length_of_the_k_loop(gpu, rows, cols, m, N):
    print("tile and a half", rows, cols, m, N, flush=True)
    vals, meta, columns = F.synthetic_vnm(rows, cols, 2, m, 128, seed=rows + cols, integer_values=True)
    rng = np.random.default_rng(N)
    B = rng.integers(-4, 5, size=(cols, N)).astype(np.float16)
    bias = rng.integers(-3, 4, size=rows).astype(np.float16)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)).to(gpu)
    plan = spatha.SpmmPlan(dev(vals), dev(meta), dev(columns), rows, cols, 2, m, 128)
    assert "tile_and_a_half" in plan.kernel_name(N, 0, 22)
    dB, dbias = dev(B), dev(bias)
    plain = oracle.spmm(vals, meta, columns, rows, cols, 2, m, 128, B)
    biased = oracle.spmm(vals, meta, columns, rows, cols, 2, m, 128, B, bias=bias, transposed_out=True)
    for kw, want in ((dict(), plain), (dict(bias=dbias, activation="none"), np.ascontiguousarray(biased.T)),
                     (dict(bias=dbias, transposed_out=True), biased), (dict(bias=dbias, transposed_out=True, activation="none"), biased)):
        got = plan.run(dB, variant=22, **kw).cpu().numpy()
        assert np.array_equal(got.view(np.uint16), want.view(np.uint16)), kw
