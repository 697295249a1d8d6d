"""GELU in the write-out on every fp16 input: a product of zeros leaves the bias, so that 65536 rows with the bias patterns 0 .. 65535 run
each value through the kernels' activation once.  Against the exact value (64 bits, rounded once to fp16) no result is more than one
step away; the shares that equal it are what the polynomial and the hardware's exponential and reciprocal give."""
import numpy as np
import pytest
import torch

from venom_amd import format as F
from venom_amd import spatha

pytestmark = pytest.mark.gpu


def fp16_steps_apart(a, b):
    def place(x):                   # fp16 values in order, +0 and -0 in one place
        bits = x.view(np.uint16).astype(np.int32)
        return np.where(bits & 0x8000, -(bits & 0x7FFF), bits)
    return np.abs(place(a) - place(b))


@pytest.fixture(scope="module")
def plan_and_operands():
    rows, cols, m, v = 65536, 8, 8, 64
    vals, meta, columns = F.synthetic_vnm(rows, cols, 2, m, v, seed=1)
    dev = lambda a: torch.from_numpy(a).cuda()
    plan = spatha.SpmmPlan(dev(vals), dev(meta.view(np.int32)), dev(columns.view(np.int32)), rows, cols, 2, m, v)
    bias = torch.arange(rows, dtype=torch.int32, device="cuda").to(torch.int16).view(torch.float16)
    return plan, bias, torch.zeros((cols, 8), dtype=torch.float16, device="cuda")


@pytest.mark.parametrize("activation,equal", [("gelu", 0.996), ("gelu_tanh", 0.9999)])
@pytest.mark.parametrize("variant", [0, 8, 11, 18, 23])
@pytest.mark.parametrize("transposed", [False, True])
def test_every_fp16_input(gpu, plan_and_operands, activation, equal, variant, transposed):
    from scipy.special import erfc

    plan, bias, B = plan_and_operands
    out = plan.run(B, bias=bias, transposed_out=transposed, activation=activation, variant=variant).cpu().numpy()
    got = np.ascontiguousarray(out[0] if transposed else out[:, 0])
    x = np.arange(65536, dtype=np.uint16).view(np.float16)
    xd = x.astype(np.float64)
    with np.errstate(all="ignore"):
        want = 0.5 * xd * erfc(-xd / np.sqrt(2)) if activation == "gelu" else \
            xd / (1 + np.exp(-2 * np.sqrt(2 / np.pi) * (xd + 0.044715 * xd ** 3)))
        want = want.astype(np.float16)
    finite = np.isfinite(x)
    assert np.isnan(got[np.isnan(x)]).all() and got[0x7C00] == np.inf
    assert got[0xFC00] == 0 if activation == "gelu" else np.isnan(got[0xFC00])         # -inf: 0, and -inf * 0
    steps = fp16_steps_apart(got[finite], want[finite])
    assert steps.max() <= 1 and (steps == 0).mean() >= equal
