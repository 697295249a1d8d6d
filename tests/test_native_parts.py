"""Which parts of the package need which native library: plans and the transposing kernel run on libspatha.so alone, the operator and
the layers need the PyTorch extension and say so."""
import sys

import pytest
import torch

from venom_amd import spatha


@pytest.fixture
def without_extension(monkeypatch):
    monkeypatch.setitem(sys.modules, "venom_amd._spatha_torch", None)       # importing it raises ImportError
    import venom_amd
    monkeypatch.delattr(venom_amd, "_spatha_torch", raising=False)
    monkeypatch.setattr(spatha, "_loaded_extension", None)
    monkeypatch.setattr(spatha, "_extension_absent", False, raising=False)


def test_plans_and_transpose_do_not_ask_for_the_extension(without_extension):
    with pytest.raises(RuntimeError, match="not built or does not load"):
        spatha.clear_plan_cache()
    with pytest.raises(ValueError, match="must be a tensor on the GPU"):        # the general path's own check
        spatha.transpose(torch.zeros(8, 8).half())


def test_with_the_extension_they_use_it():
    assert spatha._native("plan_run") is spatha._extension().plan_run and spatha._native("transpose") is spatha._extension().transpose


@pytest.mark.gpu
def test_plans_and_transpose_run_without_the_extension(gpu, without_extension):
    import numpy as np
    from venom_amd import format as F

    vals, meta, columns = F.synthetic_vnm(64, 128, 2, 8, 64, seed=1)
    dev = lambda a: torch.from_numpy(a).to(gpu)
    plan = spatha.SpmmPlan(dev(vals), dev(meta.view(np.int32)), dev(columns.view(np.int32)), 64, 128, 2, 8, 64)
    B = torch.randn(128, 24, device=gpu).half()
    dense = torch.from_numpy(F.decode(vals, meta, columns, 64, 128, 2, 8, 64)).float()
    got = plan.run(B).float().cpu()
    assert (got - dense @ B.float().cpu()).norm() <= 1.2e-3 * got.norm()          # one rounding to fp16
    assert torch.equal(spatha.transpose(B), B.T)
    # a norm that hands its feature-major copy on (to whatever reads it) asks for none either
    from venom_amd.bert import SrnmSpmm

    x = B.T.contiguous()
    SrnmSpmm.offer_transposed(x, B)
    assert SrnmSpmm._transposed(x) is B or SrnmSpmm._transposed(x).data_ptr() == B.data_ptr()
