"""Results of 96 MB and more leave by non-temporal stores: every kernel id that accepts a shape, both layouts, against the same product in
two column halves, which do not (small whole numbers, so that the order of the sums does not matter); and the layers' entry point,
which keeps the ordinary stores at any size."""
import ctypes

import pytest
import torch

from venom_amd import _lib, spatha
from venom_amd import format as F

pytestmark = pytest.mark.gpu


def make_plan(rows, cols, v, m, device):
    vals, meta, columns = F.synthetic_vnm(rows, cols, 2, m, v, seed=5, integer_values=True)
    return spatha.SpmmPlan(torch.from_numpy(vals).to(device), torch.from_numpy(meta.view("int32")).to(device),
                           torch.from_numpy(columns.view("int32")).to(device), rows, cols, 2, m, v)


@pytest.mark.parametrize("rows,cols,v,m,tokens", [(4096, 256, 64, 8, 12288), (4096, 512, 128, 16, 12304), (4096, 512, 64, 16, 12296), (4096, 256, 32, 8, 12288),
                                                  (4096, 512, 32, 16, 12312), (24576, 512, 128, 20, 2048), (24576, 1024, 128, 16, 2064)])
def test_streamed_results_equal_the_halves(gpu, rows, cols, v, m, tokens):
    assert rows * tokens * 2 >= 96 << 20
    plan = make_plan(rows, cols, v, m, gpu)
    gen = torch.Generator(device=gpu).manual_seed(rows + m)
    B = torch.randint(-4, 5, (cols, tokens), generator=gen, device=gpu).half()
    cut = tokens // 16 * 8
    halves = [B[:, :cut].contiguous(), B[:, cut:].contiguous()]
    want = torch.cat([plan.run(h) for h in halves], dim=1)
    ran = 0
    for variant in [0] + spatha.variant_ids():
        if variant and plan.kernel_name(tokens, variant=variant) is None:
            continue
        print(plan.kernel_name(tokens, variant=variant), flush=True)
        try:
            assert torch.equal(plan.run(B, variant=variant), want), variant
        except _lib.SpathaError:          # accepted by the shape checks, refused by the kernel's launcher
            continue
        assert torch.equal(plan.run(B, transposed_out=True, variant=variant), want.t()), variant
        ran += 1
    assert ran >= 3
    out = torch.empty_like(want)
    stream = ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)
    _lib.check(_lib.lib().spatha_spmm_run_layer(plan._handle, B.data_ptr(), tokens, None, out.data_ptr(), 0, 0, None, 0, stream), "run_layer")
    assert torch.equal(out, want)


@pytest.mark.parametrize("rows,cols,v,m,tokens", [(4096, 256, 64, 8, 12320), (4096, 512, 64, 16, 12320), (4096, 512, 64, 32, 12320),
                                                  (4096, 512, 128, 16, 12320), (4096, 512, 128, 32, 12320), (24576, 1024, 128, 16, 2080),
                                                  (12288, 8192, 128, 8, 4128), (4096, 512, 32, 16, 12320)])
def test_streamed_results_with_bias_and_activation(gpu, rows, cols, v, m, tokens):
    """The write-outs that add a bias or apply an activation, where the last tile column is partly empty: the same bits as in two column
    halves, whose stores are ordinary (every kernel that can be chosen adds up whole numbers exactly)."""
    plan = make_plan(rows, cols, v, m, gpu)
    gen = torch.Generator(device=gpu).manual_seed(cols + m)
    B = torch.randint(-4, 5, (cols, tokens), generator=gen, device=gpu).half()
    bias = torch.randint(-3, 4, (rows,), generator=gen, device=gpu).half()
    cut = tokens // 64 * 32
    halves = [B[:, :cut].contiguous(), B[:, cut:].contiguous()]
    kinds = [{"bias": bias, "transposed_out": True}, {"bias": bias, "activation": "none"}, {"bias": bias, "activation": "none", "transposed_out": True}]
    if v != 32:
        kinds += [{"bias": bias, "activation": "gelu"}, {"bias": bias, "activation": "gelu_tanh", "transposed_out": True}, {"activation": "gelu"}]
    for kwargs in [{}] + kinds:
        print(plan.kernel_name(tokens, int(bool(kwargs.get("transposed_out")))), sorted(k for k in kwargs), flush=True)
        want = torch.cat([plan.run(h, **kwargs) for h in halves], dim=0 if kwargs.get("transposed_out") else 1)
        got = plan.run(B, **kwargs)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), kwargs
