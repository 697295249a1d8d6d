"""Right-hand sides whose token count is no multiple of 8: the kernels that make the padded copy."""
import pytest
import torch

from venom_amd import _lib, spatha

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 7), (64, 8), (65, 9), (130, 301), (1280, 1037), (63, 4097)])
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_padded_copies(gpu, rows, cols, offset):
    buf = torch.randn(rows * cols + 16, device=gpu).half()
    x = buf[offset:offset + rows * cols].view(rows, cols)
    out = spatha._pad_columns(x)
    assert torch.equal(out, torch.nn.functional.pad(x, (0, -cols % 8)))
    if offset:
        return
    t = torch.full((cols, (rows + 7) // 8 * 8), float("nan"), dtype=torch.float16, device=gpu)
    _lib.check(_lib.lib().spatha_transpose_padded_f16(x.data_ptr(), rows, cols, t.data_ptr(), spatha._stream_ptr(gpu)), "transpose")
    assert torch.equal(t, torch.nn.functional.pad(x.t(), (0, -rows % 8)))


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 7), (64, 8), (65, 9), (130, 301), (1280, 1037), (63, 4097)])
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_cut_results(gpu, rows, cols, offset):
    full = torch.randn(rows, (cols + 7) // 8 * 8, device=gpu).half()
    buf = torch.full((rows * cols + 64,), 7.0, dtype=torch.float16, device=gpu)
    out = buf[8 + offset:8 + offset + rows * cols]
    _lib.check(_lib.lib().spatha_cut_columns_f16(full.data_ptr(), rows, cols, out.data_ptr(), spatha._stream_ptr(gpu)), "cut")
    assert torch.equal(out.view(rows, cols), full[:, :cols])
    assert bool((buf[:8 + offset] == 7.0).all()) and bool((buf[8 + offset + rows * cols:] == 7.0).all())


@pytest.mark.parametrize("rows,cols,v,m", [(64, 96, 64, 8), (128, 70, 128, 16), (1024, 1024, 64, 8), (96, 200, 32, 10), (2048, 512, 32, 16),
                                           (5120, 1280, 128, 16), (5120, 1280, 64, 10), (33024, 256, 64, 4)])
@pytest.mark.parametrize("tokens", [1, 2, 7, 15, 17, 18, 31, 33, 35, 47, 63, 65, 70, 129, 301, 1037])
def test_ragged_products_equal_the_padded_ones(gpu, rows, cols, v, m, tokens):
    """B and C as they lie (where a kernel without 16-byte pieces is chosen) or a padded copy and a cut: bit for bit the padded product,
    nothing written around C, and a NaN or infinity next to a lane's last columns stays where it belongs."""
    from venom_amd import format as F

    vals, meta, columns = F.synthetic_vnm(rows, cols, 2, m, v, seed=tokens)
    plan = spatha.SpmmPlan(torch.from_numpy(vals).to(gpu), torch.from_numpy(meta.view("int32")).to(gpu),
                           torch.from_numpy(columns.view("int32")).to(gpu), rows, cols, 2, m, v)
    gen = torch.Generator(device=gpu).manual_seed(rows + tokens)
    B = torch.randn((cols, tokens), generator=gen, device=gpu).half()
    if tokens > 2:
        B[cols // 2, 0] = float("nan")
        B[cols // 3, tokens // 2] = float("inf")
    bias = torch.randn(rows, generator=gen, device=gpu).half()
    padded = spatha._pad_columns(B)
    act = {} if v == 32 else {"activation": "gelu"}
    for kwargs in ({}, {"transposed_out": True}, {"transposed_out": True, "bias": bias}, {"bias": bias, "activation": "none"}, {"bias": bias, **act},
                   {"bias": bias, "transposed_out": True, **act}):
        if "bias" in kwargs and not kwargs.get("transposed_out") and "activation" not in kwargs:
            continue
        full = plan.run(padded, **kwargs)
        want = full[:tokens] if kwargs.get("transposed_out") else full[:, :tokens]
        got = plan.run(B, **kwargs)
        assert got.is_contiguous() and got.shape == want.shape
        assert torch.equal(got.view(torch.int16), want.contiguous().view(torch.int16)), kwargs
    out = torch.full((rows * tokens + 64,), 7.0, dtype=torch.float16, device=gpu)
    for layout in (0, 1):
        name = plan.kernel_name((tokens + 7) // 8 * 8, out_layout=layout)
        direct = "_direct_tile" in name or "skinny" in name
        large = tokens > 16 and tokens % (2 if tokens <= 32 else 4) and rows // 64 * -(-(-(-cols // m) * 2) // 32) * -(-tokens // 64) > 8000
        for src, pitch, takes in ((B, tokens, direct and not large), (padded, padded.shape[1], direct)):
            if pitch % 8 == 0 and src is B:
                continue
            status = _lib.lib().spatha_spmm_run_ragged(plan._handle, src.data_ptr(), pitch, tokens, None, out[32:].data_ptr(), layout, 0, 0,
                                                       spatha._stream_ptr(gpu))
            assert status == (0 if takes else 3), (name, pitch)
            assert bool((out[:32] == 7.0).all()) and bool((out[32 + rows * tokens:] == 7.0).all())
            if takes:
                want = plan.run(padded, transposed_out=bool(layout))
                want = want[:tokens] if layout else want[:, :tokens].contiguous()
                assert torch.equal(out[32:32 + rows * tokens].view(torch.int16), want.reshape(-1).view(torch.int16))
    with pytest.raises(Exception):
        plan.run(B, bias=bias)              # a bias needs the transposed layout or an activation, ragged or not


@pytest.mark.parametrize("shape", [(1, 128), (301, 128), (3, 5, 128), (2, 8, 128), (1, 2, 3, 128)])
def test_layers_take_any_token_count_and_stride(gpu, shape):
    """The layer's one-call path against the operator on a copy made by torch: token-major, feature-major, strided and sliced
    inputs, twice each (the second call finds the transposed copy of the first), plain and feature-major results, a chain of both."""
    from venom_amd.bert import SrnmSpmm

    torch.manual_seed(0)
    up = SrnmSpmm(torch.nn.Linear(128, 256).half().to(gpu), 2, 8, 64, magnitude=True)
    down = SrnmSpmm(torch.nn.Linear(256, 128, bias=False).half().to(gpu), 2, 16, 32, magnitude=True)

    def direct(layer, x):
        rhs = x.reshape(-1, x.shape[-1]).T.contiguous()
        bias = layer.bias if layer.bias is not None else torch.zeros(layer.nrows_sp, device=gpu).half()
        out = spatha.spmm(layer.metadata, layer.columns, layer.values, rhs, bias, layer.nrows_sp, layer.ncols_sp, rhs.shape[1], layer.v,
                          layer.n, layer.m)
        return out.reshape(*x.shape[:-1], -1)

    base = torch.randn(shape, device=gpu).half()
    wide = torch.randn(*shape[:-1], 256, device=gpu).half()
    tokens = base.numel() // 128
    feature = torch.randn(128, tokens, device=gpu).half().T.reshape(shape)
    with torch.no_grad():
        for x in (base, wide[..., 64:192], feature, torch.nn.Parameter(base.clone())):
            want = direct(up, x)
            for _ in range(2):
                got = up(x)
                assert got.shape == want.shape and torch.equal(got, want)
                mid = up.forward_feature_major(x, "none")
                assert mid.shape == want.shape and torch.equal(mid, want)
                assert torch.equal(down(mid), direct(down, mid.contiguous()))
                # an elementwise pass between the two, and the general path on what the one-call path has kept
                assert torch.equal(down(mid * 2), direct(down, mid.contiguous() * 2))
            assert torch.equal(SrnmSpmm._transposed(torch.flatten(x, 0, -2)), x.detach().reshape(-1, 128).T)
        x = base.clone()
        first = up(x)
        x.mul_(2)                                       # the kept copy is of the old contents
        assert torch.equal(up(x), direct(up, x)) and not torch.equal(up(x), first)


def test_layers_take_feature_major_views_at_any_address(gpu):
    """A feature-major input that starts in the middle of a buffer: a pitch that equals the padded token count does not make it a
    right-hand side that can be read in 16-byte pieces."""
    from venom_amd.bert import SrnmSpmm

    torch.manual_seed(0)
    up = SrnmSpmm(torch.nn.Linear(128, 256).half().to(gpu), 2, 8, 64, magnitude=True)
    down = SrnmSpmm(torch.nn.Linear(256, 128).half().to(gpu), 2, 16, 32, magnitude=True)

    def direct(layer, x):
        return spatha.spmm(layer.metadata, layer.columns, layer.values, x.T.contiguous(), layer.bias, layer.nrows_sp, layer.ncols_sp,
                           x.shape[0], layer.v, layer.n, layer.m)

    with torch.no_grad():
        views = [torch.randn(129, 8, device=gpu).half()[:128, 2:7].T, torch.randn(129, 24, device=gpu).half()[:128, 1:20].T,
                 torch.randn(129, 40, device=gpu).half()[:128, 3:40].T]
        wide = up.forward_feature_major(torch.randn(1037, 128, device=gpu).half())
        for x in views:
            assert x.data_ptr() % 16 != 0
            for _ in range(2):
                assert torch.equal(up(x), direct(up, x))
                assert torch.equal(up.forward_feature_major(x), direct(up, x))
        for first in (1, 3, 5, 8):
            x = wide[first:, :128]
            assert x.stride() == (1, 1040)
            assert torch.equal(up(x), direct(up, x)) and torch.equal(up.forward_feature_major(x), direct(up, x))
        assert torch.equal(down(wide[3:]), direct(down, wide[3:]))
        refused = torch.randn(128 * 24 + 8, device=gpu).half()[1:1 + 128 * 24].view(128, 24).T      # as by the operator: no copy is due
        with pytest.raises(RuntimeError):
            up(refused)


def test_layer_refuses_what_it_refused(gpu):
    from venom_amd.bert import SrnmSpmm

    layer = SrnmSpmm(torch.nn.Linear(128, 64).half().to(gpu), 2, 8, 64)
    with torch.no_grad():
        for x in (torch.randn(4, 128, device=gpu), torch.randn(4, 120, device=gpu).half(), torch.randn(4, 128).half()):
            with pytest.raises((RuntimeError, ValueError, TypeError)):
                layer(x)
        with pytest.raises((RuntimeError, IndexError)):
            layer(torch.randn(128, device=gpu).half())


def test_plan_run_refuses_and_writes_as_before(gpu):
    from venom_amd import format as F

    vals, meta, columns = F.synthetic_vnm(64, 128, 2, 8, 64, seed=1)
    dev = lambda a: torch.from_numpy(a).to(gpu)
    import numpy as np
    plan = spatha.SpmmPlan(dev(vals), dev(meta.view(np.int32)), dev(columns.view(np.int32)), 64, 128, 2, 8, 64)
    B = torch.randn(128, 24, device=gpu).half()
    bias = torch.randn(64, device=gpu).half()
    out = torch.empty(64, 24, device=gpu).half()
    version = out._version
    assert plan.run(B, out=out) is out and out._version > version and torch.equal(out, plan.run(B))
    with torch.inference_mode():
        assert torch.equal(plan.run(B), out)
    for bad, error in ((dict(B=B.float()), TypeError), (dict(B=B.cpu()), ValueError), (dict(B=B.T), ValueError),
                       (dict(B=B, out=out.T), ValueError), (dict(B=B, out=out[:, :16].contiguous()), ValueError),
                       (dict(B=B, bias=bias[:32], transposed_out=True), ValueError), (dict(B=B, bias=bias), RuntimeError),
                       (dict(B=B, variant=99), RuntimeError), (dict(B=B, activation="relu6"), ValueError), (dict(B=[1]), ValueError)):
        with pytest.raises(error):
            plan.run(**bad)


@pytest.mark.parametrize("rows,cols,m,v", [(64, 64, 8, 64), (128, 200, 16, 128), (256, 1024, 8, 64), (1024, 3300, 10, 128), (128, 12288, 16, 64),
                                           (32, 64, 8, 32), (96, 300, 7, 96), (512, 2048, 16, 32), (512, 4096, 16, 32)])
@pytest.mark.parametrize("tokens", [1, 2, 5, 8, 13, 16])
def test_a_few_tokens_as_they_lie(gpu, rows, cols, m, v, tokens):
    """spatha_spmm_run_tokens against the oracle, bit for bit on integer operands (eight and sixteen waves on 64-row and 32-row tiles),
    with and without a bias; one token more than it
    takes, and more columns than the LDS holds, are refused."""
    import numpy as np

    import oracle
    from venom_amd import format as F

    vals, meta, columns = F.synthetic_vnm(rows, cols, 2, m, v, seed=rows + tokens, integer_values=True)
    rng = np.random.default_rng(cols)
    x = rng.integers(-4, 5, size=(tokens, cols)).astype(np.float16)
    bias = rng.integers(-3, 4, size=rows).astype(np.float16)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)).to(gpu)
    plan = spatha.SpmmPlan(dev(vals), dev(meta), dev(columns), rows, cols, 2, m, v)
    dx, dbias = dev(x), dev(bias)
    L = _lib.lib()
    for b in (None, dbias):
        out = torch.full((tokens, rows), float("nan"), dtype=torch.float16, device=gpu)
        status = L.spatha_spmm_run_tokens(plan._handle, dx.data_ptr(), tokens, None if b is None else b.data_ptr(), out.data_ptr(),
                                          spatha._stream_ptr(gpu))
        if tokens * cols > 63 * 1024:
            assert status == 3
            continue
        assert status == 0
        want = oracle.spmm(vals, meta, columns, rows, cols, 2, m, v, np.ascontiguousarray(x.T), bias=None if b is None else bias,
                           transposed_out=True)
        assert np.array_equal(out.cpu().numpy().view(np.uint16), want.view(np.uint16))
    assert L.spatha_spmm_run_tokens(plan._handle, dx.data_ptr(), 17, None, dx.data_ptr(), spatha._stream_ptr(gpu)) == 3


def test_a_ragged_product_allocates_for_the_route_it_takes(gpu):
    """A result, and for the staged kernels the padded right-hand side and, row-major, the cut copy: nothing for the routes not taken."""
    from venom_amd import format as F

    def allocations(call):
        call()
        before = torch.cuda.memory_stats(gpu)["allocation.all.allocated"]
        call()
        return torch.cuda.memory_stats(gpu)["allocation.all.allocated"] - before

    for rows, cols, v, m, tokens, staged in [(5120, 1280, 64, 10, 1037, True), (1024, 1024, 64, 8, 187, False), (49152, 256, 64, 4, 1037, True)]:
        vals, meta, columns = F.synthetic_vnm(rows, cols, 2, m, v, seed=tokens)
        arrays = [torch.from_numpy(a.view("int32") if a.dtype != "float16" else a).to(gpu) for a in (vals, meta, columns)]
        plan = spatha.SpmmPlan(*arrays, rows, cols, 2, m, v)
        B, bias = torch.randn((cols, tokens), device=gpu).half(), torch.randn(rows, device=gpu).half()
        name = plan.kernel_name((tokens + 7) // 8 * 8)
        assert staged == ("_direct_tile" not in name and "skinny" not in name), name
        assert allocations(lambda: plan.run(B)) == (3 if staged else 1)
        assert allocations(lambda: plan.run(B, transposed_out=True)) == (2 if staged else 1)
        assert allocations(lambda: spatha.spmm(arrays[1], arrays[2], arrays[0], B, bias, rows, cols, tokens, v, 2, m)) == (2 if staged else 1)
        assert [_lib.lib().spatha_spmm_ragged_route(plan._handle, tokens, layout, 0) for layout in (0, 1)] == ([0, 0] if staged else [2, 2])


@pytest.mark.parametrize("v,tokens", [(64, 17), (64, 24), (32, 17)])
def test_refusals_carry_their_status(gpu, v, tokens):
    """A bias at an address that the kernels do not read: the same error for ragged counts as for others."""
    from venom_amd import format as F

    vals, meta, columns = F.synthetic_vnm(128, 128, 2, 8, v, seed=1)
    plan = spatha.SpmmPlan(torch.from_numpy(vals).to(gpu), torch.from_numpy(meta.view("int32")).to(gpu),
                           torch.from_numpy(columns.view("int32")).to(gpu), 128, 128, 2, 8, v)
    bias = torch.zeros(136, dtype=torch.float16, device=gpu)[1:129]
    with pytest.raises(_lib.SpathaError) as refused:
        plan.run(torch.zeros((128, tokens), dtype=torch.float16, device=gpu), bias, transposed_out=True)
    assert refused.value.status == _lib.ERR_BAD_ARGUMENT
