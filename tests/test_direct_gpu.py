"""The kernels that read their operands without LDS staging (id 13, id 23 and the 32-row form for V = 32, 96, ...): every column
width and wave count their launch can choose, on integer operands bit for bit against the oracle - one row tile and many, k-loops
shorter than the waves that share them, ragged columns and k tails, both layouts, bias and fused bias."""
import numpy as np
import pytest
import torch

import oracle
from venom_amd import format as F
from venom_amd import spatha

pytestmark = pytest.mark.gpu

CASES = [
    # rows, cols, N, m, v
    (64, 64, 8, 8, 64), (64, 300, 72, 7, 64), (256, 2048, 8, 16, 64), (128, 3300, 104, 16, 128), (1280, 5120, 304, 16, 128),
    (1024, 4096, 512, 32, 128), (1024, 1024, 520, 16, 64), (768, 3072, 1040, 32, 64), (1024, 1024, 1040, 20, 128),
    (1536, 640, 304, 20, 64), (4096, 512, 200, 16, 64), (4096, 1024, 512, 8, 64), (17408, 512, 16, 8, 64), (17408, 256, 32, 8, 64),
    (35072, 512, 8, 16, 128), (35072, 512, 64, 16, 128), (1024, 16384, 64, 8, 128),
    (32, 64, 8, 8, 32), (96, 300, 72, 7, 96), (160, 2048, 136, 16, 32), (1280, 5120, 304, 16, 32), (1024, 4096, 520, 8, 32),
    (1280, 4352, 520, 16, 64), (256, 4096, 136, 16, 32), (1024, 2048, 136, 16, 32), (1024, 1536, 264, 16, 32),
    (1024, 2048, 1040, 16, 32), (2112, 640, 264, 20, 32), (9216, 512, 8, 16, 32), (9216, 320, 32, 8, 288), (9216, 256, 64, 16, 32),
]


def test_the_cases_reach_every_form(gpu):
    """Eight forms on 64-row tiles and eight on 32-row ones: columns and waves per tile as the kernel's name reports them."""
    reached = set()
    for rows, cols, N, m, v in CASES:
        vals, meta, columns = F.synthetic_vnm(rows, cols, 2, m, v, seed=1)
        plan = spatha.SpmmPlan(torch.from_numpy(vals).to(gpu), torch.from_numpy(meta.view(np.int32)).to(gpu),
                               torch.from_numpy(columns.view(np.int32)).to(gpu), rows, cols, 2, m, v)
        reached.add(plan.kernel_name(N, 0, spatha.DIRECT_HALF_VARIANT if v % 64 else 23).split("direct_")[1])
    columns_and_waves = ("x16_splitk4", "x16_splitk8", "x16_splitk16", "x32_splitk4", "x32_splitk8", "x64_splitk4", "x64_splitk4_lean",
                         "x64_splitk8")
    assert reached == {tile + form for tile in ("tile64", "tile32") for form in columns_and_waves}, sorted(reached)


@pytest.mark.parametrize("rows,cols,N,m,v", CASES)
@pytest.mark.parametrize("transposed", [False, True])
def test_direct_kernels_bit_exact(gpu, rows, cols, N, m, v, transposed):
    print("direct", rows, cols, N, m, v, transposed, flush=True)
    vals, meta, columns = F.synthetic_vnm(rows, cols, 2, m, v, seed=rows + N, integer_values=True)
    rng = np.random.default_rng(N)
    B = rng.integers(-4, 5, size=(cols, N)).astype(np.float16)
    bias = rng.integers(-3, 4, size=rows).astype(np.float16)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)).to(gpu)
    plan = spatha.SpmmPlan(dev(vals), dev(meta), dev(columns), rows, cols, 2, m, v)
    name = plan.kernel_name(N, int(transposed), 0)
    assert "direct_tile" in name or "skinny" in name, name
    want = oracle.spmm(vals, meta, columns, rows, cols, 2, m, v, B, bias=bias if transposed else None, transposed_out=transposed)
    guarded = torch.full((cols * N + 4096,), float("nan"), dtype=torch.float16, device=gpu)
    guarded[:cols * N] = dev(B).reshape(-1)
    dB = guarded[:cols * N].view(cols, N)
    variants = [0, 23 if v % 64 == 0 else spatha.DIRECT_HALF_VARIANT]
    for variant in variants:
        got = plan.run(dB, bias=dev(bias) if transposed else None, transposed_out=transposed, variant=variant)
        assert np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16)), variant
    fused = plan.run(dB, bias=dev(bias), transposed_out=transposed, activation="none")
    want_b = oracle.spmm(vals, meta, columns, rows, cols, 2, m, v, B, bias=bias, transposed_out=True)
    want_b = want_b if transposed else np.ascontiguousarray(want_b.T)
    assert np.array_equal(fused.cpu().numpy().view(np.uint16), want_b.view(np.uint16))


# (the kernel named last is the automatic choice)  V = 32 beyond four tiles per CU: 16 and 17, 29, 30 and 93 k-steps at both ends of the column counts that go to 32-row tiles
LONG_CASES = [(12288, 2720, 136, 10, 32, 24), (12288, 2560, 136, 10, 32, 16), (12288, 2880, 192, 10, 32, 24), (12288, 2880, 200, 10, 32, 16),
              (12288, 4640, 264, 10, 32, 24), (12288, 4800, 384, 10, 32, 24), (12288, 4800, 256, 10, 32, 14), (12288, 4800, 392, 10, 32, 14),
              (12288, 14880, 256, 10, 32, 24), (12288, 14880, 392, 10, 32, 15),
              # one step into a second round of 64 x 128 tiles, B beyond 4 MB: 8 3/4 tiles per CU and more; four k-steps
              (1280, 4096, 3528, 16, 32, 24), (1280, 4096, 3592, 16, 32, 16), (1280, 2048, 3528, 32, 32, 16),
              # V = 64: 16 k-steps and 15, 32
              (36864, 4096, 72, 16, 64, 23), (36864, 3840, 72, 16, 64, 4), (36864, 8192, 72, 16, 64, 23),
              # V = 128: 32, 24 and 23, 96, 48 and 26 k-steps (kernel 20 goes with row-major output, 6 with transposed)
              (12288, 8192, 640, 16, 128, 20), (24576, 6144, 264, 16, 128, 22), (24576, 5888, 264, 16, 128, 20),
              (12288, 12288, 640, 8, 128, 12), (36864, 4096, 1024, 10, 128, 22)]


@pytest.mark.parametrize("rows,cols,N,m,v,kernel", LONG_CASES)
def test_many_tiles_with_long_k_loops(gpu, rows, cols, N, m, v, kernel):
    """The automatic choice is the kernel named last, and its result is the oracle's on rows of the first, a middle and the last V block."""
    print("long", rows, cols, N, m, v, flush=True)
    vals, meta, columns = F.synthetic_vnm(rows, cols, 2, m, v, seed=N, integer_values=True)
    B = np.random.default_rng(N).integers(-2, 3, size=(cols, N)).astype(np.float16)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)).to(gpu)
    plan = spatha.SpmmPlan(dev(vals), dev(meta), dev(columns), rows, cols, 2, m, v)
    for transposed in (False, True):
        named = 6 if kernel == 20 and transposed else kernel
        assert plan.kernel_name(N, int(transposed), 0) == plan.kernel_name(N, int(transposed), named)
    got = plan.run(dev(B)).cpu().numpy()
    turned = plan.run(dev(B), transposed_out=True).cpu().numpy()
    assert np.array_equal(turned.T.view(np.uint16), got.view(np.uint16))
    # whole matrices of one V block each: their part of the storage arrays
    blocks, groups = rows // v, len(columns) // (rows // v)
    for block in (0, blocks // 2 + 1, blocks - 1):
        part = lambda a: np.ascontiguousarray(a.reshape(blocks, -1)[block])
        want = oracle.spmm(part(vals), part(meta), part(columns), v, cols, 2, m, v, B)
        assert np.array_equal(got[block * v:(block + 1) * v].view(np.uint16), want.view(np.uint16)), block


def test_direct_kernel_activations(gpu):
    """GELU in the write-out: one rounding of the exact value of the rounded, biased sum (at most one step of fp16 apart)."""
    rows, cols, N, m, v = 256, 512, 136, 8, 64
    vals, meta, columns = F.synthetic_vnm(rows, cols, 2, m, v, seed=1, value_std=0.3)
    rng = np.random.default_rng(2)
    B = rng.standard_normal((cols, N)).astype(np.float16)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)).to(gpu)
    plan = spatha.SpmmPlan(dev(vals), dev(meta), dev(columns), rows, cols, 2, m, v)
    bias = dev(rng.standard_normal(rows).astype(np.float16))
    for transposed in (False, True):
        pre = plan.run(dev(B), bias=bias, transposed_out=transposed, activation="none", variant=23).double()
        for act, approx in (("gelu", "none"), ("gelu_tanh", "tanh")):
            got = plan.run(dev(B), bias=bias, transposed_out=transposed, activation=act, variant=23)
            want = torch.nn.functional.gelu(pre, approximate=approx).half()
            # one step of fp16 at the value's size (2^-10 relative, the subnormal step 2^-24 near zero)
            assert bool(((got.double() - want.double()).abs() <= want.double().abs() * 2.0 ** -10 + 2.0 ** -24).all())


def test_the_32_row_kernel_by_name(gpu):
    """Kernel 24 on random shapes of V = 32, 96 and 160, in every mode, whatever the automatic choice is; tune knows it; plans of 64-row
    tiles refuse it."""
    assert spatha.variant_ids() == list(range(1, spatha.num_variants())) + [24]
    rng = np.random.default_rng(17)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)).to(gpu)
    for i in range(24):
        v, m = int(rng.choice([32, 96, 160])), int(rng.choice([4, 7, 8, 10, 16, 20, 40]))
        rows, cols, N = v * int(rng.integers(1, 9)), int(rng.integers(4, 1500)), 8 * int(rng.integers(1, 200))
        print("by name", i, rows, cols, N, m, v, flush=True)
        vals, meta, columns = F.synthetic_vnm(rows, cols, 2, m, v, seed=i, integer_values=True)
        B = rng.integers(-4, 5, size=(cols, N)).astype(np.float16)
        bias = rng.integers(-3, 4, size=rows).astype(np.float16)
        plan = spatha.SpmmPlan(dev(vals), dev(meta), dev(columns), rows, cols, 2, m, v)
        plain = oracle.spmm(vals, meta, columns, rows, cols, 2, m, v, B)
        biased = oracle.spmm(vals, meta, columns, rows, cols, 2, m, v, B, bias=bias, transposed_out=True)
        for kw, want in ((dict(), plain), (dict(bias=dev(bias), transposed_out=True), biased),
                         (dict(bias=dev(bias), activation="none"), np.ascontiguousarray(biased.T))):
            got = plan.run(dev(B), variant=24, **kw).cpu().numpy()
            assert np.array_equal(got.view(np.uint16), want.view(np.uint16)), kw
    out = torch.empty((rows, N), dtype=torch.float16, device=gpu)
    best, best_ms, auto_ms, times = plan.tune(dev(B), out)
    assert best in times and best_ms == min(times.values()) <= auto_ms
    vals, meta, columns = F.synthetic_vnm(64, 64, 2, 8, 64, seed=0)
    plan = spatha.SpmmPlan(dev(vals), dev(meta), dev(columns), 64, 64, 2, 8, 64)
    assert plan.kernel_name(8, 0, 24) is None and plan.kernel_name(8, 0, 25) is None
    for variant in (24, 25, 99, -1):
        with pytest.raises(RuntimeError):
            plan.run(torch.zeros((64, 8), device=gpu).half(), variant=variant)
