"""Conversion of a matrix that lives on the GPU (search, encoding and decoding as kernels) against the path through the host (the
search kernel's winners, host masks and host builder, which the oracle checks; without equal magnitudes the host's own search too): the
same arrays bit for bit - narrow and wide tails, groups without a winner, equal magnitudes, every group count per workgroup, strided and
fp32 inputs, infinities and NaN."""
import numpy as np
import pytest
import torch

from venom_amd import _lib, bert
from venom_amd import format as F
from venom_amd.grouped_nmv_tensor import SrNMTensor, nm_vector_mask_sparsify

pytestmark = pytest.mark.gpu


def host_matrix(w, m, v):
    mask, columns = nm_vector_mask_sparsify(w, 2, m, v, gpu=True, exact_ties=False)
    return SrNMTensor(2, m, v, w, mask, columns, w.device)


def same(a, b):
    assert a.dtype == b.dtype and a.device == b.device and a.shape == b.shape
    bits = {torch.float16: torch.int16}.get(a.dtype, a.dtype)
    assert torch.equal(a.view(bits), b.view(bits))


@pytest.mark.parametrize("rows,cols,m,v", [(32, 4, 4, 32), (64, 64, 8, 32), (64, 65, 8, 32), (64, 66, 8, 64), (64, 67, 8, 32),
                                           (128, 70, 8, 128), (64, 300, 7, 32), (256, 1280, 10, 64), (128, 777, 16, 64),
                                           (64, 6, 16, 32), (64, 3, 8, 32), (64, 2, 8, 64), (32, 600, 40, 32), (64, 1024, 4, 64)])
@pytest.mark.parametrize("kind", ["gauss", "ties", "sparse", "fp32", "strided", "special"])
def test_conversion_equals_the_host_path(gpu, rows, cols, m, v, kind):
    gen = torch.Generator(device="cuda").manual_seed(rows + 3 * cols + m)
    w = torch.randn((rows, cols), generator=gen, device="cuda").half()
    if kind == "ties":
        w = torch.randint(-2, 3, (rows, cols), generator=gen, device="cuda").half()
    elif kind == "sparse":
        w = w * (torch.rand((rows, cols), generator=gen, device="cuda") < 0.2)
        w[:, :m] = 0
    elif kind == "fp32":
        w = torch.randn((rows, cols), generator=gen, device="cuda")
    elif kind == "strided":
        w = torch.randn((cols, rows + 3), generator=gen, device="cuda").half()[:, 1:rows + 1].t()
    elif kind == "special":
        w[::7, ::5] = float("inf")
        w[::11, 1::9] = float("nan")
        w[1::3, ::4] = -0.0
    got = bert.NMVectorSparsifier(2, m, v, magnitude=True)(w).wrapped_tensor
    want = host_matrix(w, m, v)
    for name in ("values", "metadata", "columns"):
        same(getattr(got, name), getattr(want, name))
    if kind == "fp32":          # no two equal magnitudes or totals: the host's own search, whatever its order among equals
        host = SrNMTensor(2, m, v, w, *nm_vector_mask_sparsify(w, 2, m, v, gpu=False), w.device)
        for name in ("values", "metadata", "columns"):
            same(getattr(got, name), getattr(host, name))
    assert (got.nrows, got.ncols, got.nnz, got.device) == (want.nrows, want.ncols, want.nnz, want.device)
    dense = F.decode(got.values.cpu().numpy(), got.metadata.cpu().numpy().view(np.uint32),
                     got.columns.cpu().numpy().astype(np.uint32), rows, cols, 2, m, v)
    same(got.to_dense(), torch.from_numpy(dense).cuda())


@pytest.mark.parametrize("rows,cols,m,v", [(96, 300, 5, 32), (96, 1029, 7, 32), (128, 2052, 9, 64), (64, 416, 11, 64), (128, 135, 17, 128),
                                           (512, 85, 40, 512), (960, 40, 40, 960), (960, 44, 4, 960)])
@pytest.mark.parametrize("kind", ["gauss", "subnormal", "large", "fp32", "nan"])
def test_search_on_packed_magnitudes_finds_the_hosts_columns(gpu, rows, cols, m, v, kind):
    """Runs of one to five subsets per triple with every remainder, four groups to a workgroup and fewer (the encoding in a launch of its
    own), blocks without a spare unit between columns; fp16 totals through subnormals and up to fp32's rounding of large sums, and a
    NaN, which sends its workgroup the other way."""
    gen = torch.Generator(device="cuda").manual_seed(rows + 5 * cols + m)
    w = torch.randn((rows, cols), generator=gen, device="cuda")
    w = {"subnormal": w * 2.0 ** -21, "large": w * 9000}.get(kind, w)
    if kind != "fp32":
        w = w.half()
    if kind == "nan":
        w[rows // 2, cols // 3] = float("nan")
    got = bert.NMVectorSparsifier(2, m, v, magnitude=True)(w).wrapped_tensor
    # the selector's GPU search runs in fp32 and needs no tie replay for its columns; the host's own search checks it without a NaN
    mask, columns = nm_vector_mask_sparsify(w, 2, m, v, gpu=True, exact_ties=False)
    want = SrNMTensor(2, m, v, w, mask, columns, w.device)
    for name in ("values", "metadata", "columns"):
        same(getattr(got, name), getattr(want, name))
    if kind != "nan":
        _, host = nm_vector_mask_sparsify(w, 2, m, v, gpu=False)
        assert torch.equal(got.columns.cpu(), host)


def test_a_column_offset_beyond_the_group_is_refused(gpu):
    a = bert.NMVectorSparsifier(2, 8, 32, magnitude=True)(torch.randn(32, 64, device="cuda").half()).wrapped_tensor
    a.columns[5] = 8
    with pytest.raises(_lib.SpathaError):
        a.to_dense()


def test_arrays_at_odd_addresses_are_decoded_as_before(gpu):
    a = bert.NMVectorSparsifier(2, 8, 32, magnitude=True)(torch.randn(64, 72, device="cuda").half()).wrapped_tensor
    want = a.to_dense()
    for offset in (1, 2):
        buf = torch.empty(a.values.numel() + 8, dtype=torch.float16, device="cuda")
        buf[offset:offset + a.values.numel()] = a.values
        a.values = buf[offset:offset + a.values.numel()]
        same(a.to_dense(), want)


def test_decoding_up_to_the_last_row_that_31_bits_count(gpu):
    """The last rows lie within one stride of 2^31: a row counter of 32 bits would pass it and start again below zero."""
    rows, cols, m, v = 2 ** 31 - 32, 4, 4, 32
    if torch.cuda.mem_get_info()[0] < 160 << 30:
        pytest.skip("needs 107 GB of GPU memory, and as much again to be a good neighbour")
    a = SrNMTensor.__new__(SrNMTensor)
    a.n, a.m, a.tileM, a.nrows, a.ncols, a.device = 2, m, v, rows, cols, torch.device("cuda:0")
    a.values = torch.ones(rows * 16, dtype=torch.float16, device="cuda")
    a.metadata = torch.full((rows // 2 * 2,), 0x44444444, dtype=torch.int32, device="cuda")             # the first two columns of every group
    a.columns = torch.arange(4, dtype=torch.int32, device="cuda").repeat(rows // v * 8)
    dense = a.to_dense()
    one = 0x3c00
    assert dense.shape == (rows, cols) and bool((dense.view(torch.int64).view(-1) == one | one << 16).all())
    del a, dense
    torch.cuda.empty_cache()
