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
