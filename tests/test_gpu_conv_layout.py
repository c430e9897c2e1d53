"""The convolution's data movement at its edges: 64-row groups that end inside an image or span several, column groups
that need more than one copy of the input rows, and the gradient's planes turned into rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c,p", [(1, 2, 2), (2, 64, 64), (3, 65, 63), (2, 130, 784), (5, 7, 49), (1, 128, 1)])
@pytest.mark.parametrize("gap", [0, 3])
def test_rows_from_planes(n, c, p, gap):
    """Bit exact at the edges of the 64 x 64 tiles; planes `gap` elements apart start on any 2-byte boundary."""
    from flash_dropout.hip import GEMM

    ext = GEMM()
    store = torch.randint(-30000, 30000, (n, c, p + gap), dtype=torch.int16, device="cuda")
    src = store[:, :, gap:]
    dst = torch.full((n * p + 1, c), 77, dtype=torch.int16, device="cuda")
    ext._call(ext.lib.sd_rows_from_planes, src.data_ptr(), src.stride(0), src.stride(1), dst.data_ptr(), n, c, p, ext._stream(dst))
    assert torch.equal(dst[:-1].view(n, p, c), src.transpose(1, 2)) and (dst[-1] == 77).all()
