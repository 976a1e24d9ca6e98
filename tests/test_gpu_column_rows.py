"""The 2D x-pass over blocks of neighbouring rows, for 2048 rows and more (1024 of
1024 points): every row length, rows of several members in one block, and a last block
that is partly empty.  Inputs and tolerance of the single grids: 1e-12 (FP64) and
1e-6 (FP32-bulk) on states of order one after three steps."""
import pytest

import test_gpu_column_pass as single

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,batch", [(16, 16, 129), (32, 16, 131), (64, 16, 133), (128, 16, 135), (256, 32, 65),
                                         (512, 16, 129), (1024, 32, 65), (1024, 512, 2)])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_rows_of_many_members(gpu, nx, ny, batch, prec):
    single.test_2d_steps_at_edges(gpu, nx, ny, batch, prec)
