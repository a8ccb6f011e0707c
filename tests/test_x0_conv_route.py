"""Which kernel a convolution of the guess network takes (host rule, no GPU):
8 or 4, the march through LDS with that many rows, where its weights fit the LDS
or it has 16 outputs, or where its tiles fill the CUs better than the gathering
kernel's single 16-voxel tiles; 0, the gathering kernel, elsewhere.  Both sides
of each line were measured beside the rule."""
import pytest

from libemmi_mgfd_amd import x0net

CASES = [
    # weights in LDS, or 16 outputs: the march at any number of planes
    ((1, 8, 32), 16, 16, 8), ((8, 9, 33), 48, 16, 8), ((96, 96, 96), 16, 48, 8), ((64, 64, 64), 32, 32, 8),
    ((2, 96, 96), 64, 16, 8), ((128, 128, 128), 96, 16, 4),
    # weights from memory on multiples of 32 along x: the gathering kernel ...
    ((32, 32, 32), 64, 64, 0), ((96, 96, 96), 48, 48, 0), ((64, 64, 64), 80, 32, 0), ((128, 128, 128), 16, 128, 0),
    # ... but for 96 channels and more into up to 48
    ((96, 96, 96), 112, 48, 4), ((64, 64, 64), 96, 32, 4),
    # tiles that leave CUs idle
    ((8, 9, 33), 48, 48, 0), ((8, 8, 32), 64, 64, 0), ((1, 128, 128), 80, 32, 4), ((8, 8, 32), 16, 128, 0),
    # one tile of 16 voxels a wave: by the fills
    ((80, 80, 80), 64, 64, 8), ((40, 40, 40), 48, 48, 8), ((48, 48, 48), 48, 48, 0), ((33, 33, 33), 48, 48, 0),
    ((80, 80, 80), 80, 32, 4),
    # narrow or flat grids, many channels
    ((64, 64, 31), 16, 16, 0), ((64, 7, 64), 16, 16, 0), ((64, 64, 64), 128, 16, 0),
]


@pytest.mark.parametrize("shape,ci,co,rows", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_conv_route(shape, ci, co, rows):
    assert x0net._lib().emmi_x0_conv_route(*shape, ci, co) == rows


def test_sizes_out_of_range():
    L = x0net._lib()
    assert L.emmi_x0_conv_route(4, 8, 32, 17, 16) == L.emmi_x0_conv_route(4, 8, 32, 16, 144) == -1
    assert L.emmi_x0_conv_route(0, 8, 32, 16, 16) == -1
