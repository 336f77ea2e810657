"""Which kernel a conv's default rule takes at the edges of the rules that choose by size, and that it gives the oracle's bytes there (exact operands)."""
import numpy as np
import pytest

from ufsm_amd import lib
import orc
from test_gpu_conv import exact_case, gpu_conv

pytestmark = pytest.mark.gpu

# (bits, N, Ci, Co, D, H, W, kernel): one block into one channel tile around 16 384 voxels, around 1 024 row tiles, with rows that runs of 32 fit worse than 16;
# three blocks into one channel tile around 128, 512 and (e2m1) 256 tiles of the K-split kernel; the flat kernel behind that kernel's 256 (more than 128 output
# channels) or 512 tiles, at rows of 41 and 42 voxels, at 256 and 512 workgroups, with odd block counts and at the e2m1 limits of blocks and runs
CASES = [(8, 1, 32, 32, 16, 32, 32, "conv3_small_k"), (8, 1, 32, 32, 15, 32, 32, "conv3_row1_k"), (4, 2, 32, 24, 16, 16, 32, "conv3_small_k"),
         (8, 4, 32, 32, 32, 32, 255, "conv3_row1_k"), (8, 4, 32, 32, 28, 32, 255, "conv3_small_k"), (4, 4, 32, 32, 32, 32, 240, "conv3_small_k"),
         (8, 1, 96, 32, 9, 30, 31, "conv3_thin_k"), (8, 1, 96, 32, 8, 32, 32, "conv3_row_k"), (8, 1, 96, 32, 32, 32, 32, "conv3_thin_k"), (8, 1, 96, 32, 33, 32, 32, "conv3_row_k"),
         (4, 1, 96, 32, 16, 32, 32, "conv3_thin_k"), (4, 1, 96, 32, 17, 32, 32, "conv3_row_k"),
         (8, 1, 128, 192, 6, 23, 21, "conv3_flat_k"), (8, 1, 128, 192, 6, 21, 21, "conv3_thin_k"), (8, 1, 64, 64, 10, 23, 41, "conv3_flat_k"), (8, 1, 64, 64, 10, 23, 42, "conv3_row_k"),
         (8, 1, 64, 64, 32, 32, 32, "conv3_flat_k"), (8, 1, 64, 64, 33, 32, 32, "conv3_row_k"), (8, 1, 96, 96, 16, 16, 24, "conv3_mx_k"),
         (4, 1, 64, 64, 16, 32, 32, "conv3_row_k"), (4, 1, 128, 64, 16, 32, 32, "conv3_flat_k"), (4, 1, 128, 64, 17, 32, 32, "conv3_wide_k")]


@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W,kern", CASES)
def test_default_rule_at_its_edges(gpu, bits, N, Ci, Co, D, H, W, kern):
    rng = np.random.default_rng(Ci + 3 * Co + D + W)
    x, w, b = exact_case(rng, N, Ci, Co, D * H * W)
    xdt = 3 if bits == 8 else 4
    xq = orc.f32_to_mx(bits, x, N, Ci, D * H * W)
    got, _ = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, xdt, cbits=bits)
    assert kern in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
    want, _ = orc.conv3(xq, xdt, N, Ci, D, H, W, w, b, Co, xdt, cbits=bits, acc64=1)
    assert np.array_equal(got, want)
