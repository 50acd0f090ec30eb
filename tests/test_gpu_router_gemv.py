"""The fp32 x fp16 GEMV (router and gate logits) at the edges of its matrix-core
tiles, through the C ABI against the CPU oracle's lane order: bits equal."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from sager_amd import ops

pytestmark = pytest.mark.gpu

# Outputs (rows x tokens) below and at 24576, the first of the 16 x 32 tiles, and
# below and at 262144, the first of the 32 x 32 ones.  Rows and tokens that are no
# multiples of the tiles; k of one ring slot, fewer slots than the ring, and more;
# k that is no multiple of a slot (the row-per-half-wave kernel).
CASES = [(256, 2048, 95), (256, 2048, 96), (1, 128, 24601), (17, 256, 1447), (60, 1280, 411),
         (33, 160, 800), (250, 384, 1048), (250, 384, 1049), (31, 640, 8461)]


@pytest.mark.parametrize("n_rows,k,T", CASES)
def test_gemv_f32_out_f16x_tiles_bit_exact(n_rows, k, T):
    rng = np.random.default_rng(n_rows * 3 + k + T)
    w = (rng.normal(0, 0.05, (n_rows, k)) * 10.0 ** rng.integers(-3, 3, (n_rows, 1))).astype(
        np.float32)
    x = rng.normal(0, 1, (T, k)).astype(np.float16)
    x[0, :7] = [0.0, -0.0, 6e-8, -6e-8, 65504.0, -65504.0, 1.0]
    guard = torch.full((T * n_rows + 64,), 7.0, device="cuda")
    ops.gemv_f32_out_f16x(torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(),
                          y=guard[:T * n_rows].view(T, n_rows))
    torch.cuda.synchronize()
    got = guard.cpu().numpy()
    np.testing.assert_array_equal(got[:T * n_rows].reshape(T, n_rows).view(np.uint32),
                                  orc.gemv_f32_lanes(w, x.astype(np.float32)).view(np.uint32))
    assert (got[T * n_rows:] == 7.0).all()


def test_gemv_f32_out_f16x_unaligned_x():
    """x 2 B off a 16-B boundary: the 16-B copies of the tiles do not apply."""
    rng = np.random.default_rng(5)
    w = rng.normal(0, 0.05, (64, 256)).astype(np.float32)
    x = rng.normal(0, 1, (500, 256)).astype(np.float16)
    buf = torch.empty(500 * 256 + 1, dtype=torch.float16, device="cuda")
    xd = buf[1:].view(500, 256)
    xd.copy_(torch.from_numpy(x))
    got = ops.gemv_f32_out_f16x(torch.from_numpy(w).cuda(), xd).cpu().numpy()
    np.testing.assert_array_equal(got.view(np.uint32),
                                  orc.gemv_f32_lanes(w, x.astype(np.float32)).view(np.uint32))
