"""The several-token Q4_K GEMV (int8 matrix cores) at the edges of its row
sets, token tiles and super-block chunks, through the C ABI against the CPU
oracle: fp32 bits equal (the kernel keeps the oracle's operation order, so the
bound is zero)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from sager_amd import ops
from sager_amd.synth import q4k_random_np

pytestmark = pytest.mark.gpu

# rows: below, at and past a 16-row set.  Below 131072 (more than 8 blocks per
# row), 262144 or (more than 8 tokens) 524288 super-blocks the direct kernel,
# from there on the streaming one, with ragged last sets; one token the one-token
# GEMV.  k: one block, counts that are no power of two, the streaming kernel's last
# (16), chunks of 16 blocks with a ragged last one.  Tokens: the token tiles of 8
# and 16, full and not.  The last three lines: both sides of the sdot4 kernel's
# lines (two to four tokens of short rows, two of 5 to 8 blocks, two and three of
# 17 to 32).
CASES = [(1, 256, 1), (15, 2048, 2), (17, 1280, 3), (16, 768, 7), (64, 4096, 16), (33, 4352, 5),
         (16000, 4352, 3), (70001, 256, 4), (65539, 256, 16), (131077, 512, 5),
         (87395, 768, 8), (37450, 1792, 4), (32769, 2048, 3), (65537, 2048, 16),
         (104861, 1280, 9), (14564, 2304, 5), (8193, 4096, 2), (8200, 4096, 16),
         (16381, 1024, 2), (65537, 256, 2), (29999, 1280, 2), (30001, 1280, 2), (52429, 1280, 2),
         (25001, 1536, 2), (18751, 2048, 2), (32771, 2048, 2), (8192, 4352, 2), (8193, 5632, 2),
         (10241, 4352, 2), (12289, 8192, 2), (12289, 8448, 2), (46261, 4352, 3), (21876, 8192, 3)]


@pytest.mark.parametrize("n_rows,k,T", CASES)
def test_gemv_batched_edges_bit_exact(n_rows, k, T):
    rng = np.random.default_rng(n_rows + 5 * k + T)
    w = q4k_random_np(rng, n_rows * k // 256)
    xq = orc.quantize_q8_k(rng.normal(0, 1, (T, k)).astype(np.float32))
    wd, xd = torch.from_numpy(w).cuda(), torch.from_numpy(xq).cuda()
    guard = torch.full((T * n_rows + 64,), 7.0, device="cuda")
    ops.gemv_q4_k_q8_batched(wd, xd, n_rows, k, T, y=guard[:T * n_rows].view(T, n_rows))
    y16 = ops.gemv_q4_k_q8_f16out_batched(wd, xd, n_rows, k, T)
    torch.cuda.synchronize()
    got = guard.cpu().numpy()
    ref = orc.gemv(w, xq, n_rows, k, T)
    np.testing.assert_array_equal(got[:T * n_rows].reshape(T, n_rows).view(np.uint32),
                                  ref.view(np.uint32))
    assert (got[T * n_rows:] == 7.0).all()
    np.testing.assert_array_equal(y16.cpu().numpy().view(np.uint16),
                                  ref.astype(np.float16).view(np.uint16))
