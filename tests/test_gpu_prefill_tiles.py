"""The prefill chunk's tiles: groups of several tiles cut evenly, the shared
expert's tiles first, and the down pass's slices per workgroup, against the CPU
oracle (output bits)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from sager_amd import ops
from sager_amd.synth import q4k_random_np

pytestmark = pytest.mark.gpu

# (hidden, n_ff, experts, k, tokens): 96 and 97 rows in the shared expert's group;
# one expert that takes every token, past three and past four tiles; several
# tiles for most experts; 2, 4, 8, 10 and 16 column slices
CASES = [(256, 256, 4, 2, 96), (512, 256, 4, 2, 97), (512, 512, 1, 1, 289), (256, 512, 1, 1, 385),
         (1280, 512, 6, 2, 300), (1024, 256, 8, 3, 500), (2048, 512, 5, 2, 33)]


@pytest.mark.parametrize("H,F,E,k,T", CASES)
@pytest.mark.parametrize("shared", [True, False])
def test_prefill_tiles_bit_exact(H, F, E, k, T, shared):
    rng = np.random.default_rng(H + F + E + k + T)
    mats = [[q4k_random_np(rng, F * H // 256) for _ in range(E + 1)] for _ in range(3)]
    dev = [[torch.from_numpy(m).cuda() for m in row] for row in mats]
    tabs = [torch.tensor([m.data_ptr() for m in row[:E]], dtype=torch.int64, device="cuda")
            for row in dev]
    pre = ops.MoePrefill(*tabs, tuple(row[E] for row in dev) if shared else None, hidden=H, n_ff=F,
                         n_expert=E, k=k, max_tokens=T)
    x = rng.normal(0, 1, (T, H)).astype(np.float32)
    lg = rng.normal(0, 1, (T, E)).astype(np.float32)
    out, idx, w = pre.forward(torch.from_numpy(x).cuda(), torch.from_numpy(lg).cuda())
    torch.cuda.synchronize()
    ref, ri, rw = orc.moe_layer(mats[0][:E], mats[1][:E], mats[2][:E],
                                tuple(row[E] for row in mats) if shared else None, x, logits=lg,
                                hidden=H, n_ff=F, k=k, prefill=True)
    np.testing.assert_array_equal(idx.cpu().numpy()[:, :k], ri[:, :k])
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32), ref.view(np.uint32))
