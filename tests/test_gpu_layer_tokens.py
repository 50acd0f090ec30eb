"""The several-token layer (routing launch, plan, Q8_K of h, back kernel) at the
edges of its ranges, against the CPU oracle: indices, weights and output bits."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from sager_amd import ops
from sager_amd.synth import q4k_random_np

pytestmark = pytest.mark.gpu

# (hidden, n_ff, experts, k, tokens, shared expert): super-block counts that are
# no power of two; an odd expert table; more than 64, 128, 256 and 512 experts (the
# routing instances); 47 and 48 h blocks (quantized by the back kernel, by a launch
# of its own); groups of the shared expert full and not; the most slots that
# LDS holds; the first entry's x in 560, 580 and (the widest hidden) 640 16-B chunks,
# where a wave's nine copy instructions hold 576; one token of other shapes than the
# model's (its down copies at the kernel's start and, with more groups, later)
CASES = [(256, 256, 8, 1, 2, False), (512, 256, 61, 7, 16, True), (1280, 768, 60, 7, 5, True),
         (768, 256, 130, 8, 13, True), (256, 256, 300, 23, 2, False),
         (256, 256, 70, 22, 2, True),
         (256, 256, 600, 11, 4, False), (512, 512, 32, 5, 4, True), (512, 256, 33, 32, 11, True),
         (7168, 256, 5, 2, 2, True), (7424, 256, 5, 2, 3, False), (8192, 256, 6, 3, 2, False),
         (8192, 256, 9, 2, 10, True), (2048, 512, 20, 16, 1, True), (512, 768, 12, 7, 1, True),
         (2048, 512, 70, 10, 1, False), (8192, 256, 5, 3, 1, True)]


def _layer(rng, H, F, E, k, T, shared):
    mats = [[q4k_random_np(rng, F * H // 256) for _ in range(E + 1)] for _ in range(3)]
    dev = [[torch.from_numpy(m).cuda() for m in row] for row in mats]
    tabs = [torch.tensor([m.data_ptr() for m in row[:E]], dtype=torch.int64, device="cuda")
            for row in dev]
    sh = tuple(row[E] for row in dev) if shared else None
    layer = ops.MoeLayer(*tabs, sh, hidden=H, n_ff=F, n_expert=E, k=k, max_tokens=T)
    layer.keep = dev
    return mats, tuple(row[E] for row in mats) if shared else None, layer


@pytest.mark.parametrize("H,F,E,k,T,shared", CASES)
def test_layer_tokens_bit_exact(H, F, E, k, T, shared):
    rng = np.random.default_rng(H + F + E + k + T)
    mats, sh, layer = _layer(rng, H, F, E, k, T, shared)
    x = rng.normal(0, 1, (T, H)).astype(np.float32)
    lg = rng.normal(0, 1.5, (T, E)).astype(np.float32)
    res = rng.normal(0, 1, (T, H)).astype(np.float32)
    for _ in range(2):  # a second pass on the same workspace
        out, idx, w = layer.forward(torch.from_numpy(x).cuda(), torch.from_numpy(lg).cuda(),
                                    residual=torch.from_numpy(res).cuda())
        torch.cuda.synchronize()
        ref, ri, rw = orc.moe_layer(mats[0][:E], mats[1][:E], mats[2][:E], sh, x, logits=lg,
                                    residual=res, hidden=H, n_ff=F, k=k)
        np.testing.assert_array_equal(idx.cpu().numpy()[:, :k], ri[:, :k])
        np.testing.assert_array_equal(w.cpu().numpy().view(np.uint32), rw.view(np.uint32))
        np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32), ref.view(np.uint32))


def test_layer_tokens_one_expert_for_all():
    """Caller routing that sends every route of 16 tokens to one expert (128
    entries in one group), beside an invalid id that zeroes its row."""
    rng = np.random.default_rng(77)
    H, F, E, k, T = 512, 256, 12, 8, 16
    mats, sh, layer = _layer(rng, H, F, E, k, T, True)
    x = rng.normal(0, 1, (T, H)).astype(np.float32)
    idx = np.full((T, k + 1), 5, np.int32)
    idx[3, 2] = E
    w = rng.uniform(0, 1, (T, k + 1)).astype(np.float32)
    out, _, wd = layer.forward(torch.from_numpy(x).cuda(), None, idx=torch.from_numpy(idx).cuda(),
                               weight=torch.from_numpy(w).cuda())
    torch.cuda.synchronize()
    ref, _, rw = orc.moe_layer(mats[0][:E], mats[1][:E], mats[2][:E], sh, x, idx=idx, weight=w,
                               hidden=H, n_ff=F, k=k)
    np.testing.assert_array_equal(wd.cpu().numpy().view(np.uint32), rw.view(np.uint32))
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32), ref.view(np.uint32))


# (hidden, n_ff, experts, k, tokens, small workspace).  The split shared expert's extra
# plan entries past a 256-B boundary of the workspace (32 groups against 35: 63744 and
# 64512 B), or past the back kernel's LDS (163840 B with four row buffers: 163824 B and,
# exactly, 163840 with one group, 163856 and more with the split)
ONE_GROUP = [(512, 256, 31, 3, 13, True), (512, 256, 33, 30, 12, False),
             (1024, 768, 33, 7, 16, False), (512, 512, 12, 11, 16, False)]


@pytest.mark.parametrize("H,F,E,k,T,small", ONE_GROUP)
def test_layer_of_one_shared_group(H, F, E, k, T, small):
    """Without room for the split shared expert's extra plan entries, in the caller's
    workspace or in LDS, the layer takes the layout of one shared group."""
    rng = np.random.default_rng(78 + E)
    mats, sh, layer = _layer(rng, H, F, E, k, T, True)
    x = rng.normal(0, 1, (T, H)).astype(np.float32)
    lg = rng.normal(0, 1, (T, E)).astype(np.float32)
    kw = {}
    if small:
        al = lambda n: (n + 255) // 256 * 256
        g, e = min(T * k, E) + 1, T * k + T
        n = (256 + al(4 * (g + 1)) + 2 * al(4 * e) + 3 * al(8 * g) + al(4 * T)
             + al(4 * T * (k + 1) * F) + al(4 * 80 * T * H // 256))
        assert n < ops.load().sg_moe_layer_workspace_bytes(T, H, F, E, k)
        kw["workspace"] = torch.zeros(n, dtype=torch.uint8, device="cuda")
    out, idx, w = layer.forward(torch.from_numpy(x).cuda(), torch.from_numpy(lg).cuda(), **kw)
    torch.cuda.synchronize()
    ref, ri, _ = orc.moe_layer(mats[0][:E], mats[1][:E], mats[2][:E], sh, x, logits=lg, hidden=H,
                               n_ff=F, k=k)
    np.testing.assert_array_equal(idx.cpu().numpy()[:, :k], ri[:, :k])
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32), ref.view(np.uint32))
