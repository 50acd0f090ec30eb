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


@pytest.mark.parametrize("n_rows,E,k,dup", [(1, 8, 2, False), (31, 700, 32, False),
                                            (512, 1024, 32, False), (512, 61, 5, True),
                                            (513, 61, 5, False), (32, 5, 5, False),
                                            (512, 1024, 14, False), (512, 1024, 15, True),
                                            (512, 256, 16, True), (512, 256, 17, True),
                                            (512, 32, 32, False), (512, 33, 20, False)])
def test_plan_of_one_launch(n_rows, E, k, dup):
    """For up to 512 rows of few routes the plan is one launch: every array against
    the oracle's scan, with invalid ids and (dup) a row that names an expert twice, at
    its last row count and the two-launch form's first, at its last route counts
    and one past them (up to 32 experts all), more and fewer experts than threads,
    and a full and a partial last group of 32 rows."""
    rng = np.random.default_rng(n_rows + E)
    idx = np.stack([rng.choice(E, k, replace=False) for _ in range(n_rows)]).astype(np.int32)
    idx = np.concatenate([idx, np.full((n_rows, 1), -1, np.int32)], axis=1)
    if n_rows > 1:
        idx[n_rows - 1, k - 1] = E
        idx[n_rows // 2, 0] = -3
    if dup:
        idx[n_rows - 3, 1] = idx[n_rows - 3, 0]
    w = rng.uniform(0, 1, (n_rows, k + 1)).astype(np.float32)
    ref = orc.dispatch_scan(idx, w, k, E, tok_per=96)
    wd = torch.from_numpy(w).cuda()
    got = ops.moe_dispatch_plan(torch.from_numpy(idx).cuda(), wd, E, k, tok_per=96,
                                shared_tail=n_rows)
    torch.cuda.synchronize()
    R = int(ref["meta"][0])
    host = {n: v.cpu().numpy() for n, v in got.items()}
    np.testing.assert_array_equal(host["meta"][:3], ref["meta"][:3])
    np.testing.assert_array_equal(host["off"][:E + 1], ref["off"])
    np.testing.assert_array_equal(host["toff"][:E + 1], ref["toff"])
    np.testing.assert_array_equal(host["gslot"], ref["gslot"])
    np.testing.assert_array_equal(host["grows"][:R], ref["grows"][:R])
    np.testing.assert_array_equal(host["grows"][R:R + n_rows], np.arange(n_rows))
    np.testing.assert_array_equal(wd.cpu().numpy(), ref["weight"])


# (hidden, n_ff, tokens): every token of the one expert in one tile.  One weight
# block, one slice; one, four, five and eight tokens; the first tile past them; 73 and
# 74 staged blocks (the most, and one too many: the general tile); three blocks per
# down row, where its workgroups take one slice
FEW = [(256, 256, 1), (512, 256, 4), (512, 512, 5), (2048, 512, 8), (2048, 512, 9),
       (73 * 256, 256, 1), (37 * 256, 256, 2), (256, 37 * 256, 2), (512, 768, 3)]


@pytest.mark.parametrize("H,F,T", FEW)
@pytest.mark.parametrize("f16", [False, True])
def test_few_token_tiles_bit_exact(H, F, T, f16):
    rng = np.random.default_rng(H + F + T)
    mats = [q4k_random_np(rng, F * H // 256) for _ in range(3)]
    dev = [torch.from_numpy(m).cuda() for m in mats]
    tabs = [torch.tensor([m.data_ptr()], dtype=torch.int64, device="cuda") for m in dev]
    pre = ops.MoePrefill(*tabs, None, hidden=H, n_ff=F, n_expert=1, k=1, max_tokens=T)
    x = rng.normal(0, 1, (T, H)).astype(np.float16 if f16 else np.float32)
    lg = rng.normal(0, 1, (T, 1)).astype(np.float32)
    args = ([mats[0]], [mats[1]], [mats[2]], None, x)
    kw = dict(logits=lg, hidden=H, n_ff=F, k=1, prefill=True)
    if f16:
        out, _, _ = pre.forward_f16(torch.from_numpy(x).cuda(), None, torch.from_numpy(lg).cuda())
        ref = orc.moe_layer_f16(*args, **kw)[0]
    else:
        out, _, _ = pre.forward(torch.from_numpy(x).cuda(), torch.from_numpy(lg).cuda())
        ref = orc.moe_layer(*args, **kw)[0]
    bits = np.uint16 if f16 else np.uint32
    np.testing.assert_array_equal(out.cpu().numpy().view(bits), ref.view(bits))


def test_prefill_down_rows_past_2_gib():
    """A chunk whose Q8 of h passes 2 GiB (110700 positions of 64 super-blocks, 304 B
    each): its last tokens, and a few at the start, equal a short chunk of the same
    tokens bit for bit (tokens do not meet)."""
    rng = np.random.default_rng(3)
    H, F, T = 256, 16384, 110700
    mats = [q4k_random_np(rng, F * H // 256) for _ in range(3)]
    dev = [torch.from_numpy(m).cuda() for m in mats]
    tabs = [torch.tensor([m.data_ptr()], dtype=torch.int64, device="cuda") for m in dev]
    x = torch.randn(T, H, device="cuda", generator=torch.Generator("cuda").manual_seed(4))
    lg = torch.zeros(T, 1, device="cuda")

    def run(xs):
        pre = ops.MoePrefill(*tabs, None, hidden=H, n_ff=F, n_expert=1, k=1, max_tokens=len(xs))
        return pre.forward(xs, lg[:len(xs)])[0]

    out = run(x)
    for part in (slice(0, 200), slice(T - 500, T), slice(T - 5, T)):
        assert torch.equal(out[part].view(torch.int32), run(x[part].contiguous()).view(torch.int32))
