"""The float32 state passes at key heads of 128, whose tiles fit LDS once only: refilled tile by tile between the groups
of products on the two-wave form (the output pass at value splits 4 and 8, the reverse pass at 8 only, of one column
slice), all at once between chunks elsewhere (splits 1 and 2, the reverse pass at 4).  One chunk, two, the last one a single token, and packed rows with one-token and empty sequences: the same bits."""
import pytest
import torch

from macai.gated_delta import chunk_gated_delta_rule, op
from oracle import gdr

pytestmark = pytest.mark.gpu


def _run(inp, dsT, cu, split, recompute):
    names = ("query", "key", "value", "g", "beta", "initial_state")
    leaves = [inp[n].cuda().requires_grad_(True) for n in names]
    kw = {} if cu is None else {"cu_seqlens": torch.tensor(cu, dtype=torch.int32, device="cuda")}
    old = op.VALUE_SPLIT, op.RECOMPUTE_STATES
    try:
        op.VALUE_SPLIT, op.RECOMPUTE_STATES = split, recompute
        o, sT = chunk_gated_delta_rule(*leaves[:5], initial_state=leaves[5], output_final_state=True,
                                       use_qk_l2norm_in_kernel=True, **kw)
        grads = torch.autograd.grad([o, sT], leaves, [inp["do"].cuda(), dsT.cuda()])
    finally:
        op.VALUE_SPLIT, op.RECOMPUTE_STATES = old
    torch.cuda.synchronize()
    return [o, sT, *grads]


@pytest.mark.parametrize("T,cu", [(1, None), (64, None), (65, None), (129, None), (256, None),
                                  (200, [0, 1, 1, 66, 194, 200])])
def test_tile_by_tile_refill_changes_no_bits(T, cu):
    print("case float32 phased", T, cu, flush=True)
    inp = gdr.make_inputs(1, T, 3, 3, 128, 128, torch.float32, s0=True, seed=T)
    inp["g"] = inp["g"] * 0.05               # the state carries over the chunks
    gen = torch.Generator().manual_seed(T + 1)
    n = 1 if cu is None else len(cu) - 1
    inp["initial_state"] = torch.randn(n, 3, 128, 128, generator=gen)
    dsT = torch.randn(n, 3, 128, 128, generator=gen)
    ref = _run(inp, dsT, cu, 1, True)
    for split in (4, 8):
        for recompute in (True, False):
            got = _run(inp, dsT, cu, split, recompute)
            assert all(torch.equal(a, b) for a, b in zip(ref, got)), (split, recompute)
