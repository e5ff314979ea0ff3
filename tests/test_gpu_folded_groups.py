"""The per-chunk backward that sums a key head's two value heads itself (macai_gdr_chunk_bwd_folded) against the
per-head form and macai_gdr_group_sum: the same bits of every gradient, one to several pairs a workgroup, ragged last
chunks, packed rows with one-token sequences, each head width of the persistent form; and the rule that picks it."""
import pytest
import torch

from macai.gated_delta import _native as N
from macai.gated_delta import chunk_gated_delta_rule, op
from oracle import gdr

pytestmark = pytest.mark.gpu


def _grads(inp, Hk, cu):
    rep = inp["value"].shape[2] // Hk
    leaves = [inp[n][:, :, ::rep].contiguous().cuda() for n in ("query", "key")]
    leaves = [x.requires_grad_(True) for x in leaves + [inp[n].cuda() for n in ("value", "g", "beta")]]
    kw = {} if cu is None else {"cu_seqlens": torch.tensor(cu, dtype=torch.int32, device="cuda")}
    o, _ = chunk_gated_delta_rule(*leaves, use_qk_l2norm_in_kernel=True, **kw)
    grads = torch.autograd.grad(o, leaves, inp["do"].cuda())
    torch.cuda.synchronize()
    return grads


@pytest.mark.parametrize("B,T,Hk,D,cu", [(1, 64 * 19 + 5, 8, 128, None), (2, 130, 40, 64, None), (2, 90, 64, 32, None),
                                         (2, 64 * 16, 16, 128, None), (1, 1300, 8, 128, [0, 1, 300, 301, 1300])])
def test_folded_pairs_give_the_group_sums_bits(B, T, Hk, D, cu, monkeypatch):
    print("case folded groups", B, T, Hk, D, cu, flush=True)
    inp = gdr.make_inputs(B, T, Hk, 2 * Hk, D, D, torch.bfloat16, seed=B + T)
    names = []
    launch = op._launch
    monkeypatch.setattr(op, "_launch", lambda name, entry, *a: (names.append(entry), launch(name, entry, *a))[1])
    folded = _grads(inp, Hk, cu)
    assert "macai_gdr_chunk_bwd_folded" in names and "macai_gdr_group_sum" not in names
    monkeypatch.setattr(N.lib(), "macai_gdr_chunk_bwd_folds", lambda *a: 0)
    per_head = _grads(inp, Hk, cu)
    assert names.count("macai_gdr_group_sum") == 2
    assert all(torch.equal(a, b) for a, b in zip(folded, per_head))


def test_folding_rule():
    """Only whole pairs that make no workgroup's run longer, at 256 compute units: 320 and 512 chunk-heads (two a
    workgroup either way) and 1,024 fold; 256 and fewer run one a workgroup, 624 would run four instead of three."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the counts below are for 256 compute units")
    folds = lambda chunks, H=16, Hk=8, D=128, DV=128, dtype=N.BF16: N.lib().macai_gdr_chunk_bwd_folds(
        1, 64 * chunks, H, Hk, D, DV, dtype, None, 0)
    assert [folds(n) for n in (16, 20, 32, 39, 64)] == [0, 1, 1, 0, 1]
    assert not folds(64, DV=64) and not folds(64, Hk=16) and not folds(64, Hk=4) and not folds(64, dtype=N.F32)


def test_folds_only_the_widths_the_kernel_takes():
    """At widths that the bf16 per-chunk backward does not take, the rule says no, as the folded entry point does."""
    folds = lambda D: N.lib().macai_gdr_chunk_bwd_folds(1, 64 * 64, 16, 8, D, D, N.BF16, None, 0)
    assert [D for D in range(32, 257, 32) if folds(D)] == [32, 64, 128]


def test_plan_reports_the_folding():
    """op.plan says what macai_gdr_chunk_bwd_folds answers, over chunk counts, widths and groups."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for H, Hk, D in ((16, 8, 128), (2, 1, 64), (32, 16, 32), (8, 2, 128)):
        for chunks in (1, 16, 17, 20, 32, 39, 64, 129, 300, 1000):
            folds = N.lib().macai_gdr_chunk_bwd_folds(1, 64 * chunks, H, Hk, D, D, N.BF16, None, 0)
            p = op.plan(1, 64 * chunks, H, D, D, True, Hk=Hk, cus=cus)
            assert p["head_sum"] == ("chunk_bwd" if folds else "group_sum"), (H, Hk, D, chunks)
