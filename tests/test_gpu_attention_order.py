"""Attention with the sequences worked through by length: every call has the bits of the sequences as they come."""

import random

import pytest
import torch

from pypto_amd import workloads
from pypto_amd.runtime import paged_attention

pytestmark = pytest.mark.gpu


# one pair over and under a band of one per CU, an odd last band, as many sequences as keys and more (which keep their order),
# equal and empty sequences, a power of two of them; partitions 1 to several; both forms
@pytest.mark.parametrize("batch,heads,kv_heads,head_dim,block,lo,hi,e4m3", [
    (2, 8, 8, 128, 64, 1, 900, False), (33, 32, 8, 128, 64, 0, 700, False), (32, 8, 8, 128, 128, 0, 0, False), (64, 16, 4, 128, 32, 5, 300, True),
    (96, 32, 8, 128, 64, 200, 3000, True), (129, 2, 2, 256, 64, 30, 1500, False), (255, 4, 1, 128, 64, 0, 520, False), (256, 4, 2, 256, 32, 0, 200, True),
    (257, 2, 1, 128, 64, 0, 300, False), (40, 64, 1, 128, 64, 100, 2500, False)])
@pytest.mark.parametrize("variant", [0, 2])
def test_by_length_or_as_they_come(worker, batch, heads, kv_heads, head_dim, block, lo, hi, e4m3, variant):
    lens = [random.Random(batch * hi + i).randint(lo, hi) for i in range(batch)]
    lens[-1] = hi
    if batch > 3:
        lens[0], lens[1] = lo, lens[2]
    a = workloads.paged_attention_inputs(batch=batch, num_heads=heads, kv_head_num=kv_heads, head_dim=head_dim, block_size=block,
                                         ctx_range=(max(lo, 1), max(hi, 1)), context_lens=lens, fp8_kv=e4m3, seed=batch, device="cuda")
    got = []
    worker.set_option("attn_variant", variant)
    try:
        with worker.register(paged_attention) as h:
            for order in (0, 1, 1):
                worker.set_option("attn_order", order)
                a.out.fill_(float("nan"))
                h(*a.args())
                worker.sync()
                got.append(a.out.clone())
    finally:
        worker.set_option("attn_variant", -1)
        worker.set_option("attn_order", -1)
    assert bool(got[0].isfinite().all())
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


@pytest.mark.parametrize("e4m3", [False, True])
def test_the_choice_reads_as_settled_only_once_it_stays(worker, e4m3):
    """Four or five shapes are measured four times each, then two or three by length: -1 until all of it is over, and no change afterwards."""
    lens = [random.Random(i).randint(200, 3000) for i in range(64)]
    a = workloads.paged_attention_inputs(batch=64, num_heads=32, kv_head_num=8, head_dim=128, block_size=64, ctx_range=(1, 3000), context_lens=lens,
                                         fp8_kv=e4m3, seed=5, device="cuda")
    worker.set_option("attn_autotune", 0)  # forget what earlier tests settled
    worker.set_option("attn_autotune", 1)
    names = ("attn_tuned_waves_per_cu", "attn_tuned_workgroup_form", "attn_tuned_order")
    said, outs = [], []
    with worker.register(paged_attention) as h:
        for _ in range(80):
            a.out.fill_(float("nan"))
            h(*a.args())
            worker.sync()
            said.append(tuple(worker.get_option(n) for n in names))
            outs.append(a.out.clone())
    measured = said.count((-1, -1, -1))
    assert (4 + 2) * 4 - 1 <= measured <= (5 + 3) * 4
    assert said[measured] == said[-1] and all(v >= 0 for v in said[-1])
    assert all(s == said[0] for s in said[:measured]) and all(s == said[-1] for s in said[measured:])
    assert all(torch.equal(o, outs[0]) for o in outs)
