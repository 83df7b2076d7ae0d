"""The certified per-pair router with Q8_K inputs (K-quant and IQ layers), and the one-token lists.

Its workgroups also write the layer's quantized inputs: whole waves a super-block each where the input is
Q8_K, 8-lane groups a 32-block where it is Q8_0.  The cases sit at the rule's edges: one token (the selection
writes the lists), 1024 pairs (a workgroup per pair) and past them (four experts per workgroup), an expert
count that is no multiple of four there (the exact router takes the call), the most pairs (5120, from 65
experts 7168) and one token past them (the exact router again), more super-blocks than a workgroup has waves,
the shared FFN's input of the other format, and 8 assignments per expert (the matrix cores' copies).  Routing, lists and products are the oracle's bit for bit (check_layer)."""
import numpy as np
import pytest

from test_gpu_parity import check_layer, say

pytestmark = pytest.mark.gpu

CASES = {
    "q4k_q6k_T1": (dict(idx=71, T=1, d=2816, E=64, k=4, nf=352, gu=12, dn=14), 1),
    "q4k_shared_q8_0_T1": (dict(idx=72, T=1, d=1024, E=8, k=2, nf=256, gu=12, dn=14, nff=256, sh=8), 1),
    "q4_0_gu_q6k_dn_shared_q5k_T3": (dict(idx=73, T=3, d=768, E=8, k=2, nf=256, gu=2, dn=14, nff=512, sh=13), 3),
    "q6k_1024_pairs": (dict(idx=74, T=64, d=512, E=16, k=2, nf=256, gu=14, dn=12), 64),
    "q4k_past_1024_pairs": (dict(idx=75, T=65, d=4096, E=16, k=2, nf=256, gu=12, dn=14), 65),
    "q5k_no_multiple_of_four": (dict(idx=76, T=80, d=512, E=14, k=2, nf=256, gu=13, dn=13), 80),
    "q4k_5120_pairs": (dict(idx=91, T=80, d=512, E=64, k=4, nf=256, gu=12, dn=14), 80),
    "q4k_past_5120_pairs": (dict(idx=91, T=81, d=512, E=64, k=4, nf=256, gu=12, dn=14), 81),
    "q6k_7168_pairs": (dict(idx=92, T=56, d=512, E=128, k=2, nf=256, gu=14, dn=12), 56),
    "q6k_past_7168_pairs": (dict(idx=92, T=57, d=512, E=128, k=2, nf=256, gu=14, dn=12), 57),
    "iq_T1": (dict(idx=77, T=1, d=512, E=8, k=2, nf=256, gu=21, dn=16), 1),
    "q8_0_wide_T1": (dict(idx=78, T=1, d=4096, E=8, k=8, nf=256, gu=8, dn=14), 1),
    "q4k_bias_kmma_T40": (dict(idx=79, T=40, d=1024, E=4, k=2, nf=256, gu=12, dn=12, hot=0.9), 40),
}


@pytest.mark.parametrize("case", list(CASES))
def test_q8k_inputs_from_the_router(ctx, pkg, orc, case):
    cfg, T = CASES[case]
    say(f"k route {case}: T={T}")
    L = pkg.synth.make_layer(cfg, norms="random")
    x = pkg.synth.make_input(cfg, T=T)
    ctx.upload(0, L)
    check_layer(ctx, orc, L, x, tag=f"k route {case}")


def test_one_token_lists_with_ties(ctx, pkg, orc):
    """Identical router rows (the exact selection runs) at one token: the lists still follow the ids."""
    say("k route: one token, tied experts")
    cfg = dict(idx=80, T=1, d=512, E=16, k=4, nf=256, gu=12, dn=14)
    L = pkg.synth.make_layer(cfg)
    L["gate_inp"][:] = L["gate_inp"][5]
    x = pkg.synth.make_input(cfg, T=1)
    before = ctx.fallback_counts()[1]
    ctx.upload(0, L)
    check_layer(ctx, orc, L, x, tag="k route ties")
    assert ctx.fallback_counts()[1] > before
    np.testing.assert_array_equal(ctx.routing()[0][0], [0, 1, 2, 3])
