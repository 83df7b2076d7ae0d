"""Layers of a few assignments per expert, on both sides of the matrix cores' thresholds, and the shared FFN
beside the experts (it runs on the context's second stream, joined before the combine).

Q4_0 / Q8_0 products move to the matrix cores at three assignments per expert, K-quant ones at three and a half
where the matrix-core workgroups would be many, else at one where the VALU rows' workgroups are; all are the
reference's chains, so every stage equals the oracle bit for bit.  The stream test queues calls without
waits, over two layers, several token counts and both routers, and replays a captured stack: every result
equals the same call made alone."""
import numpy as np
import pytest

from test_gpu_parity import check_layer

pytestmark = pytest.mark.gpu


def say(s):
    print(s, flush=True)


CASES = {
    "q4_0_below": (dict(idx=91, T=11, d=1024, E=8, k=2, nf=256, gu=2, dn=2, nff=288, sh=2), 11),
    "q4_0_at": (dict(idx=92, T=12, d=1024, E=8, k=2, nf=256, gu=2, dn=2, nff=288, sh=2), 12),
    "q8_0_at_shared_mfma": (dict(idx=93, T=36, d=512, E=24, k=2, nf=256, gu=8, dn=8, nff=256, sh=8), 36),
    "q4k_q6k_few_workgroups": (dict(idx=94, T=8, d=512, E=8, k=2, nf=512, gu=12, dn=14), 8),
    "q4k_q6k_matrix_cores": (dict(idx=95, T=20, d=512, E=8, k=2, nf=1024, gu=12, dn=14), 20),
    "q4k_q6k_many_below": (dict(idx=98, T=55, d=768, E=64, k=4, nf=1280, gu=12, dn=14), 55),
    "q4k_q6k_many_at": (dict(idx=99, T=56, d=768, E=64, k=4, nf=1280, gu=12, dn=14), 56),
    "q6k_q4k_shared_q5k": (dict(idx=96, T=24, d=512, E=8, k=2, nf=1024, gu=14, dn=12, nff=512, sh=13), 24),
}


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("case", list(CASES))
def test_mid_sized_layers_match_oracle(ctx, pkg, orc, case, exact):
    cfg, T = CASES[case]
    say(f"mid layer {case} exact={exact}")
    L = pkg.synth.make_layer(cfg, norms="random")
    ctx.upload(0, L)
    check_layer(ctx, orc, L, pkg.synth.make_input(cfg, T=T), tag=f"mid {case}", exact=exact)


@pytest.mark.parametrize("case", ["q4_0_at", "q8_0_at_shared_mfma", "q4k_q6k_matrix_cores"])
def test_mid_sized_calls_are_not_prefill_sized(ctx, pkg, case):
    """Under eight assignments per expert a call keeps its gate and up products unasked, and the tolerance flag
    leaves the experts' products exact (the shared FFN follows its own rule, so it is given here)."""
    cfg, T = CASES[case]
    say(f"mid layer flags {case}")
    L = pkg.synth.make_layer(cfg, norms="random")
    ctx.upload(0, L)
    x = pkg.synth.make_input(cfg, T=T)
    sh = x[::-1].copy()
    want = ctx.ffn(0, x, sh, keep_intermediates=True)
    inter = ctx.intermediates()
    for kw in ({}, dict(fast_math=True)):
        np.testing.assert_array_equal(ctx.ffn(0, x, sh, **kw), want)
        for a, b in zip(ctx.intermediates(), inter):
            np.testing.assert_array_equal(a, b)


def test_mid_sized_fast_call_folds_only_the_shared_ffn(ctx, pkg):
    """The tolerance flag at 36 tokens, 72 assignments of 24 experts, with the layer's own shared FFN: from 32 tokens
    the shared FFN follows the flag (its own rule), the experts' products under eight assignments per expert do not.
    Bound: the folded operands' fp16 rounding (2^-11 each) flips a few percent of the shared down input's integers
    by one quantum of their block, 1/127 of its largest value: under 1/127 = 8e-3 of the outputs' size in the mean
    square and less than 0.25 of it anywhere (the limits of test_gpu_fast_math.py are 2e-2 and 0.25)."""
    cfg, T = CASES["q8_0_at_shared_mfma"]
    say("mid layer: fast shared FFN")
    L = pkg.synth.make_layer(cfg, norms="random")
    ctx.upload(0, L)
    x = pkg.synth.make_input(cfg, T=T)
    want = ctx.ffn(0, x, keep_intermediates=True)
    inter = ctx.intermediates()
    got = ctx.ffn(0, x, fast_math=True)
    for a, b in zip(ctx.intermediates(), inter):
        np.testing.assert_array_equal(a, b)
    assert not np.array_equal(got, want)
    err, rms = (got - want).astype(np.float64), np.sqrt(np.mean(want.astype(np.float64) ** 2))
    assert np.sqrt(np.mean(err ** 2)) <= rms / 127 and np.abs(err).max() <= 0.25 * rms


def test_shared_branch_stream_order(pkg):
    say("shared FFN beside the experts: queued calls and a captured stack")
    cfg = dict(idx=97, T=40, d=512, E=16, k=2, nf=256, gu=2, dn=2, nff=512, sh=2)
    layers = pkg.synth.make_stack(cfg, 2)
    P = pkg.PHX
    with pkg.MoeContext(0) as c:
        for i, L in enumerate(layers):
            c.upload(i, L)
        rng = np.random.default_rng(3)
        Ts = [40, 700, 19, 130, 40, 513, 33]
        xs = [rng.standard_normal((T, 512)).astype(np.float32) for T in Ts]
        alone = [[c.ffn(i % 2, x, exact_router=e) for e in (False, True)] for i, x in enumerate(xs)]
        xb, ob = [], []
        for x in xs:
            xb.append(c.alloc(x.nbytes))
            xb[-1].upload(x)
            ob.append([c.alloc(x.nbytes), c.alloc(x.nbytes)])
        for _ in range(3):
            for i, T in enumerate(Ts):
                for e, flag in enumerate((0, P.FLAG_EXACT_ROUTER)):
                    c.ffn_device(i % 2, T, xb[i].ptr, None, ob[i][e].ptr, flag | P.FLAG_ASYNC)
        c.sync()
        for i, x in enumerate(xs):
            for e in range(2):
                np.testing.assert_array_equal(ob[i][e].download(x.shape), alone[i][e], err_msg=f"call {i} exact={e}")
        c.stack_capture(0, 2, 40)
        first = c.stack_run(xs[0])
        y = xs[0].copy()
        for i in range(2):
            _, y = c.ffn(i, y, residual=True)
        np.testing.assert_array_equal(first, y)
        for _ in range(3):
            np.testing.assert_array_equal(c.stack_run(xs[0]), first)
        for b in xb + [o for p in ob for o in p]:
            b.free()
