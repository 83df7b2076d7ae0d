"""K-quant products on the vector units (k_grouped_k): rounds, tiles, alignments and grid against the oracle.

A workgroup takes a 64-row group and a tile of up to four input rows, a wave per super-block in rounds of up
to 16 (a launch that fills less than the chip) or about four.  The cases sit at those edges: one super-block,
a whole round, one past it and a ragged last round; one row, whole and ragged tiles; row counts around a row
group; enough workgroups for the narrow rounds; and the caller's rows at addresses that are 4 but not 16
bytes aligned.  Every sum is the reference's chain, so results are equal bit for bit."""
import numpy as np
import pytest

from test_gpu_parity import check_layer
from test_gpu_quant import gguf_k_rows

pytestmark = pytest.mark.gpu


def say(s):
    print(s, flush=True)


@pytest.mark.parametrize("wtype", [11, 12, 13, 14])
@pytest.mark.parametrize("T,rows,cols", [(1, 1, 256), (1, 65, 4096), (2, 64, 4352), (4, 130, 1536), (5, 63, 8448),
                                         (7, 4700, 1280)])
def test_few_rows_match_oracle(ctx, orc, wtype, T, rows, cols):
    say(f"k rows: type={wtype} T={T} rows={rows} cols={cols}")
    rng = np.random.default_rng(7 * rows + cols + wtype + T)
    w = gguf_k_rows(rng, wtype, rows, cols)
    x = rng.standard_normal((T, cols)).astype(np.float32)
    qs, d, _ = ctx.Q8K(0, x)
    h = ctx.weight_upload(wtype, w, rows, cols)
    bufs = [ctx.alloc(qs.nbytes + 16), ctx.alloc(d.nbytes), ctx.alloc(T * rows * 4)]
    try:
        bufs[1].upload(d)
        for shift in (0, 4):
            bufs[0].upload(np.concatenate([np.zeros(shift, np.int8), qs.reshape(-1)]))
            ctx.matmul_k_device(h, T, bufs[0].ptr + shift, bufs[1].ptr, bufs[2].ptr)
            ctx.sync()
            y = bufs[2].download((T, rows))
            for t in range(T):
                np.testing.assert_array_equal(y[t], orc.matvec(wtype, w, rows, cols, x[t]), err_msg=f"token {t}")
    finally:
        for b in bufs:
            b.free()
        ctx.weight_free(h)


# Past 6144 assignments times row groups (24 per compute unit) a wave walks whole rows (k_grouped_k_walk), eight
# super-blocks staged at a time, four row groups to a workgroup: the last size below that, a super-block, a whole
# stage and one past it, a row group alone and one past a multiple of four, ragged tiles.
@pytest.mark.parametrize("T,rows,cols", [(94, 4100, 512), (95, 4100, 256), (97, 4100, 2304), (6145, 63, 2048)])
def test_walk_matches_oracle(ctx, orc, T, rows, cols):
    say(f"k walk: T={T} rows={rows} cols={cols}")
    rng = np.random.default_rng(T + cols)
    w = gguf_k_rows(rng, 13, rows, cols)
    x = rng.standard_normal((T, cols)).astype(np.float32)
    qs, d, _ = ctx.Q8K(0, x)
    h = ctx.weight_upload(13, w, rows, cols)
    try:
        y = ctx.MatMulK(h, rows, cols, qs, d)
    finally:
        ctx.weight_free(h)
    for t in sorted({0, 1, T - 2, T - 1, *rng.choice(T, 12).tolist()}):
        np.testing.assert_array_equal(y[t], orc.matvec(13, w, rows, cols, x[t]), err_msg=f"token {t}")


WALK_LAYERS = {  # 192 assignments, 33 or more row groups; gate|up and down of different kinds stay on the vector units
    "q4k_gate_nb9": dict(idx=101, d=2304, E=8, k=2, nf=1056, gu=12, dn=8),
    "q6k_gate_nb1": dict(idx=102, d=256, E=8, k=2, nf=1056, gu=14, dn=2),
    "q5k_both": dict(idx=103, d=2304, E=8, k=2, nf=1056, gu=13, dn=13),
    "q6k_down": dict(idx=104, d=2112, E=8, k=2, nf=288, gu=8, dn=14),
    "q4k_down": dict(idx=105, d=2112, E=8, k=2, nf=288, gu=2, dn=12),
}


@pytest.mark.parametrize("case", list(WALK_LAYERS))
def test_walk_layer_matches_oracle(ctx, pkg, orc, case):
    cfg = dict(WALK_LAYERS[case], T=96)
    say(f"k walk layer {case}")
    L = pkg.synth.make_layer(cfg, norms="random")
    ctx.upload(0, L)
    check_layer(ctx, orc, L, pkg.synth.make_input(cfg, T=96), tag=f"k walk {case}")


def test_grid_past_one_dimension(ctx, orc):
    """The largest T of a Q5_K product (no matrix-core kernel takes it) over 1024 row groups: 16384 tiles x 1024 row
    groups x 256 threads are 2^32, one more than a grid's dimension holds."""
    wtype, T, rows, cols = 13, 65535, 65473, 1024
    say(f"k rows: grid past one dimension T={T} rows={rows}")
    rng = np.random.default_rng(5)
    w = gguf_k_rows(rng, wtype, rows, cols)
    x = rng.standard_normal((7, cols)).astype(np.float32)
    qs, d, _ = ctx.Q8K(0, x)
    h = ctx.weight_upload(wtype, w, rows, cols)
    at = np.arange(T) % len(x)
    bufs = [ctx.alloc(T * cols), ctx.alloc(T * cols // 256 * 4), ctx.alloc(T * rows * 4)]
    try:
        bufs[0].upload(qs.reshape(-1, cols)[at])
        bufs[1].upload(d.reshape(len(x), -1)[at])
        ctx.matmul_k_device(h, T, bufs[0].ptr, bufs[1].ptr, bufs[2].ptr)
        ctx.sync()
        for t in (0, 3, T // 2, T - 2, T - 1):
            y = np.empty(rows, np.float32)
            ctx._check(ctx.lib.phx_moe_memcpy_d2h(ctx.h, y.ctypes.data, bufs[2].ptr + t * rows * 4, y.nbytes))
            np.testing.assert_array_equal(y, orc.matvec(wtype, w, rows, cols, x[t % len(x)]), err_msg=f"token {t}")
    finally:
        for b in bufs:
            b.free()
        ctx.weight_free(h)
