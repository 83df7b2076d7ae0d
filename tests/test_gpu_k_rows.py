"""K-quant products on the vector units (k_grouped_k): rounds, tiles, alignments and grid against the oracle.

A workgroup takes a 64-row group and a tile of up to four input rows, a wave per super-block in rounds of up
to 16 (a launch that fills less than the chip) or about four.  The cases sit at those edges: one super-block,
a whole round, one past it and a ragged last round; one row, whole and ragged tiles; row counts around a row
group; enough workgroups for the narrow rounds; and the caller's rows at addresses that are 4 but not 16
bytes aligned.  Every sum is the reference's chain, so results are equal bit for bit."""
import numpy as np
import pytest

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
