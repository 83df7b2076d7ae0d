"""Dense Q4_0 / Q8_0 and K-quant products over rows in order (no lists): the whole-row kernel k_grouped_q_wide
and the matrix-core kernels' tile sizes, against the oracle.

phx_matmul runs up to 16 rows, and more while that gives few workgroups, through k_grouped_q_wide on the
caller's planar rows: eight blocks per wave, up to 16 waves a round, four input rows per tile.  The cases sit at
those edges: one block, one wave, one block more, a full round and one block past it, ragged tiles and row
groups, and rows whose address is 4 but not 16 bytes aligned.  Larger calls run on the matrix cores in tiles
chosen by the size of the launch (of Q4_0 / Q8_0 32 rows, of one block and of three too, and 128; of K-quants 16,
32 and 48).  A layer of few experts and few assignments takes the whole-row kernel with its fused
requantization; a shared FFN of many row groups and long rows the ring kernel (k_grouped_q_ring) with its
activations in several chunks.  Every sum is the reference's chain, so results are equal bit for bit."""
import numpy as np
import pytest

from test_gpu_parity import check_layer
from test_gpu_quant import gguf_k_rows

pytestmark = pytest.mark.gpu


def say(s):
    print(s, flush=True)


def check_rows(y, ref, T, rng):
    for t in range(T) if T <= 32 else sorted({0, 15, 16, 31, 32, T - 1, *rng.choice(T, 12).tolist()}):
        np.testing.assert_array_equal(y[t], ref(t), err_msg=f"token {t}")


@pytest.mark.parametrize("wtype", [2, 8])
@pytest.mark.parametrize("T,rows,cols", [(1, 1, 32), (3, 130, 256), (5, 63, 288), (1, 65, 4096), (2, 64, 4128),
                                         (4, 64, 8224), (17, 2112, 704), (19, 9300, 32), (19, 9300, 96),
                                         (33, 9300, 32), (48, 4224, 96),
                                         (300, 4224, 256), (2047, 4224, 256)])
def test_dense_rows_match_oracle(ctx, pkg, orc, wtype, T, rows, cols):
    say(f"q rows: type={wtype} T={T} rows={rows} cols={cols}")
    rng = np.random.default_rng(rows + cols + wtype + T)
    w = pkg.synth.quantize(wtype, rng.standard_normal((rows, cols)).astype(np.float32))
    x = rng.standard_normal((T, cols)).astype(np.float32)
    qs, d = ctx.Q80(0, x)
    h = ctx.weight_upload(wtype, w, rows, cols)
    bufs = [ctx.alloc(qs.nbytes + 16), ctx.alloc(d.nbytes + 16), ctx.alloc(T * rows * 4)]
    try:
        for shift in (0, 4):
            bufs[0].upload(np.concatenate([np.zeros(shift, np.int8), qs.reshape(-1)]))
            bufs[1].upload(np.concatenate([np.zeros(shift // 4, np.uint16), d.reshape(-1)]))
            ctx.matmul_device(h, T, bufs[0].ptr + shift, bufs[1].ptr + shift // 2, bufs[2].ptr)
            ctx.sync()
            y = bufs[2].download((T, rows))
            check_rows(y, lambda t: orc.matvec(wtype, w, rows, cols, x[t]), T, rng)
    finally:
        for b in bufs:
            b.free()
        ctx.weight_free(h)


@pytest.mark.parametrize("wtype", [12, 14])
@pytest.mark.parametrize("T", [100, 200, 300])
def test_k_tiles_match_oracle(ctx, orc, wtype, T):
    rows, cols = 4224, 256
    say(f"k tiles: type={wtype} T={T}")
    rng = np.random.default_rng(wtype + T)
    w = gguf_k_rows(rng, wtype, rows, cols)
    x = rng.standard_normal((T, cols)).astype(np.float32)
    qs, d, _ = ctx.Q8K(0, x)
    h = ctx.weight_upload(wtype, w, rows, cols)
    try:
        y = ctx.MatMulK(h, rows, cols, qs, d)
    finally:
        ctx.weight_free(h)
    check_rows(y, lambda t: orc.matvec(wtype, w, rows, cols, x[t]), T, rng)


@pytest.mark.parametrize("wtype", [2, 8])
@pytest.mark.parametrize("d,nf,nff,T", [(1024, 512, 1024, 11), (512, 96, 288, 9)])
def test_few_expert_layer_matches_oracle(ctx, pkg, orc, wtype, d, nf, nff, T):
    """Under three assignments per expert (22 and 18 over 8), exact router: no decode path, no matrix cores."""
    say(f"q rows layer: type={wtype} d={d} nf={nf} T={T}")
    cfg = dict(idx=90, T=T, d=d, E=8, k=2, nf=nf, gu=wtype, dn=wtype, nff=nff, sh=wtype)
    L = pkg.synth.make_layer(cfg, norms="random")
    ctx.upload(0, L)
    check_layer(ctx, orc, L, pkg.synth.make_input(cfg, T=T), tag=f"q rows layer {wtype}", exact=True)


@pytest.mark.parametrize("wtype", [2, 8])
def test_ring_chunks_match_oracle(ctx, pkg, orc, wtype):
    """k_grouped_q_ring over rows of 136 blocks (a chunk of 128 and one of 8) and its fused requantization: 29
    tokens' shared gate and up rows, eight tiles (the last of one row) of 257 row groups, past the 2048 workgroups
    that the whole-row kernel takes."""
    say(f"q rows ring chunks: type={wtype}")
    cfg = dict(idx=94, T=29, d=4352, E=8, k=2, nf=64, gu=wtype, dn=wtype, nff=8224, sh=wtype)
    L = pkg.synth.make_layer(cfg, norms="random")
    ctx.upload(0, L)
    check_layer(ctx, orc, L, pkg.synth.make_input(cfg, T=29), tag=f"q rows ring chunks {wtype}", exact=True)


@pytest.mark.parametrize("wtype,T,rows,cols", [(2, 3, 130, 256), (8, 40, 130, 512), (2, 300, 4224, 256),
                                               (12, 5, 300, 512), (13, 20, 130, 512), (14, 20, 130, 512)])
@pytest.mark.parametrize("over", ["integers", "scales"])
def test_output_over_the_input_rows(ctx, pkg, orc, wtype, T, rows, cols, over):
    """y written over the integers or the scales of the call's own input rows: the result is that of rows apart."""
    say(f"q rows: type={wtype} T={T} y over the {over}")
    rng = np.random.default_rng(T + wtype)
    x = rng.standard_normal((T, cols)).astype(np.float32)
    if wtype in (2, 8):
        w = pkg.synth.quantize(wtype, rng.standard_normal((rows, cols)).astype(np.float32))
        qs, d = ctx.Q80(0, x)
        mm = ctx.matmul_device
    else:
        w = gguf_k_rows(rng, wtype, rows, cols)
        qs, d, _ = ctx.Q8K(0, x)
        mm = ctx.matmul_k_device
    h = ctx.weight_upload(wtype, w, rows, cols)
    ny = T * rows * 4
    pool, other = ctx.alloc(max(ny, qs.nbytes) + 64), ctx.alloc(max(qs.nbytes, d.nbytes))
    try:
        inside = qs if over == "integers" else d
        at = max(0, ny - inside.nbytes) // 2 // 16 * 16  # in the middle of y
        buf = np.zeros(pool.nbytes, np.uint8)
        buf[at:at + inside.nbytes] = inside.reshape(-1).view(np.uint8)
        for _ in range(3):
            pool.upload(buf)
            other.upload(d if over == "integers" else qs)
            q, s = (pool.ptr + at, other.ptr) if over == "integers" else (other.ptr, pool.ptr + at)
            mm(h, T, q, s, pool.ptr)
            ctx.sync()
            y = pool.download((T, rows))
            check_rows(y, lambda t: orc.matvec(wtype, w, rows, cols, x[t]), T, rng)
    finally:
        pool.free()
        other.free()
        ctx.weight_free(h)
