"""GPU parity of the one-tile-per-workgroup GEMM (csrc/gemm_tile.hpp) at the
edges of its tiles: every tile of its table, rows and columns one past a tile
edge, column counts off the 8- and 16-column store groups, K ending inside a
slice, a step and a ring."""
import ctypes

import numpy as np
import pytest
import torch

from parity import assert_parity, bf16_to_f32
from test_gpu_parity import bits, rand_bf16, up

pytestmark = pytest.mark.gpu


def sample(m):
    """All rows of a small call, else the first, the tile edges and the last."""
    return np.arange(m) if m <= 64 else np.unique(np.r_[0, 31, 32, 63, 64, 127, 128, m // 2, m - 2, m - 1].clip(0, m - 1))


def plan(fp8lin, m, n, k, scale_cols, split):
    """(kernel, tile rows, tile columns, K ranges, workgroups per CU) of a call."""
    out = (ctypes.c_int * 5)()
    fp8lin.check(fp8lin.lib().fp8lin_gemm_plan(m, n, k, scale_cols, int(split), out))
    return tuple(out)


FEW_ROWS, SMALL_M, PERSISTENT, TILES, BLOCK, ELEMENTS = range(6)


# One row per tile (32x32, 64x32, 64x64, 128x64, 128x128 with K over two waves
# and at two per CU, 192x128, 256x160, 256x256), then longer K and whole steps.
@pytest.mark.parametrize("m,n,k", [(9, 261, 40), (33, 4100, 136), (9, 8200, 200), (65, 8195, 136), (65, 17412, 200),
                                   (2050, 17412, 40), (129, 17412, 136), (2050, 4100, 136), (2050, 6658, 136),
                                   (515, 257, 1160), (1036, 4307, 1160), (2050, 4300, 1160), (2050, 2052, 136),
                                   (129, 17412, 40), (256, 2048, 512)])
def test_bf16_tile(fp8lin, gpu, oracle, m, n, k):
    """BF16 weights with a bias through the engine: the rows of the oracle's
    product, the bias added to the rounded outputs, and no row touched by
    another row's infinities."""
    rng = np.random.default_rng(m + 3 * n + k)
    w, x, b = rand_bf16(rng, (n, k), 0.05), rand_bf16(rng, (m, k)), rand_bf16(rng, (n,))
    y = fp8lin.gemm_bf16(up(x, gpu), up(w, gpu))
    rows = sample(m)
    assert_parity(bits(y)[rows], oracle.linear_bf16w(x[rows], w), f"bf16 tile {m}x{n}x{k}")
    eng = fp8lin.LinearEngine()
    eng.add("p.weight", up(w, gpu))
    eng.add("p.bias", up(b, gpu))
    assert torch.equal(eng.linear(up(x, gpu), "p"), fp8lin.add_bias(y.clone(), up(b, gpu)))
    x[m // 2] = 0x7f80  # +inf
    z = fp8lin.gemm_bf16(up(x, gpu), up(w, gpu))
    keep = np.arange(m) != m // 2
    assert torch.equal(z[keep], y[keep])
    assert not np.isfinite(bf16_to_f32(bits(z)[m // 2])).any()


def test_bf16_tile_output_stride_and_unaligned(fp8lin, gpu, oracle):
    """A column slice of a wider output off the 16-byte grid (scalar stores),
    and operands off it (the general kernel), give the aligned call's rows."""
    rng = np.random.default_rng(5)
    m, n, k = 70, 300, 264
    w, x = rand_bf16(rng, (n, k), 0.05), rand_bf16(rng, (m, k))
    ref = oracle.linear_bf16w(x, w)
    wide = torch.zeros((m, n + 13), dtype=torch.bfloat16, device=gpu)
    fp8lin.gemm_bf16(up(x, gpu), up(w, gpu), out=wide[:, 3:3 + n])
    assert_parity(bits(wide[:, 3:3 + n]), ref, "strided output")
    assert not wide[:, :3].any() and not wide[:, 3 + n:].any()
    xs = torch.empty(m * k + 1, dtype=torch.bfloat16, device=gpu)[1:].view(m, k).copy_(up(x, gpu))
    assert_parity(bits(fp8lin.gemm_bf16(xs, up(w, gpu))), ref, "unaligned x")


@pytest.mark.parametrize("off,extra", [(0, 4), (4, 4), (2, 2), (6, 12), (1, 0), (3, 13), (8, 8)])
@pytest.mark.parametrize("m,n,k", [(9, 264, 40), (70, 312, 264), (129, 17416, 40), (515, 264, 1160), (1036, 4312, 72),
                                   (2050, 4096, 136), (2050, 6664, 136)])
def test_tile_output_rows_off_16_bytes(fp8lin, gpu, m, n, k, off, extra):
    """Output rows that start on 8, 4 or 2 bytes (staged stores) hold the bits of
    the aligned call, with nothing written beside them."""
    rng = np.random.default_rng(m + n + k)
    x, w = up(rand_bf16(rng, (m, k)), gpu), up(rand_bf16(rng, (n, k), 0.05), gpu)
    ref = fp8lin.gemm_bf16(x, w)
    for cols in (n, n - 3):
        wide = torch.full((m, off + n + extra), 7.0, dtype=torch.bfloat16, device=gpu)
        fp8lin.gemm_bf16(x, w[:cols], out=wide[:, off:off + cols])
        part = wide[:, off:off + cols]
        assert torch.equal(part, ref[:, :cols]) if cols == n else (part.float() - ref[:, :cols].float()).abs().max() < 0.1
        assert (wide[:, :off] == 7).all() and (wide[:, off + cols:] == 7).all()


# The FP8 tiles (32x32, 64x32, 64x64, 96x64, 128x64, 64x128, 96x192, 128x128
# with K over two waves and at two per CU, 256x256) and K ranges of unequal
# length.  K % 256 != 0 keeps the calls off the persistent GEMM.
FP8_TILES = [(9, 261, 48), (70, 1030, 1168), (40, 4100, 400), (70, 4100, 144), (100, 8195, 272), (96, 16000, 144),
             (33, 17412, 144), (129, 17412, 48), (520, 4096, 1168), (513, 8195, 144), (1030, 12290, 144), (9, 261, 4112),
             (65, 4100, 4112), (300, 8200, 144), (150, 4120, 400)]


@pytest.mark.parametrize("m,n,k", FP8_TILES)
@pytest.mark.parametrize("rows_scaled", [False, True])
def test_fp8_tile(fp8lin, gpu, oracle, m, n, k, rows_scaled):
    """Block and row scales against the oracle on a sample of rows; the fused
    SwiGLU equal to SwiGLU of the plain form, with and without a workspace; a
    split only reorders sums."""
    rng = np.random.default_rng(m + 3 * n + k)
    codes = rng.integers(0, 127, (n, k), dtype=np.uint8) | (rng.integers(0, 2, (n, k), dtype=np.uint8) << 7)
    scales = (rng.random(n if rows_scaled else (n, (k + 127) // 128)) * .01 + .001).astype(np.float32)
    x = rand_bf16(rng, (m, k))
    xd, cd, sd = up(x, gpu), up(codes, gpu), up(scales, gpu)
    rows = sample(m)
    ref = oracle.linear(x[rows], codes, scales)
    for split in (False, True):
        y = fp8lin.fp8_linear(xd, cd, sd, split=split)
        assert_parity(bits(y)[rows], ref, f"fp8 tile {m}x{n}x{k} split={split}")
        if n % 2 == 0:
            assert torch.equal(fp8lin.linear_swiglu(xd, cd, sd, split=split), fp8lin.fused_swiglu(y))


@pytest.mark.parametrize("m,n,k", [(9, 8195, 2320), (33, 4100, 2192), (97, 8200, 3248), (129, 16400, 1808), (200, 16400, 1168),
                                   (513, 21000, 1168), (300, 2304, 9296), (65, 4100, 9296)])
@pytest.mark.parametrize("rows_scaled", [False, True])
def test_fp8_tile_long_k(fp8lin, gpu, oracle, m, n, k, rows_scaled):
    """K over several windows of scales, ending inside a step, whole and in K
    ranges that start inside a block: a column sample against the oracle, with
    scales that differ by powers of two from block to block."""
    rng = np.random.default_rng(m + n + k)
    codes = rng.integers(0, 127, (n, k), dtype=np.uint8) | (rng.integers(0, 2, (n, k), dtype=np.uint8) << 7)
    shape = n if rows_scaled else (n, (k + 127) // 128)
    scales = np.exp2(-rng.integers(6, 12, shape)).astype(np.float32)
    x = rand_bf16(rng, (m, k))
    xd, cd, sd = up(x, gpu), up(codes, gpu), up(scales, gpu)
    rows, cols = sample(m), np.r_[0:33, n // 2:n // 2 + 33, n - 33:n]
    ref = oracle.linear(x[rows], codes[cols], scales[cols])
    for split in (False, True):
        y = fp8lin.fp8_linear(xd, cd, sd, split=split)
        assert_parity(bits(y)[rows][:, cols], ref, f"long K {m}x{n}x{k} split={split}")


@pytest.mark.parametrize("m,n,k", [(512, 25088, 320), (512, 25090, 448), (466, 24578, 1216), (705, 17410, 1344)])
@pytest.mark.parametrize("rows_scaled", [False, True])
def test_fp8_block_template(fp8lin, gpu, oracle, m, n, k, rows_scaled):
    """One round of 256x256 tiles on more than 0.6 of the CUs with K % 64 == 0:
    against the oracle, fused SwiGLU equal to the plain form's, a bias added to
    the rounded outputs, a row of NaN in its row."""
    assert plan(fp8lin, m, n, k, 1 if rows_scaled else -(-k // 128), True)[0] == BLOCK
    rng = np.random.default_rng(m + n + k)
    codes = rng.integers(0, 127, (n, k), dtype=np.uint8) | (rng.integers(0, 2, (n, k), dtype=np.uint8) << 7)
    scales = (rng.random(n if rows_scaled else (n, (k + 127) // 128)) * .01 + .001).astype(np.float32)
    x = rand_bf16(rng, (m, k))
    cd, sd, b = up(codes, gpu), up(scales, gpu), up(rand_bf16(rng, (n,)), gpu)
    y = fp8lin.fp8_linear(up(x, gpu), cd, sd)
    rows, cols = sample(m), np.r_[0:65, n - 65:n]
    assert_parity(bits(y)[rows][:, cols], oracle.linear(x[rows], codes[cols], scales[cols]), f"block {m}x{n}x{k}")
    assert torch.equal(fp8lin.linear_swiglu(up(x, gpu), cd, sd), fp8lin.fused_swiglu(y))
    eng = fp8lin.LinearEngine()
    eng.add("p.weight", cd, sd)
    eng.add("p.bias", b)
    assert torch.equal(eng.linear(up(x, gpu), "p"), fp8lin.add_bias(y.clone(), b))
    x[m // 2] = 0x7fc0  # NaN
    bad = fp8lin.fp8_linear(up(x, gpu), cd, sd)
    keep = np.arange(m) != m // 2
    assert torch.equal(bad[keep], y[keep]) and torch.isnan(bad[m // 2]).all()


@pytest.mark.parametrize("m,n,k", FP8_TILES)
@pytest.mark.parametrize("rows_scaled", [False, True])
def test_fp8_tile_infinite_scale(fp8lin, gpu, m, n, k, rows_scaled):
    """K ends inside a step of every shape: the zeros past it add nothing also
    where the scale they share with the last codes is infinite.  Positive codes
    and activations, so those outputs are +inf; all others keep their bits."""
    rng = np.random.default_rng(m + 3 * n + k)
    codes = up(rng.integers(1, 127, (n, k), dtype=np.uint8), gpu)
    scales = up((rng.random(n if rows_scaled else (n, (k + 127) // 128)) * .01 + .001).astype(np.float32), gpu)
    x = up(rand_bf16(rng, (m, k)) & 0x7fff | 1, gpu)
    cols = [0, n // 2, n - 1]
    bad = scales.clone()
    if rows_scaled:
        bad[cols] = float("inf")
    else:
        bad[cols, -1] = float("inf")
    for split in (False, True):
        ref = fp8lin.fp8_linear(x, codes, scales, split=split)
        ref[:, cols] = float("inf")
        assert torch.equal(fp8lin.fp8_linear(x, codes, bad, split=split), ref)


@pytest.mark.parametrize("m,n,k", [(70, 4096, 2048), (93, 5120, 3072), (129, 2048, 1024), (200, 1536, 4096),
                                   (320, 2048, 2048), (513, 1030, 1280), (65, 17408, 4096)])
def test_fp8_tile_beside_persistent_gemm(fp8lin, gpu, oracle, m, n, k):
    """K the persistent GEMM takes too: with a workspace the tiles may run the
    call, whole or in K ranges; the same product as the persistent GEMM's to
    the parity bar, whatever workspace is brought."""
    rng = np.random.default_rng(m + n + k)
    codes = rng.integers(0, 127, (n, k), dtype=np.uint8) | (rng.integers(0, 2, (n, k), dtype=np.uint8) << 7)
    scales = (rng.random((n, k // 128)) * .01 + .001).astype(np.float32)
    x = rand_bf16(rng, (m, k))
    xd, cd, sd = up(x, gpu), up(codes, gpu), up(scales, gpu)
    rows = sample(m)
    ref = oracle.linear(x[rows], codes, scales)
    whole = fp8lin.fp8_linear(xd, cd, sd, split=False)
    split = fp8lin.fp8_linear(xd, cd, sd)
    assert_parity(bits(whole)[rows], ref, f"whole {m}x{n}x{k}")
    assert_parity(bits(split)[rows], ref, f"split {m}x{n}x{k}")
    assert torch.equal(split, fp8lin.fp8_linear(xd, cd, sd))
    x[m // 2] = 0x7fc0  # NaN
    bad = fp8lin.fp8_linear(up(x, gpu), cd, sd)
    keep = np.arange(m) != m // 2
    assert torch.equal(bad[keep], split[keep]) and torch.isnan(bad[m // 2]).all()


@pytest.mark.parametrize("m,n,k", [(9, 5120, 8704), (27, 8192, 5120), (40, 2304, 7424), (64, 2304, 8192), (77, 4100, 2880),
                                   (70, 32896, 6656), (200, 7168, 5120), (24, 9728, 3840), (24, 17920, 3840)])
@pytest.mark.parametrize("rows_scaled", [False, True])
def test_engine_operator_and_fused_agree(fp8lin, gpu, oracle, m, n, k, rows_scaled):
    """The engine's projection, the operator and the fused gate/up of one weight
    run one plan: the same bits, with row scales as with block scales (9..64
    rows: the GEMM with row scales, the small-M kernels with block scales)."""
    rng = np.random.default_rng(m + n + k)
    codes = rng.integers(0, 127, (n, k), dtype=np.uint8) | (rng.integers(0, 2, (n, k), dtype=np.uint8) << 7)
    scales = (rng.random(n if rows_scaled else (n, (k + 127) // 128)) * .01 + .001).astype(np.float32)
    x, c, s = up(rand_bf16(rng, (m, k)), gpu), up(codes, gpu), up(scales, gpu)
    eng = fp8lin.LinearEngine()
    eng.add("p.weight", c, s)
    y = eng.linear(x, "p")
    assert torch.equal(y, fp8lin.fp8_linear(x, c, s))
    pair = fp8lin.fused_swiglu(y)
    assert torch.equal(pair, fp8lin.linear_swiglu(x, c, s))
    assert torch.equal(pair, eng._linear_swiglu(x, "p"))
    cols = np.r_[0:32, n - 32:n]
    rows = sample(m)
    assert_parity(bits(y)[rows][:, cols], oracle.linear(bits(x)[rows], codes[cols], scales[cols]), f"{m}x{n}x{k}")


@pytest.mark.parametrize("m,n,k", [(9, 256, 5344), (200, 24, 160), (3351, 130, 1056), (77, 256, 640), (97, 200, 200), (97, 256, 352)])
@pytest.mark.parametrize("bias", [False, True])
def test_dequant_branch_few_weight_rows(fp8lin, gpu, m, n, k, bias):
    """Dequantize-then-GEMM on at most 256 weight rows: the BF16 product of the
    decoded weight, bit for bit where K leaves only the BF16 matrix-core kernel
    (K % 32 == 0, K % 128 != 0) and its rows are many, else at the parity bar."""
    rng = np.random.default_rng(m + n + k)
    codes = up(rng.integers(0, 127, (n, k), dtype=np.uint8) | (rng.integers(0, 2, (n, k), dtype=np.uint8) << 7), gpu)
    scales = up((rng.random((n, (k + 127) // 128)) * .01 + .001).astype(np.float32), gpu)
    x = up(rand_bf16(rng, (m, k)), gpu)
    eng = fp8lin.LinearEngine(fp8lin.LinearOptions(cublas_prefill=True))
    eng.add("p.weight", codes, scales)
    ref = fp8lin.gemm_bf16(x, fp8lin.fp8_decode(codes, scales))
    if bias:
        b = up(rand_bf16(rng, (n,)), gpu)
        eng.add("p.bias", b)
        ref = fp8lin.add_bias(ref, b)
    y, path = eng.linear(x, "p", return_path=True)
    assert path == fp8lin.PATH_DEQUANT_GEMM
    if m > 96 and k % 32 == 0 and k % 128:
        assert torch.equal(y, ref)
    else:
        assert_parity(bits(y), bits(ref), f"dequant {m}x{n}x{k}")


# Every tile at a shape that runs it: rows one past a tile edge, ragged columns,
# K that ends inside a step and spans two to three windows of scales.
@pytest.mark.parametrize("tile,m,n,k", [
    ((32, 32, 1), 9, 261, 1168), ((64, 32, 1), 33, 4100, 1168), ((64, 64, 1), 9, 8195, 1168), ((64, 128, 1), 9, 16400, 1168),
    ((96, 64, 1), 65, 8195, 1168), ((96, 192, 1), 65, 16400, 1168), ((128, 64, 1), 97, 8195, 1168),
    ((128, 128, 1), 97, 16400, 1168), ((128, 128, 2), 200, 16400, 1168), ((256, 256, 1), 769, 14340, 1168)])
@pytest.mark.parametrize("rows_scaled", [False, True])
def test_every_fp8_tile(fp8lin, gpu, oracle, tile, m, n, k, rows_scaled):
    assert plan(fp8lin, m, n, k, 1 if rows_scaled else -(-k // 128), False) == (TILES, *tile[:2], 1, tile[2])
    rng = np.random.default_rng(m + n + k)
    codes = rng.integers(0, 127, (n, k), dtype=np.uint8) | (rng.integers(0, 2, (n, k), dtype=np.uint8) << 7)
    scales = np.exp2(-rng.integers(6, 12, n if rows_scaled else (n, -(-k // 128)))).astype(np.float32)
    x = rand_bf16(rng, (m, k))
    xd, cd, sd = up(x, gpu), up(codes, gpu), up(scales, gpu)
    rows, cols = sample(m), np.r_[0:65, n // 2:n // 2 + 65, n - 65:n]
    y = fp8lin.fp8_linear(xd, cd, sd, split=False)
    assert_parity(bits(y)[rows][:, cols], oracle.linear(x[rows], codes[cols], scales[cols]), f"tile {tile}")
    if n % 2 == 0:
        assert torch.equal(fp8lin.linear_swiglu(xd, cd, sd, split=False), fp8lin.fused_swiglu(y))


@pytest.mark.parametrize("tile,m,n,k", [
    ((32, 32, 1), 9, 261, 136), ((64, 32, 1), 33, 4100, 136), ((64, 64, 1), 9, 8195, 136), ((128, 64, 1), 65, 8195, 136),
    ((128, 128, 1), 9, 16400, 136), ((128, 128, 2), 200, 16400, 136), ((192, 128, 1), 129, 16400, 136),
    ((256, 160, 1), 385, 16400, 136), ((256, 256, 1), 1030, 12290, 136)])
def test_every_bf16_tile(fp8lin, gpu, oracle, tile, m, n, k):
    assert plan(fp8lin, m, n, k, 0, False) == (TILES, *tile[:2], 1, tile[2])
    rng = np.random.default_rng(m + n + k)
    x, w = rand_bf16(rng, (m, k)), rand_bf16(rng, (n, k), 0.05)
    rows, cols = sample(m), np.r_[0:65, n // 2:n // 2 + 65, n - 65:n]
    y = fp8lin.gemm_bf16(up(x, gpu), up(w, gpu))
    assert_parity(bits(y)[rows][:, cols], oracle.linear_bf16w(x[rows], w[cols]), f"bf16 tile {tile}")


# K ranges of every tile that takes them, with and without a bias.
@pytest.mark.parametrize("tile,m,n,k", [
    ((32, 32, 7), 9, 1030, 4112), ((64, 32, 7), 33, 1030, 4112), ((64, 64, 7), 9, 2052, 6160), ((64, 128, 7), 9, 4100, 6160),
    ((96, 64, 7), 65, 1542, 6160), ((96, 192, 2), 65, 16400, 2192), ((128, 64, 7), 97, 2052, 6160),
    ((128, 128, 7), 193, 2052, 6160), ((256, 256, 7), 193, 8195, 6160), ((96, 64, 3), 129, 2052, 4112)])
def test_tile_k_ranges(fp8lin, gpu, oracle, tile, m, n, k):
    """Against the oracle, the bias added to the rounded sums, and the same bits
    again; fused SwiGLU equal to the plain form's where the pair halves are off
    the 16-byte grid too."""
    assert plan(fp8lin, m, n, k, -(-k // 128), True)[:4] == (TILES, *tile)
    rng = np.random.default_rng(m + n + k)
    codes = rng.integers(0, 127, (n, k), dtype=np.uint8) | (rng.integers(0, 2, (n, k), dtype=np.uint8) << 7)
    scales = np.exp2(-rng.integers(6, 12, (n, -(-k // 128)))).astype(np.float32)
    x, b = rand_bf16(rng, (m, k)), up(rand_bf16(rng, (n,)), gpu)
    xd, cd, sd = up(x, gpu), up(codes, gpu), up(scales, gpu)
    rows, cols = sample(m), np.r_[0:65, n // 2:n // 2 + 65, n - 65:n]
    y = fp8lin.fp8_linear(xd, cd, sd)
    assert_parity(bits(y)[rows][:, cols], oracle.linear(x[rows], codes[cols], scales[cols]), f"K ranges {tile}")
    assert torch.equal(y, fp8lin.fp8_linear(xd, cd, sd))
    eng = fp8lin.LinearEngine()
    eng.add("p.weight", cd, sd)
    eng.add("p.bias", b)
    assert torch.equal(eng.linear(xd, "p"), fp8lin.add_bias(y.clone(), b))
    if n % 2 == 0:
        assert torch.equal(fp8lin.linear_swiglu(xd, cd, sd), fp8lin.fused_swiglu(y))


@pytest.mark.parametrize("m,n,k,rows_scaled", [(65, 1542, 6160, False), (9, 1030, 4112, True), (65, 17408, 4096, False),
                                               (97, 17408, 5120, False)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_workspace_of_any_size(fp8lin, gpu, oracle, m, n, k, rows_scaled, swiglu):
    """From the size that a call is refused without (the persistent GEMM's
    partials; none for K % 256 != 0) to more than the reported one, each meets
    the bar and writes nothing behind the bytes it was given."""
    L = fp8lin.lib()
    cols = 1 if rows_scaled else -(-k // 128)
    query = L.fp8lin_linear_swiglu_scaled_workspace_bytes if swiglu else L.fp8lin_linear_scaled_workspace_bytes
    need = query(m, n, k, cols)
    assert need > 0
    rng = np.random.default_rng(m + n + k)
    codes = rng.integers(0, 127, (n, k), dtype=np.uint8) | (rng.integers(0, 2, (n, k), dtype=np.uint8) << 7)
    scales = np.exp2(-rng.integers(6, 12, n if rows_scaled else (n, cols))).astype(np.float32)
    x = rand_bf16(rng, (m, k))
    xd, cd, sd = up(x, gpu), up(codes, gpu), up(scales, gpu)
    out = n // 2 if swiglu else n
    ref = fp8lin.fp8_linear(xd, cd, sd, split=False)
    ref = bits(fp8lin.fused_swiglu(ref) if swiglu else ref)
    kind, _, _, ranges, _ = plan(fp8lin, m, n, k, cols, True)
    partials = ranges * m * (-(-n // 8) * 8 + 8) * 4 if kind == TILES and ranges > 1 else need
    sizes = {need, need + 4096, max(partials, 16)} | ({partials - 16, 0} if k % 256 else set())
    for size in sorted(sizes):
        if k % 256 == 0 and size < need:
            continue
        ws = torch.full((size + 4096,), 0x5A, dtype=torch.uint8, device=gpu)
        y = torch.empty((m, out), dtype=torch.bfloat16, device=gpu)
        ptr = ws.data_ptr() if size else None
        stream = torch.cuda.current_stream().cuda_stream
        if swiglu:
            rc = L.fp8lin_linear_swiglu_ws(xd.data_ptr(), cd.data_ptr(), sd.data_ptr(), cols, y.data_ptr(), m, n, k, ptr, size, stream)
        else:
            rc = L.fp8lin_linear_ws(xd.data_ptr(), cd.data_ptr(), sd.data_ptr(), cols, y.data_ptr(), m, n, k, 0, ptr, size, stream)
        fp8lin.check(rc)
        assert (ws[size:] == 0x5A).all(), f"{size} of {need} bytes"
        assert_parity(bits(y), ref, f"workspace {size} of {need}", elementwise=False)


# 256-row tiles of the persistent GEMM, unsplit (two tile rows at 200 to 512 rows
# of a wide weight would be half padding at 192).
@pytest.mark.parametrize("m,n,k", [(200, 33000, 512), (256, 34000, 512), (256, 33794, 1280), (512, 50000, 512), (2300, 7000, 768)])
@pytest.mark.parametrize("rows_scaled", [False, True])
def test_fp8_256_row_tiles(fp8lin, gpu, oracle, m, n, k, rows_scaled):
    """Bit for bit the rows of a 128-row call, on 128-row tiles, which meets the
    oracle; SwiGLU likewise; a row of NaN stays in its row."""
    cols = 1 if rows_scaled else k // 128
    assert plan(fp8lin, m, n, k, cols, False) == (PERSISTENT, 256, 256, 1, 1)
    wide = n > 8192  # narrower weights run 65..128 rows as small-M halves
    if wide:
        assert plan(fp8lin, 128, n, k, cols, False) == (PERSISTENT, 128, 256, 1, 1)
    rng = np.random.default_rng(m + n + k)
    codes = rng.integers(0, 127, (n, k), dtype=np.uint8) | (rng.integers(0, 2, (n, k), dtype=np.uint8) << 7)
    scales = (rng.random(n if rows_scaled else (n, cols)) * .01 + .001).astype(np.float32)
    x = rand_bf16(rng, (m, k))
    x[m // 2] = 0x7fc0  # NaN
    xd, cd, sd = up(x, gpu), up(codes, gpu), up(scales, gpu)
    y = fp8lin.fp8_linear(xd, cd, sd, split=False)
    assert torch.isnan(y[m // 2]).all()
    if wide:
        for i in (0, m - 128):
            part = fp8lin.fp8_linear(xd[i:i + 128].contiguous(), cd, sd, split=False)
            assert torch.equal(y[i:i + 128].nan_to_num(1e30), part.nan_to_num(1e30))
    pair = fp8lin.linear_swiglu(xd, cd, sd, split=False)
    assert torch.equal(pair.nan_to_num(1e30), fp8lin.fused_swiglu(y).nan_to_num(1e30))
    rows = np.array([0, 127, m - 1])
    cs = np.r_[0:64, n - 64:n]
    assert_parity(bits(y)[rows][:, cs], oracle.linear(x[rows], codes[cs], scales[cs]), f"256-row tiles {m}x{n}x{k}")


# 192-row tiles of the persistent GEMM (two or three rows of them in one round
# where 256-row tiles fill half the chip to all of it): one row into a tile,
# one short of it, whole, ragged columns, the fewest K steps that choose them.
@pytest.mark.parametrize("m,n,k", [(385, 17408, 1024), (512, 17300, 512), (575, 21504, 768), (576, 20002, 1280),
                                   (512, 17408, 5120), (129, 33000, 512), (192, 32770, 1024)])
@pytest.mark.parametrize("rows_scaled", [False, True])
def test_fp8_192_row_tiles(fp8lin, gpu, oracle, m, n, k, rows_scaled):
    """Unsplit sums do not depend on the tile height: bit for bit the rows of
    calls of at most 128 rows (128-row tiles), which meet the oracle; SwiGLU
    likewise; a row of NaN stays in its row."""
    rng = np.random.default_rng(m + n + k)
    codes = rng.integers(0, 127, (n, k), dtype=np.uint8) | (rng.integers(0, 2, (n, k), dtype=np.uint8) << 7)
    scales = (rng.random(n if rows_scaled else (n, k // 128)) * .01 + .001).astype(np.float32)
    x = rand_bf16(rng, (m, k))
    x[m // 2] = 0x7fc0  # NaN
    assert plan(fp8lin, m, n, k, 1 if rows_scaled else k // 128, False)[:2] == (PERSISTENT, 192)
    xd, cd, sd = up(x, gpu), up(codes, gpu), up(scales, gpu)
    y = fp8lin.fp8_linear(xd, cd, sd, split=False)
    assert torch.isnan(y[m // 2]).all()
    parts = [fp8lin.fp8_linear(xd[i:i + 128], cd, sd, split=False) for i in range(0, m - 64, 128)]
    low = torch.cat(parts)
    assert torch.equal(y[:low.size(0)].nan_to_num(1e30), low.nan_to_num(1e30))
    rows = np.array([0, 191, m - 1])
    rows = rows[(rows < m) & (rows != m // 2)]
    cols = np.r_[0:64, n - 64:n]
    assert_parity(bits(y)[rows][:, cols], oracle.linear(x[rows], codes[cols], scales[cols]), f"192-row tiles {m}x{n}x{k}")
    pair = fp8lin.linear_swiglu(xd, cd, sd, split=False)
    assert torch.equal(pair.nan_to_num(1e30), fp8lin.fused_swiglu(y).nan_to_num(1e30))


@pytest.mark.parametrize("m", [1, 4, 27, 70, 300])
@pytest.mark.parametrize("option", ["plain", "bias", "cached", "dequant", "profiled"])
def test_engine_mlp_swiglu_forms(fp8lin, gpu, oracle, m, option):
    """LinearEngine.mlp's gate/up, one launch or two: SwiGLU of the engine's
    own product within one ulp where a split reorders sums, else bit for bit;
    three-dimensional inputs stay refused."""
    rng = np.random.default_rng(m)
    d, k = 1040, 1024
    eng = fp8lin.LinearEngine(fp8lin.LinearOptions(cublas_prefill=option == "dequant"), profile_kernels=option == "profiled",
                              weight_cache_bytes=1 << 30 if option == "cached" else 0)
    for name, rows, cols in (("l.gate_up", 2 * d, k), ("l.down_proj", 512, d - 16)):
        codes, scales = fp8lin.gen_weights(rows, cols, seed=3, tag=rows, device=gpu)
        eng.add(name + ".weight", codes, scales)
    if option == "bias":
        eng.add("l.gate_up.bias", up(rand_bf16(rng, (2 * d,)), gpu))
    if option == "cached":
        eng.build_cache()
    x = up(rand_bf16(rng, (m, k)), gpu)
    ref = fp8lin.fused_swiglu(eng.linear(x, "l.gate_up"))
    got = eng._linear_swiglu(x, "l.gate_up")
    if m in (70, 300):
        assert_parity(bits(got), bits(ref), f"mlp {option} m={m}")
    else:
        assert torch.equal(got, ref)
    with pytest.raises(fp8lin.Fp8linError):
        eng._linear_swiglu(x[None], "l.gate_up")
