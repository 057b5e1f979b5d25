"""Products with resident bfloat16 matrices: one row and many rows, at shapes that
select every tile of the many-row kernel, against float64 sums of the same operands."""
import numpy as np
import pytest
import torch

import nukopel_oracle as N
from tile_report import tiles_run

pytestmark = pytest.mark.gpu


def make(bh, K, Nout, seed):
    rng = np.random.default_rng(seed)
    w = N.bf16(rng.standard_normal((Nout, K)) / np.sqrt(K))
    dev = torch.from_numpy(N.to_bf16_bits(w).view(np.int16)).cuda()
    tiles = torch.empty(bh.buddy_hip_bf16_tiles_bytes(K, Nout), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    assert bh.buddy_hip_pack_bf16_tiles(dev.data_ptr(), K, Nout, tiles.data_ptr(), None) == 0
    torch.cuda.synchronize()
    return w, tiles


def test_tiles_hold_what_the_layout_says(bh):
    K, Nout = 70, 21
    w, tiles = make(bh, K, Nout, 1)
    got = tiles.cpu().numpy().view(np.uint16)
    assert got.size == 2 * 4 * 512
    want = np.zeros((32, 128), np.uint16)
    want[:Nout, :K] = N.to_bf16_bits(w)
    lanes = np.arange(64)
    for g in range(2):
        for c in range(4):
            tile = got[(g * 4 + c) * 512:][:512].reshape(64, 8)
            for j in range(8):
                np.testing.assert_array_equal(
                    tile[:, j], want[g * 16 + lanes % 16, c * 32 + lanes // 16 * 8 + j])


# rows <= 16, <= 32, 64-row tiles narrow and wide, 128-row tiles; K that ends inside a
# step, a tile and a run of eight
@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("M,K,Nout", [
    (1, 64, 16), (3, 100, 40), (16, 7, 5), (16, 96, 16500), (20, 130, 65), (32, 64, 17000),
    (50, 1, 1), (64, 333, 96), (200, 192, 130), (300, 320, 4100), (513, 71, 200),
    (1000, 264, 8200), (2048, 512, 4096), (1300, 40, 12000)])
def test_many_rows(bh, M, K, Nout, dtype):
    w, tiles = make(bh, K, Nout, M + K)
    rng = np.random.default_rng(M)
    a = rng.standard_normal((M, K)).astype(np.float32)
    if dtype == 0:
        a = N.bf16(a)
    lda, ldc = (K + 7) // 8 * 8 + 8, (Nout + 15) // 16 * 16 + 4
    # what lies beside the rows must not get in
    if dtype == 0:
        buf = np.full((M, lda), 0x7FC0, np.uint16)
        buf[:, :K] = N.to_bf16_bits(a)
        A = torch.from_numpy(buf.view(np.int16)).cuda()
    else:
        buf = np.full((M, lda), np.nan, np.float32)
        buf[:, :K] = a
        A = torch.from_numpy(buf).cuda()
    C = torch.full((M, ldc), 7.0, device="cuda")
    torch.cuda.synchronize()
    assert bh.buddy_hip_gemm_bf16(A.data_ptr(), lda, dtype, tiles.data_ptr(), C.data_ptr(), ldc,
                                  M, K, Nout, None) == 0
    torch.cuda.synchronize()
    got = C.cpu().numpy()
    want = np.asarray(a, np.float64) @ w.T
    err = np.abs(got[:, :Nout] - want).max()
    assert err < 3e-6 * max(1.0, np.abs(want).max()), err
    assert (got[:, (Nout + 15) // 16 * 16:] == 7.0).all()      # nothing past the padding


def sums64(a, w):
    """float64 sums, on the GPU where the CPU would take seconds."""
    d = torch.from_numpy(np.asarray(a, np.float64)).cuda() @ torch.from_numpy(w).cuda().T
    return d.cpu().numpy()


# f32: tiles of 32 x 128 and 32 x 256 with a remainder in rows, in pairs of channel groups
# and in K: below, at and beyond a step, and fewer steps than the kernel asks for ahead.
# bfloat16: 16 x 64 tiles for the first five, 64 x 128 and 128 x 256 (see also below)
@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("M,K,Nout", [
    (17, 63, 33), (31, 64, 16), (33, 65, 48), (32, 129, 130), (65, 193, 144), (97, 1000, 8200),
    (129, 260, 40016), (2000, 1200, 4080), (1921, 1161, 4096)])
def test_wide_tiles(bh, M, K, Nout, dtype):
    w, tiles = make(bh, K, Nout, M + K)
    a = np.random.default_rng(M).standard_normal((M, K)).astype(np.float32)
    if dtype == 0:
        a = N.bf16(a)
    lda, ldc = (K + 7) // 8 * 8, (Nout + 15) // 16 * 16 + 4
    if dtype == 0:
        buf = np.full((M, lda), 0x7FC0, np.uint16)
        buf[:, :K] = N.to_bf16_bits(a)
        A = torch.from_numpy(buf.view(np.int16)).cuda()
    else:
        buf = np.full((M, lda), np.nan, np.float32)
        buf[:, :K] = a
        A = torch.from_numpy(buf).cuda()
    C = torch.full((M, ldc), 7.0, device="cuda")
    torch.cuda.synchronize()
    assert bh.buddy_hip_gemm_bf16(A.data_ptr(), lda, dtype, tiles.data_ptr(), C.data_ptr(), ldc,
                                  M, K, Nout, None) == 0
    torch.cuda.synchronize()
    got, want = C.cpu().numpy(), sums64(a, w)
    err = np.abs(got[:, :Nout] - want).max()
    assert err < 3e-6 * max(1.0, np.abs(want).max()), err
    assert (got[:, (Nout + 15) // 16 * 16:] == 7.0).all()


# the same edges of K in bfloat16, at row and channel counts for which the estimate takes
# each of the wide tiles: <RT tiles of 32 rows, GT tiles of 32 channels per wavefront>
WIDE = {(1, 1): [(129, 1, 40016), (129, 63, 40016), (161, 64, 33001), (97, 65, 24001),
                 (449, 129, 4100), (65, 193, 20020), (513, 260, 1500), (33, 8960, 6001)],
        (2, 1): [(161, 1, 40016), (225, 63, 30000), (289, 64, 24001), (97, 65, 30000),
                 (129, 129, 20020), (97, 193, 15001), (257, 260, 5000)],
        (4, 2): [(1931, 193, 20020), (257, 8960, 20020)]}


@pytest.mark.parametrize("tile,M,K,Nout", [(t, *c) for t, cs in WIDE.items() for c in cs])
def test_wide_tiles_of_bfloat16_rows(bh, tile, M, K, Nout):
    w, tiles = make(bh, K, Nout, M + K)
    a = N.bf16(np.random.default_rng(M).standard_normal((M, K)).astype(np.float32))
    lda, ldc = (K + 7) // 8 * 8, (Nout + 15) // 16 * 16 + 4
    buf = np.full((M, lda), 0x7FC0, np.uint16)
    buf[:, :K] = N.to_bf16_bits(a)
    A = torch.from_numpy(buf.view(np.int16)).cuda()
    C = torch.full((M, ldc), 7.0, device="cuda")
    torch.cuda.synchronize()
    bh.buddy_hip_variant_reset()
    assert bh.buddy_hip_gemm_bf16(A.data_ptr(), lda, 0, tiles.data_ptr(), C.data_ptr(), ldc,
                                  M, K, Nout, None) == 0
    torch.cuda.synchronize()
    assert {k for k, v in tiles_run(bh).items() if v} == {
        "rows_gemm_wide_kernel<0, %d, %d, 0, 0>" % tile}
    want = torch.from_numpy(np.asarray(a, np.float64)).cuda() @ torch.from_numpy(w).cuda().T
    err = float((C[:, :Nout] - want).abs().max())
    assert err < 3e-6 * max(1.0, float(want.abs().max())), err
    assert bool((C[:, (Nout + 15) // 16 * 16:] == 7.0).all())


def test_f32_rows_keep_every_bit_and_their_infinities(bh):
    """f32 rows go through three bfloat16 terms: a row times one weight of 1 per channel is
    the row itself, whatever its size; an infinity or a NaN reaches its own row alone."""
    M, K = 40, 96
    w = np.eye(K)
    dev = torch.from_numpy(N.to_bf16_bits(w).view(np.int16)).cuda()
    tiles = torch.empty(bh.buddy_hip_bf16_tiles_bytes(K, K), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    assert bh.buddy_hip_pack_bf16_tiles(dev.data_ptr(), K, K, tiles.data_ptr(), None) == 0
    rng = np.random.default_rng(4)
    a = (rng.standard_normal((M, K)) * 10.0 ** rng.uniform(-25, 25, (M, K))).astype(np.float32)
    a[3, 5], a[3, 6] = np.float32(3.4028235e38), np.float32(-3.4028235e38)
    w2 = rng.standard_normal((K, K))
    for weights, bad in ((w, None), (w2, np.inf), (w2, -np.inf), (w2, np.nan)):
        x = a if bad is None else rng.standard_normal((M, K)).astype(np.float32)
        if bad is not None:
            x[7, 30] = bad
        b = N.bf16(weights)
        dev = torch.from_numpy(N.to_bf16_bits(b).view(np.int16)).cuda()
        A, C = torch.from_numpy(x).cuda(), torch.empty((M, K), device="cuda")
        torch.cuda.synchronize()
        assert bh.buddy_hip_pack_bf16_tiles(dev.data_ptr(), K, K, tiles.data_ptr(), None) == 0
        assert bh.buddy_hip_gemm_bf16(A.data_ptr(), K, 1, tiles.data_ptr(), C.data_ptr(), K,
                                      M, K, K, None) == 0
        torch.cuda.synchronize()
        got = C.cpu().numpy()
        if bad is None:
            np.testing.assert_array_equal(got, x)
            continue
        rest = np.arange(M) != 7
        assert np.isfinite(got[rest]).all()
        if np.isnan(bad):
            assert np.isnan(got[7]).all()
        else:
            np.testing.assert_array_equal(got[7], bad * np.sign(b[:, 30]))


@pytest.mark.parametrize("dtype,M", [(1, 2_100_000), (0, 4_200_000)])
def test_more_row_blocks_than_a_grid_dimension_has(bh, dtype, M):
    K, Nout = 8, 16
    w, tiles = make(bh, K, Nout, 9)
    g = torch.Generator(device="cuda").manual_seed(1)
    A = torch.randn((M, K), generator=g, device="cuda").to(torch.float32 if dtype else torch.bfloat16)
    C = torch.zeros((M, Nout), device="cuda")
    torch.cuda.synchronize()
    assert bh.buddy_hip_gemm_bf16(A.data_ptr(), K, dtype, tiles.data_ptr(), C.data_ptr(), Nout,
                                  M, K, Nout, None) == 0
    torch.cuda.synchronize()
    want = A.double() @ torch.from_numpy(w).cuda().T
    assert float((C - want).abs().max()) < 3e-6 * float(want.abs().max())


@pytest.mark.parametrize("M,K,Nout", [(17, 96, 33), (40, 100, 130), (33, 1000, 8200)])
def test_f32_rows_times_infinite_weights(bh, M, K, Nout):
    """An infinite weight makes its channel infinite with the sign of the product, whatever
    terms the row's value has; NaN beside another infinity or a row's zero.  Every other
    channel is what it is without."""
    rng = np.random.default_rng(K)
    w = N.bf16(rng.standard_normal((Nout, K)))
    a = rng.standard_normal((M, K)).astype(np.float32)
    a[::2] = N.bf16(a[::2])   # one term
    a[1, 50] = 0.0
    w[7, 50], w[20, 90], w[Nout - 1, K - 1] = np.inf, -np.inf, np.inf
    w[21, 3], w[21, 4] = np.inf, np.inf  # +-inf or NaN, by the signs of two values
    dev = torch.from_numpy(N.to_bf16_bits(w).view(np.int16)).cuda()
    tiles = torch.empty(bh.buddy_hip_bf16_tiles_bytes(K, Nout), dtype=torch.uint8, device="cuda")
    lda, ldc = (K + 7) // 8 * 8, (Nout + 15) // 16 * 16
    buf = np.full((M, lda), np.nan, np.float32)
    buf[:, :K] = a
    A, C = torch.from_numpy(buf).cuda(), torch.empty((M, ldc), device="cuda")
    torch.cuda.synchronize()
    assert bh.buddy_hip_pack_bf16_tiles(dev.data_ptr(), K, Nout, tiles.data_ptr(), None) == 0
    assert bh.buddy_hip_gemm_bf16(A.data_ptr(), lda, 1, tiles.data_ptr(), C.data_ptr(), ldc,
                                  M, K, Nout, None) == 0
    torch.cuda.synchronize()
    got = C.cpu().numpy()[:, :Nout]
    with np.errstate(invalid="ignore"):
        want = a.astype(np.float64) @ w.astype(np.float64).T
    assert np.isnan(want).any() and np.isinf(want).any()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    fin = np.isfinite(want)
    assert np.abs(got[fin] - want[fin]).max() < 3e-6 * np.abs(want[fin]).max()


@pytest.mark.parametrize("K,Nout", [(64, 16), (1, 3), (37, 50), (2048, 96), (2052, 70), (4100, 33),
                                    (8200, 17), (9001, 20), (1536, 40000), (300, 4100)])
def test_one_row(bh, K, Nout):
    w, tiles = make(bh, K, Nout, K)
    x = np.random.default_rng(K).standard_normal(K).astype(np.float32)
    X = torch.from_numpy(x).cuda()
    y = torch.empty((Nout + 15) // 16 * 16, device="cuda")
    torch.cuda.synchronize()
    assert bh.buddy_hip_gemv_bf16(X.data_ptr(), tiles.data_ptr(), y.data_ptr(), K, Nout, None) == 0
    torch.cuda.synchronize()
    want = w @ x.astype(np.float64)
    err = np.abs(y.cpu().numpy()[:Nout] - want).max()
    assert err < 3e-6 * max(1.0, np.abs(want).max()), err


def test_refusals(bh):
    t = torch.zeros(4096, device="cuda")
    p = t.data_ptr()
    ok = (p, 64, 1, p, p, 16, 4, 64, 16, None)
    for i, bad in ((1, 60), (1, 32), (2, 5), (5, 8), (5, 18), (0, p + 4), (6, 0)):
        args = list(ok)
        args[i] = bad
        assert bh.buddy_hip_gemm_bf16(*args) != 0
    assert bh.buddy_hip_gemv_bf16(None, p, p, 64, 16, None) != 0
    assert bh.buddy_hip_bf16_tiles_bytes(0, 4) == 0


# The tile of 128 rows, which come past the registers: no whole step of 64 k, one to seven of them
# (a ring of four, its rounds and every rest of one), and what is left of K behind them
@pytest.mark.parametrize("M,K,Nout", [(1931, 40, 30000), (1931, 64, 30000), (1931, 100, 12001), (1931, 128, 12000),
                                      (1025, 230, 12001), (1025, 256, 12000), (1025, 320, 12000), (257, 390, 20016),
                                      (257, 448, 20016)])
def test_steps_of_the_tile_of_128_rows(bh, M, K, Nout):
    test_wide_tiles_of_bfloat16_rows(bh, (4, 2), M, K, Nout)


# The tile of 128 rows goes two to a compute unit: a few more than one to each, and no more than that
@pytest.mark.parametrize("tile,M,K,Nout", [((2, 1), 777, 2048, 11008), ((4, 2), 640, 2048, 11008)])
def test_where_the_tile_of_128_rows_fills_the_chip(bh, tile, M, K, Nout):
    test_wide_tiles_of_bfloat16_rows(bh, tile, M, K, Nout)
