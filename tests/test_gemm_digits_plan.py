"""How the products over digit planes are cut (host arithmetic behind
buddy_hip_gemm_w8_digits_plan; nothing is launched)."""
import ctypes

import pytest

PAIR, TWO = 8, 16


class Plan(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int32) for n in
                ("row_blocks", "channel_tiles", "slices", "tail_from")]


def plan(bh, M, K, N, flags=0):
    p = Plan()
    assert bh.buddy_hip_gemm_w8_digits_plan(M, K, N, flags, ctypes.byref(p)) == 0, \
        bh.buddy_hip_last_error()
    return p


@pytest.mark.parametrize("two", [0, TWO])
@pytest.mark.parametrize("K,N", [
    (65536, 65536), (65536, 65552), (131072, 32768), (131072, 49152), (1536, (1 << 22) // 24 * 16 + 16)])
def test_second_matrix_of_a_pair_is_in_reach(bh, K, N, two):
    """Tiles whose lanes reach a pair's second matrix by 32 bits are not for matrices of 2^32 bytes."""
    assert -(-K // 64) * -(-N // 16) * 1024 >= 1 << 32
    for M in [17, 31, 64, 65, 96, 97, 100, 128, 150, 192, 256, 512, 777, 1931, 2048, 4096]:
        p = plan(bh, M, K, N, PAIR | two)
        assert p.tail_from == 0 and (p.row_blocks == 1 or p.channel_tiles != 2), M


def test_large_tiles_up_to_there(bh):
    # 2^22 - 64 tiles a matrix
    p = plan(bh, 64, 4096, 65535 * 16, PAIR)
    assert (p.row_blocks, p.channel_tiles) == (2, 2)
    p = plan(bh, 512, 1536, 8960, PAIR)
    assert (p.row_blocks, p.channel_tiles, p.tail_from) == (2, 2, 7)


def test_large_tiles_alone_with_k_whole(bh):
    """o of Qwen2-1.5B, three planes: tiles of 32 x 256 two to a compute unit, not one of 64 x 256 each."""
    for M in (1100, 1400, 1600, 1800, 1931, 2000):
        p = plan(bh, M, 1536, 1536)
        assert (p.row_blocks, p.channel_tiles, p.slices) == (1, 2, 1), M


def test_refusals(bh):
    p = Plan()
    for M, K, N in [(0, 64, 16), (17, 0, 16), (17, 64, 0), (17, (1 << 17) + 1, 16), (1 << 24, 64, 16)]:
        assert bh.buddy_hip_gemm_w8_digits_plan(M, K, N, 0, ctypes.byref(p)) != 0
    assert bh.buddy_hip_gemm_w8_digits_plan(17, 64, 16, 0, None) != 0
