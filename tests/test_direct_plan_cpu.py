"""Which tile, and how many pieces of K, a product over operands in memory takes (gemm_direct.hip.h's two estimates): host code, looked at without a GPU."""
import ctypes as C
import itertools

import pytest

from ntransformer_amd import _lib

# rows, columns, tiles at once on a CU, us a chunk alone / beside others, us beside the chunks, the part that goes with the rows a tile has
BF16 = [(256, 256, 1, 1.45, 1.45, 12, 0), (256, 128, 1, .84, .84, 9, 0), (128, 256, 1, .85, .85, 9, 0), (128, 128, 2, .72, .475, 7, 0), (128, 128, 1, .50, .57, 7, 0), (64, 128, 2, .42, .35, 5, 0),
        (64, 64, 3, .33, .22, 4, 0)]
HALF = [(128, 256, 1, 1.65, 1.65, 12, .6), (64, 128, 2, .82, .495, 5, 0), (64, 64, 2, .47, .315, 4, 0)]
COUNTS = (1, 2, 3, 4, 5, 6, 8, 12, 16)


def plan(fn, *args):
    f = getattr(_lib.lib(), fn)
    f.argtypes, f.restype = [C.c_int] * (len(args) - 1) + [C.c_longlong, C.POINTER(C.c_int)], C.c_int
    out = (C.c_int * 4)()
    _lib.check(f(*args, out), fn)
    return tuple(out)


def bf16(rows, groups, N, K, room=1 << 40):
    return plan("ntk_dense_direct_plan", rows, groups, N, K, room)


def half(rows, N, K, room=1 << 40):
    return plan("ntk_gemm_half_plan", rows, N, K, room)


def estimates(forms, rows, groups, N, K, cut):
    """(first, second estimate, plan) of every form and count of pieces, in 64 bits"""
    chunks, out = -(-K // 64), []
    for i, (TM, TN, res, alone, busy, over, even) in enumerate(forms):
        mean = rows / groups / TM
        row_tiles = groups * (1.0 if mean < 0.5 else mean + 0.5) if groups > 1 else -(-rows // TM)
        tiles = row_tiles * -(-N // TN)
        for s in COUNTS:
            if s > 1 and (not cut or chunks < 4 * s):
                break
            n = int((tiles * s + 255) // 256)
            each, rest = -(-chunks // s) * (1 - even * (1 - min(1, mean / row_tiles))), n % res
            beside = over * -(-n // res) + (3 + (s + 1) * rows * N * 4 / 7e6 if s > 1 else 0)
            one = each * (alone if n == 1 else n * busy) + beside
            two = each * (alone if n == 1 else (n - rest) * busy + (max(alone, rest * busy) if rest else 0)) + beside
            out.append((1e30 if s == 5 else one, two if s != 5 or tiles * 6 > 256 else 1e30, (TM, TN, res, s)))
    return out


def expected(forms, rows, groups, N, K, cut, both):
    """the plans that may be taken (both sides of a comparison within a rounding of 32 bits): the first estimate's, or (both) the second one's that has its tile in fewer pieces or is ahead by a tenth"""
    e = estimates(forms, rows, groups, N, K, cut)
    best = min(x[0] for x in e)
    near = lambda a, b: a <= b * (1 + 1e-5)
    ok = set()
    for one, two, p in e:
        if near(one, best):
            least = min(x[1] for x in e)
            for q in [q for _, t, q in e if near(t, least)] if both else [p]:
                fewer = q[:3] == p[:3] and q[3] < p[3]
                if fewer or near(least * 1.1, two):
                    ok.add(q)
                if not fewer and not least * 1.1 * (1 + 1e-5) < two:
                    ok.add(p)
    return ok


SIZES = list(itertools.product((9, 33, 65, 150, 200, 273, 464, 700, 1053, 1500, 1999), (512, 1536, 2048, 4096, 6240, 7488, 14976), (768, 1536, 2048, 4096, 7488)))


def test_plans_are_those_of_the_two_estimates():
    for rows, N, K in SIZES:
        assert bf16(rows, 1, N, K) in expected(BF16, rows, 1, N, K, True, True), (rows, N, K)
        assert bf16(rows, 1, N, K, 0) in expected(BF16, rows, 1, N, K, False, True), (rows, N, K)
        assert half(rows, N, K) in expected(HALF, rows, 1, N, K, True, True), (rows, N, K)
        assert half(rows, N, K, 0) in expected(HALF, rows, 1, N, K, False, True), (rows, N, K)
        for groups in (8, 32):
            assert bf16(rows, groups, N, K, 0) in expected(BF16, rows, groups, N, K, False, False), (rows, groups, N, K)


@pytest.mark.parametrize("args,want", [
    # one tile a CU at the pace of a tile alone: 19 .. 27 us a unit each, 24 .. 31 in the tiles of 64 columns
    ((150, 1, 14976, 2048, 0), (128, 128, 1, 1)), ((273, 1, 7488, 2048, 0), (128, 128, 1, 1)), ((178, 1, 14976, 1536, 0), (128, 128, 1, 1)), ((1463, 1, 2048, 2048), (128, 128, 1, 1)),
    # groups: the first estimate alone
    ((1024, 8, 2048, 2048, 0), (128, 128, 1, 1)), ((300, 8, 4096, 2048, 0), (128, 128, 1, 1)),
    # the second estimate where it is clearly ahead, or has the same tile in fewer pieces
    ((150, 1, 2048, 2048), (64, 64, 3, 5)), ((186, 1, 2144, 1600), (64, 64, 3, 4)),
    ((1438, 1, 11008, 4096, 0), (128, 128, 2, 1)), ((65, 1, 6240, 2048), (64, 64, 3, 1)), ((700, 1, 4096, 14336), (256, 256, 1, 5)), ((1181, 1, 7488, 7488, 0), (256, 256, 1, 1))])
def test_plans_by_name(args, want):
    assert bf16(*args) == want


def test_room_bounds_the_pieces():
    for rows, N, K in SIZES:
        for pieces in (0, 1, 2, 5, 7):
            assert bf16(rows, 1, N, K, pieces * rows * N)[3] <= max(pieces, 1) and half(rows, N, K, pieces * rows * N)[3] <= max(pieces, 1)


@pytest.mark.parametrize("T,N,K,norm,gate", [(65, 2048, 256, 0, 0), (24, 4096, 256, 0, 0), (300, 1024, 256, 0, 0), (1000, 2048, 256, 1, 1), (48, 512, 768, 1, 0), (24, 1024, 768, 1, 0), (24, 1024, 1024, 1, 1),
                                             (12, 4096, 4096, 1, 1), (150, 1024, 2048, 1, 1), (128, 4096, 1024, 1, 1), (1024, 3072, 768, 1, 1), (1999, 2048, 2048, 1, 1), (8, 4096, 4096, 0, 0),
                                             (65, 2048, 2050, 0, 0)])
def test_rows_left_as_bfloat16_where_that_is_ahead(T, N, K, norm, gate):
    """(up to 8 rows, and rows of no whole chunks, the direct form does not take at all)"""
    f = _lib.lib().ntk_dense_direct_ahead
    f.argtypes, f.restype = [C.c_int] * 4 + [C.c_size_t], C.c_int
    assert (f(T, N, K, 0, 64 << 20), f(T, N, K, 1, 64 << 20)) == (norm, gate)
