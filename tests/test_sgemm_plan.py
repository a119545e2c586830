"""The tile and K split that the fp32 GEMM's plan picks (sgemm_x3.hip), on the
CPU: it is host code."""
import ctypes as C

import pytest


def plan(m, n, k, ta=0, tb=0, batch=1):
    """(tile rows, tile columns, K slices, threads), or None where another
    kernel takes the product."""
    import ghostflow_hip
    f = C.CDLL(ghostflow_hip.lib()._name).gfh_internal_sgemm_x3_plan
    f.argtypes = [C.c_int, C.c_int, C.c_int64, C.c_int64, C.c_int64, C.c_int64, C.POINTER(C.c_int64)]
    out = (C.c_int64 * 4)()
    return tuple(out) if f(ta, tb, m, n, k, batch, out) else None


@pytest.mark.parametrize("m,n,k,batch", [(1 << 29, 1, 32, 1), (1 << 30, 1, 32, 1), (1 << 30, 40, 32, 1),
                                         ((1 << 31) - 1000, 8, 32, 1), (1, 1 << 21, 32, 500), (200, 1 << 21, 32, 500),
                                         (1 << 14, 1, 32, 65535)])
def test_launches_stay_within_32_bits(m, n, k, batch):
    """A grid of 2^32 threads is refused by the runtime: tiles that would need
    one are not picked."""
    bm, bn, slices, threads = plan(m, n, k, batch=batch)
    assert threads < 1 << 32


def test_beyond_every_tile():
    """Where the largest tile's grid is too large the product is left to the
    f32 tile kernel."""
    assert plan((1 << 31) - 1, 8, 32) is None and plan(1, 1 << 21, 32, batch=512) is None
    assert plan(1 << 30, 128, 32) is not None and plan(1 << 30, 129, 32) is None


def test_shapes_of_the_gpu_tests_reach_every_tile():
    """The kernel's tests name shapes, not tiles: a refit of the plan must not
    leave a tile, or its split form, without its remainders."""
    from test_sgemm_pieces_gpu import LARGE, SHAPES
    tiles = {(32, 64), (64, 64), (128, 64), (128, 128), (256, 128)}
    plans = {s: plan(*s) for s in SHAPES + LARGE}
    ragged = {s: p for s, p in plans.items() if s[0] % p[0] and s[1] % p[1] and s[2] % 32}
    assert {p[:2] for p in ragged.values()} == tiles
    assert all(plans[s][:2] == (256, 128) for s in LARGE)
    assert {p[2] > 1 for s, p in ragged.items() if s in LARGE} == {False, True}
    # the four layouts run the same tile
    for s, p in plans.items():
        assert {plan(*s, ta, tb) for ta in (0, 1) for tb in (0, 1)} == {p}


def test_long_k_of_small_products_fills_the_gpu():
    """A few tiles over a long K: enough slices for the CUs, at least four
    stages of 32 each."""
    for m, n, k in ((64, 64, 3000000), (100, 100, 500000), (33, 20, 8190), (33, 20, 2000)):
        bm, bn, slices, _ = plan(m, n, k, 0, 1)
        tiles = -(-m // bm) * -(-n // bn)
        assert min(200, k // 32 // 8) <= slices * tiles and k // 32 // slices >= 4
