"""CPU checks of the geometry header the host code, the debug exports and every kernel share
(dl_templates_amd/csrc/dlt_geom.h): window ranges against the oracle's neighbour masks
(src/tiled_swa.py:701-713), the idx decode (src/fused_rope2d.py:40-45), the token -> pixel map of the
image layout (src/tiled_swa.py:753-755), the exact multiply-shift division it uses, and the split of a grid into bands.  The header is
compiled with the host compiler through tests/geom_shim.cpp; no GPU is involved."""
import ctypes
import os
import random
import shutil
import subprocess

import numpy as np
import pytest

from oracle import attn_oracle as orc

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    out = str(tmp_path_factory.mktemp("geom") / "libgeom_shim.so")
    subprocess.run([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "geom_shim.cpp"), "-o", out], check=True)
    lib = ctypes.CDLL(out)
    lib.shim_fastdiv.restype = ctypes.c_uint
    lib.shim_fastdiv.argtypes = [ctypes.c_uint, ctypes.c_uint]
    return lib


def test_fastdiv_is_exact_below_2_pow_31(shim):
    rng = random.Random(0)
    divisors = [1, 2, 3, 5, 7, 16, 17, 48, 63, 64, 65, 100, 4095, 4096, 4097, 65535, 65537, 1000003, (1 << 30) - 1, 1 << 30,
                (1 << 31) - 1] + [rng.randrange(1, 1 << rng.randrange(1, 31)) for _ in range(200)]
    for d in divisors:
        edge = [0, 1, d - 1, d, d + 1, 2 * d - 1, 2 * d, (1 << 31) - 1, ((1 << 31) - 1) // d * d, ((1 << 31) - 1) // d * d - 1]
        for n in edge + [rng.randrange(0, 1 << 31) for _ in range(50)]:
            n = max(0, min(n, (1 << 31) - 1))
            assert shim.shim_fastdiv(n, d) == n // d, (n, d)


@pytest.mark.parametrize("th,tw,bh,bw", [(2, 3, 4, 4), (3, 2, 2, 5), (4, 5, 1, 1), (1, 4, 3, 1), (5, 1, 1, 7), (16, 16, 4, 4), (7, 9, 6, 8)])
def test_token_pixel_map_matches_the_oracle(shim, th, tw, bh, bw):
    index = orc.image_token_index(th, tw, bh, bw)              # [IH, IW] -> token
    y, x = ctypes.c_uint(), ctypes.c_uint()
    for n in range(th * tw * bh * bw):
        shim.shim_token_pixel(bh, bw, tw, n, ctypes.byref(y), ctypes.byref(x))
        assert index[y.value, x.value] == n
    i = ctypes.c_uint()
    S = bh * bw
    for xs in range(tw * S):                                    # slot inside one grid row
        shim.shim_slot_pixel(bh, bw, tw, xs, ctypes.byref(i), ctypes.byref(x))
        assert index[i.value, x.value] == xs                    # grid row 0: token == slot


def test_window_ranges_match_the_neighbour_masks(shim):
    out = (ctypes.c_int * 8)()
    rng = random.Random(1)
    for _ in range(60):
        th, tw, S = rng.randint(1, 6), rng.randint(1, 7), rng.choice([1, 1, 2, 16])
        WR, WC = rng.randint(0, 4), rng.randint(0, 4)
        mask = orc.neighbor_mask(th, tw, WR, WC)
        XL = tw * S
        for r in range(th):
            for c in range(tw):
                x = c * S + rng.randrange(S)
                shim.shim_key_range(0, th, tw, S, min(WR, th), min(WC, tw), XL, XL, r, x, out)
                got = np.zeros((th, tw), dtype=bool)
                assert out[2] % S == 0 and out[3] % S == 0
                got[out[0]:out[1] + 1, out[2] // S:out[3] // S] = True
                assert np.array_equal(got.reshape(-1), mask[r * tw + c])
                assert list(out[4:8]) == list(out[0:4])      # the window is symmetric: queries of a key == keys of a query


def test_dense_and_causal_ranges(shim):
    out = (ctypes.c_int * 8)()
    shim.shim_key_range(1, 1, 1, 1, 0, 0, 50, 70, 0, 13, out)     # dense: every key, every query
    assert list(out) == [0, 0, 0, 70, 0, 0, 0, 50]
    shim.shim_key_range(2, 1, 1, 1, 0, 0, 64, 64, 0, 13, out)     # causal: keys 0..13, queries 13..63
    assert list(out) == [0, 0, 0, 14, 0, 0, 13, 64]


def test_idx_decode_matches_the_oracle(shim):
    vals = [-1, 0, 0xFFFF, 0x7FFF0000 | 5, (3 << 16) | 0xFFFF, (0x8000 << 16) | 7, (12 << 16) | 34, -65536, 65535]
    vals = [v - (1 << 32) if v >= (1 << 31) else v for v in vals]
    rows, cols = orc.decode_idx(np.array(vals, dtype=np.int32))
    for v, r, c in zip(vals, rows, cols):
        assert shim.shim_rope_row(v) == r and shim.shim_rope_col(v) == c


def test_band_plan_is_the_best_split_and_cheap_to_find(shim):
    """Same split as a search over every band count, in at most 2 sqrt(n) + 2 steps, and few where the grid is long and thin: the plan
    is made in front of every launch."""
    def search(units, cols, slots):
        best = None
        for nb in range(1, units + 1):
            per = -(-units // nb)
            if -(-units // per) == nb:
                cost = -(-cols * nb // slots) * (per + 2)
                if best is None or cost < best[0]:
                    best = (cost, per, nb)
        return best[1:]

    per, nb = ctypes.c_int(), ctypes.c_int()
    plan = lambda units, cols, slots: shim.shim_band_plan(units, ctypes.c_longlong(cols), ctypes.c_longlong(slots), ctypes.byref(per), ctypes.byref(nb))
    rng = random.Random(2)
    for _ in range(3000):
        units, cols, slots = rng.choice([rng.randint(1, 40), rng.randint(1, 2000)]), int(2 ** rng.uniform(0, 12)), rng.choice([1, 7, 256, 512])
        tried = plan(units, cols, slots)
        assert (per.value, nb.value) == search(units, cols, slots), (units, cols, slots)
        assert tried <= 2 * units ** 0.5 + 2
    for units in (65536, 262144, 2 ** 28):
        for cols in (1, 8, 64, 4096):
            assert plan(units, cols, 512) <= 1100, (units, cols)


def test_image_forward_alone_only_where_it_is_faster(shim):
    """One workgroup per CU: full strips of 8 tiles, 1, 2 or 4 full rounds of them, many rows, 8 heads and more (256 CUs)."""
    def alone(B, H, th, tw, d=32, S=16, WR=1, WC=1):
        return bool(shim.shim_image_fwd_alone(d, S, WR, WC, th, tw, H, ctypes.c_longlong(B * H * -(-tw * S // 128)), ctypes.c_longlong(256)))

    for shape in [(4, 8, 64, 64), (32, 8, 64, 8), (8, 8, 40, 64), (16, 8, 48, 64), (4, 8, 100, 60), (8, 8, 64, 62),
                  (2, 16, 32, 64), (4, 16, 24, 60), (8, 16, 32, 64), (3, 32, 24, 40)]:
        assert alone(*shape), shape
    for shape in [(128, 8, 32, 1), (64, 8, 24, 5), (16, 8, 64, 9), (32, 8, 64, 7), (8, 8, 64, 33), (2, 8, 96, 61),     # ragged strips
                  (4, 8, 63, 64), (32, 8, 16, 8), (8, 8, 39, 64), (8, 8, 1, 64), (16, 8, 47, 64), (2, 16, 31, 64), (4, 16, 23, 64),   # few rows
                  (12, 8, 64, 64), (20, 8, 64, 64), (24, 8, 64, 64), (6, 8, 64, 64), (4, 32, 64, 56),                      # other rounds
                  (16, 2, 64, 64), (8, 7, 64, 64), (3, 8, 64, 64)]:                                                        # heads, idle CUs
        assert not alone(*shape), shape
    assert not alone(4, 8, 64, 64, d=64) and not alone(4, 8, 64, 64, S=32) and not alone(4, 8, 64, 64, WC=2) and not alone(4, 8, 64, 64, WR=2)


def test_narrow_tile_grids_take_two_backward_launches(shim):
    """d = 32: grids of few tile columns with 12 rows and more per CU (256 CUs); everything else with a 3 x 3 window of 16-token tiles is one launch."""
    one = lambda slabs, th, tw, img, d=32, S=16, WR=1, WC=1: bool(
        shim.shim_tile_bwd_one_launch(d, S, WR, WC, img, tw, ctypes.c_longlong(slabs * th), ctypes.c_longlong(256)))
    for slabs, th, tw in [(256, 24, 1), (512, 6, 3), (1024, 6, 5), (64, 64, 2)]:
        assert not one(slabs, th, tw, 0) and one(slabs, th, tw, 1) == (tw > 2)
        assert one(slabs, th, tw, 0, d=64)
    for slabs, th, tw in [(64, 6, 1), (256, 11, 5), (1024, 64, 6), (4, 2000, 8)]:
        assert one(slabs, th, tw, 0) and one(slabs, th, tw, 1)
    assert not one(4, 16, 16, 0, S=32) and not one(4, 16, 16, 0, WC=2) and not one(4, 16, 16, 0, WR=2)


def test_flash_backward_workgroups_of_64_tokens(shim):
    """One per CU, two under a mask; dK/dV at 64/128 under a mask always below 3072 keys and up to four per CU below 8192 (256 CUs)."""
    def small(slabs, own, causal, kv_64_128):
        return bool(shim.shim_flash_bwd_64(causal, kv_64_128, own, ctypes.c_longlong(slabs * -(-own // 64)), ctypes.c_longlong(256)))

    for kv in (0, 1):
        assert small(8, 2048, 0, kv) and not small(12, 2048, 0, kv) and small(1, 16384, 0, kv)
        assert small(8, 4096, 1, kv) and small(2, 16384, 1, kv) and not small(4, 12000, 1, kv)
    for slabs, own in [(10, 4096), (16, 4096), (8, 6000), (6, 8192), (8, 8192), (64, 2048), (256, 1024)]:
        assert small(slabs, own, 1, 1) and not small(slabs, own, 1, 0), (slabs, own)
    for slabs, own in [(17, 4096), (32, 4096), (9, 8192), (4, 8200)]:
        assert not small(slabs, own, 1, 1), (slabs, own)


def test_band_plan_of_the_long_band_cases(shim):
    """tests/test_swa_tiles_gpu.py means its LONG_BANDS to march beyond the ring of 3 rows, over several strips, the last one ragged (256 CUs)."""
    from tests.test_swa_tiles_gpu import LONG_BANDS
    per, nb = ctypes.c_int(), ctypes.c_int()
    for th, tw, slabs, d in LONG_BANDS:
        strip = 8 if d == 32 else 4   # tiles
        strips = -(-tw // strip)
        assert shim.shim_tile_bwd_one_launch(d, 16, 1, 1, 0, tw, ctypes.c_longlong(slabs * th), ctypes.c_longlong(256)) and strips > 1 and tw % strip
        shim.shim_band_plan(th, ctypes.c_longlong(slabs * strips), ctypes.c_longlong(256), ctypes.byref(per), ctypes.byref(nb))
        assert per.value > 4, (th, tw, slabs, d, per.value)
