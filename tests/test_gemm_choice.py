"""cch_gemm_kernel_for: which of the tiled GEMM kernels a problem goes to on 256 CUs.  Host code, no GPU."""
import csv
import math
import os

import pytest

from catccos_amd import _abi

TILE, MID1, MID2, MID3, STREAM4, STREAM8, TAIL, MID192 = range(8)
I8, E4M3, E2M1 = -1, _abi.FMT_E4M3, _abi.FMT_E2M1


def chosen(fmt, swiglu, e, t, n, k, trans_b):
    return _abi.lib().cch_gemm_kernel_for(fmt, swiglu, e, t, n, k, trans_b, 256)


def test_every_kernel_is_chosen_for_some_size():
    got = {chosen(fmt, swiglu, e, t, n, k, tb)
           for fmt in (I8, E4M3, E2M1) for e, swiglu in ((0, 0), (16, 0), (16, 1)) for tb in (0, 1)
           for t in (1, 64, 512, 3072, 16384) for n in (1024, 4096) for k in (1024, 4096, 7168)}
    assert got == set(range(7))


def test_what_the_tiled_kernels_do_not_take():
    assert chosen(E4M3, 0, 0, 64, 100, 1024, 0) == -1            # n % 8
    assert chosen(I8, 0, 0, 64, 128, 40, 0) == -1                # K no multiple of 16 bytes
    assert chosen(E4M3, 1, 4, 64, 129, 1024, 1) == -1            # no halves
    assert chosen(E4M3, 0, 0, 0, 128, 1024, 1) == -1             # no rows
    assert chosen(E4M3, 0, 257, 64, 128, 1024, 1) == -1
    assert chosen(I8, 0, 0, 16, 1 << 21, 512, 0) == TILE         # [K, N] rows of 2 MiB: the smaller kernels' offsets end there
    assert chosen(I8, 0, 0, 16, (1 << 21) - 16, 512, 0) != TILE


def test_mxfp4_scale_rows_off_dwords_never_go_to_128x256_tiles():
    for t in (64, 512, 700, 1024, 3072, 4096):
        for n in (1024, 2048, 4096, 7168):
            for e in (0, 8, 16):
                for tb in (0, 1):
                    assert chosen(E2M1, 0, e, t, n, 4160, tb) != MID3


def test_the_switch_names_a_kernel():
    L = _abi.lib()
    for bad in (-2, 7):
        assert L.cch_set_option(b"gemm_kernel", bad) == _abi.EINVAL
        assert "gemm_kernel" in L.cch_last_error().decode()
    for v in (*range(7), -1):
        assert L.cch_set_option(b"gemm_kernel", v) == _abi.OK


@pytest.mark.parametrize("fmt", [E4M3, _abi.FMT_E5M2, E2M1])
def test_one_round_of_192x192_tiles(fmt):
    """Dense products with [N, K] weights: more than two 128 x 128 tiles to a CU and at most one of 192 x 192, at either bound."""
    for t, n, k in ((3000, 3000, 448 if fmt != E2M1 else 384), (2881, 3072, 128), (1335, 6856, 256), (5466, 1528, 5120)):
        assert chosen(fmt, 0, 0, t, n, k, 1) == MID192
    assert chosen(fmt, 0, 0, 16 * 192, 16 * 192, 1024, 1) == MID192              # 256 tiles of 192 x 192
    assert chosen(fmt, 0, 0, 16 * 192 + 1, 16 * 192, 1024, 1) != MID192          # 272
    assert chosen(fmt, 0, 0, 128 * 27, 128 * 19, 1024, 1) == MID192              # 513 of 128 x 128, 234 of 192 x 192
    assert chosen(fmt, 0, 0, 128 * 32, 128 * 16, 1024, 1) != MID192              # 512
    for other in (chosen(fmt, 0, 0, 3000, 3000, 1024, 0), chosen(fmt, 0, 1, 3000, 3000, 1024, 1), chosen(fmt, 1, 0, 3000, 3008, 1024, 1),
                  chosen(fmt, 1, 16, 3000, 3008, 1024, 1), chosen(I8, 0, 0, 3000, 3000, 1024, 1)):
        assert other != MID192                                                   # [K, N], groups, SwiGLU, int8


def test_192x192_tiles_and_mxfp4_scale_rows_off_dwords():
    assert chosen(E2M1, 0, 0, 3000, 3000, 1984, 1) != MID192 and chosen(E4M3, 0, 0, 3000, 3000, 1984, 1) == MID192


def test_a_last_round_of_short_tiles_is_a_second_launch():
    for fmt, swiglu, trans_b in ((E4M3, 0, 0), (E4M3, 0, 1), (E4M3, 1, 1), (I8, 0, 1), (I8, 1, 1)):
        assert chosen(fmt, swiglu, 16, 3072, 4096, 7168, trans_b) == TAIL     # 1.2 rounds of 256 x 256 tiles
        assert chosen(fmt, swiglu, 16, 8192, 4096, 7168, trans_b) == TILE     # 2.5
    assert chosen(E4M3, 1, 16, 3072, 4096, 7168, 0) != TAIL                   # [K, N] gate and up columns


@pytest.mark.parametrize("fmt,swiglu,e,t,n,k,trans_b", [
    (E4M3, 0, 32, 5120, 4096, 7168, 1),     # 300 us on 128 x 256 tiles, 244 on 256 x 256 (means over alike to Zipf-sized groups)
    (E4M3, 1, 64, 9593, 5120, 2048, 1),     # 239, 187
    (E4M3, 1, 16, 2512, 7168, 6400, 1),     # 233, 189
    (E4M3, 0, 32, 4297, 5504, 2048, 1),     # 124, 99
    (I8, 0, 8, 1216, 6144, 2048, 1),        # 38 on 128 x 128 tiles, 31
])
def test_groups_of_nearly_whole_tiles_stay_on_256x256(fmt, swiglu, e, t, n, k, trans_b):
    assert chosen(fmt, swiglu, e, t, n, k, trans_b) in (TILE, TAIL)


@pytest.mark.parametrize("swiglu", [0, 1])
def test_the_second_launch_does_not_decide_between_tile_sizes(swiglu):
    """[N, K] weights: on either side of where a second launch is tried (32 steps of K, 1 and 1.4 rounds of tiles) the choice of tiles is the same."""
    def tiles(t, k):
        kernel = chosen(E4M3, swiglu, 16, t, 4096, k, 1)
        return TILE if kernel == TAIL else kernel
    for t in (2060, 2560, 3072, 3680):
        assert tiles(t, 3968) == tiles(t, 4096)
    for k in (4096, 5120, 7168):
        assert tiles(2040, k) == tiles(2060, k)
        assert tiles(3680, k) == tiles(3700, k)


def test_choices_against_measured_times():
    """profiles/gemm_kernel_times.csv: every kernel's time on 1300 problems that no constant was fitted to (dense ones with weights
    from HBM and from the caches, whose geometric mean counts)."""
    path = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles", "gemm_kernel_times.csv")
    times = {}
    with open(path) as f:
        for r in csv.DictReader(f):
            key = tuple(int(r[x]) for x in ("fmt", "swiglu", "experts", "t", "n", "k", "trans_b")) + (r["groups"],)
            times.setdefault(key, []).append([float(r["us%d" % i] or "inf") for i in range(7)])
    lost, of_256 = {True: [], False: []}, {True: [], False: []}
    for key, rows in times.items():
        us = [math.exp(sum(math.log(r[i]) for r in rows) / len(rows)) for i in range(7)]
        got = us[chosen(*key[:7])]
        lost[key[2] > 0].append(got / min(us[:6]))
        of_256[key[2] > 0].append(got / us[0])

    def mean(v):
        return math.exp(sum(map(math.log, v)) / len(v))
    assert len(lost[True]) > 1500 and len(lost[False]) > 200
    assert mean(lost[True]) <= 1.03 and mean(lost[False]) <= 1.02
    assert mean(of_256[True]) <= 0.76 and mean(of_256[False]) <= 0.463
    assert sum(v > 1.1 for v in of_256[True] + of_256[False]) <= 18
