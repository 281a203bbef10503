"""cch_gemm_kernel_for: which of the tiled GEMM kernels a problem goes to on 256 CUs.  Host code, no GPU."""
import pytest

from catccos_amd import _abi

TILE, MID1, MID2, MID3, STREAM4, STREAM8, TAIL = range(7)
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


def test_a_last_round_of_short_tiles_is_a_second_launch():
    for fmt, swiglu, trans_b in ((E4M3, 0, 0), (E4M3, 0, 1), (E4M3, 1, 1), (I8, 0, 1), (I8, 1, 1)):
        assert chosen(fmt, swiglu, 16, 3072, 4096, 7168, trans_b) == TAIL     # 1.2 rounds of 256 x 256 tiles
        assert chosen(fmt, swiglu, 16, 8192, 4096, 7168, trans_b) == TILE     # 2.5
    assert chosen(E4M3, 1, 16, 3072, 4096, 7168, 0) != TAIL                   # [K, N] gate and up columns
