"""CPU checks of how the prefill product's calls are routed
(logan_hip_affine_qmm_route, host code on addresses and sizes alone)."""
import ctypes as C

import pytest

from logan_amd import _lib as L

BASE = 1 << 20


def route(M, Os, I, bits, gs, fp16=False, off=(0, 0, 0)):
    """(form, tile rows, k ranges); off: bytes the weights, scales and biases
    lie past an aligned address."""
    ws = (L.Affine * len(Os))(*[L.Affine(BASE + off[0], BASE + off[1], BASE + off[2], O, I, bits, gs, int(fp16))
                                for O in Os])
    r = (C.c_int * 3)()
    rc = L.lib().logan_hip_affine_qmm_route(ws, len(Os), M, I, r)
    return tuple(r) if rc == 1 else None


@pytest.fixture(scope="module", autouse=True)
def built():
    if not L.LIB_PATH.exists():
        from logan_amd import build

        build.build()


@pytest.mark.parametrize("off", [(4, 0, 0), (8, 0, 0), (0, 2, 2), (0, 2, 0), (0, 0, 2), (4, 2, 2)])
@pytest.mark.parametrize("bits", [4, 5, 6, 8])
def test_operands_off_alignment_keep_the_tile_kernel(bits, off):
    """Weights off 16 bytes and sidecars off 4 (a row slice of a matrix with an
    odd number of groups per row) take the tile kernel above 64 rows, with the
    tiles of the aligned call: the 64 x 64 kernel forms every weight once per 64
    rows (2048 x 4096 x 4096: 282 us against 74)."""
    for M, Os, I, gs in [(100, [4096], 2880, 64), (512, [4096], 4096, 64), (2048, [4096], 4096, 64),
                         (300, [4096], 4096, 32), (65, [2880], 1920, 192), (300, [512, 130], 2048, 128)]:
        aligned, r = route(M, Os, I, bits, gs), route(M, Os, I, bits, gs, off=off)
        assert aligned[0] == 1
        # 5-bit rows are copied by dwords anyway
        assert r[0] == (1 if bits == 5 and off[1:] == (0, 0) else 2), (M, Os, I)
        assert r[1:] == aligned[1:] or (bits == 8 and gs != 64 and aligned[1] == 256)
        if r[0] == 2:
            assert route(64, Os, I, bits, gs, off=off)[0] == 0


def test_routes_fit_the_launch():
    """Partial sums fit a slot, every k range has a step, grids fit the launch
    limit of 2^32 threads; odd addresses and wide rows stay off the tile kernel."""
    for M in (1, 17, 33, 64, 65, 100, 255, 512, 1999, 4096, 65536):
        for Os in ([1], [33], [512], [4096], [12288, 64], [8192, 512, 512], [152064]):
            for I in (64, 192, 576, 2048, 2880, 14336):
                for bits in (4, 5, 6, 8):
                    for off in ((0, 0, 0), (4, 2, 2)):
                        form, rows, split = route(M, Os, I, bits, 64, off=off)
                        if form == 0:
                            continue
                        cols = sum((O + 3) & ~3 for O in Os)
                        tiles = sum((O + 127) // 128 for O in Os)
                        steps = I // 64
                        assert rows in (32, 64, 128, 192, 256)
                        assert split == 1 or split * M * cols <= 1 << 23
                        assert (split - 1) * ((steps + split - 1) // split) < steps
                        assert ((M + rows - 1) // rows * tiles * split + 7) // 8 * 8 * 512 < 1 << 32
    assert route(512, [4096], 4096, 8, 64, off=(0, 1, 0))[0] == 0
    assert route(512, [4096], 4096, 8, 64, off=(2, 0, 0)) is None
    assert route(512, [4096], 96, 8, 32) is None


def test_tile_form_cases_reach_every_form():
    """The device test's cases are routed to the tile kernel's every
    instantiation: (bits, rows, 64-code groups or not, aux type, aligned) and
    (bits, rows, groups) of the dword form."""
    from test_qmm_gpu import TILE_KINDS, TILE_OS, TILE_ROWS, tile_rows

    hit = set()
    for bits in (4, 5, 6, 8):
        for rows, M in TILE_ROWS:
            for I, gs, fp16, off in TILE_KINDS:
                r = route(M, TILE_OS, I, bits, gs, fp16, off or (0, 0, 0))
                assert r == (2 if off else 1, tile_rows(rows, bits, gs, off), 1)
                hit.add((bits, r[1], gs == 64, None if off else fp16))
    want = {(b, r, g, t) for b in (4, 5, 6, 8) for r in (32, 64, 128, 192, 256) for g in (True, False)
            for t in (True, False, None)} - {(8, 256, False, None)}
    assert hit == want
