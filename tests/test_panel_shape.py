"""The panels' host side without a GPU: the tiling that panel_shape picks, and launchers that refuse what is not
built (their callers then return an error instead of going on with the results of the call before)."""
import ctypes

import pytest

import chpe_amd as ca

PANEL, TILES = 512, {2: (32, 64, 80, 96, 112), 4: (32, 64, 80, 96, 112), 16: (32,)}
# (16-row units, 128-column groups) of every projection launch: 3B, 9B and its hybrid layers, 72B
LAUNCHES = [(160, 16), (128, 16), (1376, 16), (128, 86), (384, 32), (256, 32), (1536, 32), (256, 96), (640, 32), (772, 32),
            (640, 64), (512, 64), (3696, 64), (512, 231), (2, 32)]


class Shape(ctypes.Structure):
    _fields_ = [(n, ctypes.c_uint32) for n in ("tile", "ntt", "nrt", "ranges")]


def shape(units, ng, m, bits, room):
    f = ca.load_engine_lib()._ZN4chpe11panel_shapeEjjjjm
    f.restype, f.argtypes = Shape, [ctypes.c_uint32] * 4 + [ctypes.c_size_t]
    return f(units, ng, m, bits, room)


@pytest.mark.parametrize("bits", [2, 4, 16])
def test_shapes_are_built_and_fit(bits):
    seen = set()
    for units, ng in LAUNCHES:
        room = max(2 * units * 16 * (PANEL + 112), 32 << 20)  # (the engine's buffer at least)
        for m in range(1, PANEL + 1):
            s = shape(units, ng, m, bits, room)
            assert s.tile in TILES[bits] and (s.ntt - 1) * s.tile < m <= s.ntt * s.tile <= PANEL + 112
            assert s.ntt <= 16 and s.nrt * (8 if bits == 16 else 16) >= units
            assert 1 <= s.ranges <= min(ng, 32) and s.ranges * units * 16 * s.ntt * s.tile <= room
            seen.add(s.tile)
    assert seen == set(TILES[bits])


def test_no_room_is_no_shape():
    assert shape(640, 64, 300, 4, 640 * 16 * 300 - 1).tile == 0


def test_launchers_refuse_what_is_not_built():
    lib, args = ca.load_engine_lib(), ctypes.create_string_buffer(4096)
    gemm = lib._ZN4chpe17launch_panel_gemmERKNS_13PanelGemmArgsEjjP12ihipStream_t
    gemm.restype, gemm.argtypes = ctypes.c_bool, [ctypes.c_void_p, ctypes.c_uint32, ctypes.c_uint32, ctypes.c_void_p]
    for bits, tile in ((4, 0), (4, 48), (4, 128), (2, 0), (2, 16), (16, 0), (16, 64)):
        assert gemm(args, bits, tile, None) is False, (bits, tile)
    dn = lib._ZN4chpe15launch_dn_blockERKNS_11DnBlockArgsEP12ihipStream_t
    dn.restype, dn.argtypes = ctypes.c_bool, [ctypes.c_void_p, ctypes.c_void_p]
    assert dn(args, None) is False


def test_gpu_lengths_reach_every_tile():
    """The prompt lengths of the GPU tests take every token tile, on the 72B launches (test_gpu_models.py, both code widths)
    and on the 3B and 9B ones (test_gpu_panel.py)."""
    def tiles(launches, lengths):
        room = max(2 * max(u for u, _ in launches) * 16 * (PANEL + 112), 32 << 20)
        return {shape(u, g, m, b, room).tile for u, g in launches for m in lengths for b in (2, 4)}

    assert tiles([(640, 64), (512, 64), (3696, 64), (512, 231)], (17, 43, 70, 90, 105)) == set(TILES[4])
    assert tiles([(160, 16), (128, 16), (1376, 16), (128, 86)], (17, 32, 33, 64, 65, 90, 129, 200)) == set(TILES[4])
    assert tiles([(772, 32), (640, 32), (256, 32), (1536, 32), (256, 96)], (17, 32, 33, 65, 90, 100, 200)) == set(TILES[4])
