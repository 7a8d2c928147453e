"""Which kernels a paged call runs (kvmi_paged_kernels, host only): wave tiles only where whole
tokens of one block fill enough of a tile's 32 rows, by the rule and the measured times at
tile_faster in csrc/kvmi_tile_stats.hip.  A tile costs the same however full it is: one head in
one-token blocks filled one row of 32 and took up to 11 times the time of the kernels it
replaced."""

import ctypes

import pytest

from kvserve_amd import _lib

M, T, Q, R = _lib.KERNELS_MFMA, _lib.KERNELS_TILE, _lib.KERNELS_QUAD, _lib.KERNELS_ROWS
PLAIN, KTOK, VCH = _lib.F_NO_TRANSFORM, _lib.F_K_TOKEN, _lib.F_V_CHANNEL


def kernels(H, D, S, bits=4, flags=0, blocks=64, jobs=8):
    """((family, launch shape) of compress, the same of decode)."""
    geo = _lib.Geometry(block_size=S, num_heads=H, head_dim=D, bits=bits, max_groups=1, flags=flags)
    out = []
    for decode in (0, 1):
        shape = (ctypes.c_int32 * 4)()
        family = _lib.load().kvmi_paged_kernels(ctypes.byref(geo), jobs, blocks, decode, shape)
        assert (family == T) == (shape[0] > 0)
        out.append((family, tuple(shape)))
    return out


@pytest.mark.parametrize("H,D,S,flags,compress,decode", [
    # default axes, heads that divide 128: the quad kernels compete
    (8, 128, 16, 0, M, M), (8, 128, 1, 0, Q, Q), (4, 128, 2, 0, Q, Q), (1, 128, 1, 0, Q, Q), (1, 64, 8, 0, Q, Q),
    (8, 128, 2, 0, T, Q), (4, 128, 4, 0, T, Q), (1, 128, 16, 0, T, Q), (8, 64, 2, 0, Q, Q), (1, 64, 16, PLAIN, Q, Q),
    (8, 128, 4, PLAIN, T, T), (2, 64, 16, PLAIN, T, T), (1, 128, 1, PLAIN, Q, Q),
    # other axes, head counts and head sizes: the row kernels compete
    (1, 128, 1, KTOK, R, R), (8, 128, 1, KTOK | VCH, R, R), (8, 128, 2, KTOK | VCH, T, R), (8, 128, 4, KTOK, T, T),
    (5, 128, 1, 0, R, R), (5, 128, 2, 0, T, R), (10, 128, 1, 0, T, R), (12, 128, 2, 0, T, T),
    (6, 96, 1, 0, R, R), (8, 96, 1, 0, T, R), (12, 96, 1, 0, T, T), (6, 96, 2, 0, T, T), (6, 96, 16, 0, T, T), (1, 96, 4, 0, R, R),
    (12, 112, 1, 0, T, R), (8, 112, 1, 0, R, R), (1, 192, 16, 0, T, T), (1, 224, 16, 0, T, R),
    # one token a tile; many heads without a transform decode on the row kernels
    (17, 96, 16, 0, T, R), (20, 96, 16, 0, T, T), (32, 64, 1, KTOK, T, T), (32, 64, 16, PLAIN, T, R), (33, 64, 16, 0, R, R),
    # the LDS of a workgroup: at most one a CU compresses, two decode
    (10, 256, 16, KTOK | VCH, T, T), (10, 256, 16, VCH, T, R), (12, 256, 16, VCH, R, R), (3, 224, 16, 0, T, T), (4, 224, 16, 0, R, R),
    # forced families
    (6, 96, 16, _lib.F_ROW_FWHT, R, R), (8, 128, 16, _lib.F_VALU_FWHT, Q, Q),
])
def test_route(H, D, S, flags, compress, decode):
    (c, _), (d, _) = kernels(H, D, S, flags=flags)
    assert (c, d) == (compress, decode)


def test_route_does_not_depend_on_the_batch():
    """A request's kernels (and with them its bytes) are the same alone and in any batch."""
    for H, D, S in ((6, 96, 16), (8, 128, 2), (5, 128, 2), (1, 128, 1), (3, 224, 16)):
        for flags in (0, PLAIN, KTOK | VCH):
            got = {tuple(f for f, _ in kernels(H, D, S, flags=flags, blocks=b, jobs=j)) for b in (1, 64, 4096) for j in (1, 32, 512)}
            assert len(got) == 1, (H, D, S, flags, got)


def test_bad_geometry_is_refused():
    geo = _lib.Geometry(block_size=16, num_heads=65, head_dim=128, bits=4, max_groups=1)
    assert _lib.load().kvmi_paged_kernels(ctypes.byref(geo), 1, 1, 0, None) == _lib.EINVAL
    assert _lib.load().kvmi_paged_kernels(None, 1, 1, 0, None) == _lib.EINVAL


def test_widths_other_than_4_bits_decode_on_tiles_from_20_rows():
    for bits, decode in ((4, T), (5, R), (3, R)):
        assert [f for f, _ in kernels(12, 96, 1, bits=bits)] == [T, decode]
        assert [f for f, _ in kernels(6, 96, 16, bits=bits)] == [T, T]
