"""The wave-tile kernels (csrc/kvmi_tile*) against the generic row kernels on the same calls.

`fwht="rows"` forces the row kernels, which the oracle pins bit for bit with the same flag
(tests/test_gpu_configs.py, tests/test_gpu_axes.py, tests/test_gpu_sweep.py).  Every plan is held
to the kernels it means to run (kvmi_paged_kernels).  The transform on the matrix cores adds
in another fp32 order, so a value may land on the other side of a bf16 rounding boundary:
symbols one level apart on at most 1e-4 of the elements, decoded values one bf16 ulp apart
on at most 1e-3 of them (the bars of tests/test_gpu_configs.py), and over the many tokens of the
long requests a minimum or maximum one ulp and with it a scale up to two (its ulp may be half
the range's) on at most 1e-3.  Without a transform both
do the same arithmetic and have to agree bit for bit.
"""

import ctypes

import pytest
import torch

from kvserve_amd import _lib
from kvserve_amd.engine import FusedKVCodec
from kvserve_amd.profiles import rademacher_sign_bits, section_profile, whole_layer_profile

pytestmark = pytest.mark.gpu

TOP = {1: 2, 2: 3, 3: 7, 4: 15, 5: 31, 6: 60, 7: 100, 8: 200}
CT = ("channel", "token")
CASES = [
    # heads, head_dim, block, bits, layout, axes, transform, blocks
    (6, 96, 16, 4, "permuted", CT, True, 9),          # 5 tokens a tile, straddling blocks; 64 + 32 channels
    (6, 96, 16, 4, "native", CT, True, 40),
    (5, 80, 16, 3, "permuted", CT, True, 7),          # 16-channel tail, 30-byte rows
    (6, 112, 4, 7, "permuted", CT, True, 3),          # T limited by the block size
    (32, 64, 1, 5, "permuted", CT, True, 17),         # one token a tile, one-token blocks
    (7, 160, 3, 6, "native", CT, True, 5),            # block size not a power of two
    (3, 224, 16, 4, "permuted", CT, True, 2),         # whole rows staged: the most heads at 4 bits
    (12, 192, 16, 4, "permuted", CT, True, 5),        # 24 of 32 rows
    (3, 256, 8, 4, "permuted", CT, True, 6),
    (8, 128, 16, 4, "permuted", ("token", "channel"), True, 33),
    (8, 64, 16, 4, "permuted", ("tensor", "tensor"), True, 33),
    (2, 80, 16, 2, "native", ("tensor", "token"), True, 1),
    (10, 128, 16, 1, "permuted", ("channel", "channel"), True, 4),
    (8, 128, 16, 4, "permuted", CT, False, 33),
    (6, 96, 16, 8, "native", ("token", "token"), False, 9),
    (16, 80, 2, 3, "permuted", ("tensor", "channel"), False, 9),
]
# Requests long enough for the launch shapes of real ones: several tiles in a wave's image (from
# the second on its rows lie behind other tiles' rows), K and V in one workgroup (the step from
# one to the other), and with LOOPS a wave that goes on to another super-tile; the last workgroup's
# super-tiles are ragged.  (case, tiles of an image)
LOOPS = 2
LONG = [
    ((6, 96, 16, 4, "permuted", CT, True, 3001), 2, LOOPS),
    ((6, 96, 16, 3, "native", CT, True, 3001), 3, 1),
    ((8, 64, 16, 4, "permuted", ("token", "channel"), True, 4003), 4, 1),
    ((8, 64, 16, 5, "native", ("channel", "channel"), True, 4003), 3, LOOPS),
    ((20, 64, 4, 4, "permuted", CT, True, 3001), 6, 1),
    ((12, 192, 16, 4, "permuted", CT, True, 1001), 3, 1),
    ((8, 128, 16, 4, "permuted", CT, False, 2003), 2, 1),
    ((6, 96, 16, 8, "native", ("token", "token"), False, 2003), 1, LOOPS),
]


def _bits(t):
    return t.view(torch.int16).to(torch.int32)


def _unpack(stream, bits):
    body = stream[16:].to(torch.int64)
    at = torch.arange(body.numel() * 8 // bits, device=body.device) * bits
    pad = torch.nn.functional.pad(body, (0, 2))
    word = pad[at // 8] | (pad[at // 8 + 1] << 8)
    return (word >> (at % 8)) & ((1 << bits) - 1)


def _kernels(plan):
    """(family, launch shape) of the plan's call."""
    shape = (ctypes.c_int32 * 4)()
    family = _lib.load().kvmi_paged_kernels(ctypes.byref(plan.geo), plan.num_jobs, plan.max_blocks,
                                            int(plan.kind == "decompress"), shape)
    return family, tuple(shape)


FAMILY = {"mfma": _lib.KERNELS_TILE, "rows": _lib.KERNELS_ROWS}


def _run(case, pools, ids, profiles, fwht):
    H, D, S, bits, layout, axes, transform, _ = case
    codec = FusedKVCodec(H, D, S, bits, 7, transform=transform, layout=layout, axes=axes, fwht=fwht)
    plan = codec.plan_compress(pools, ids, profiles)
    assert _kernels(plan)[0] == FAMILY[fwht]
    plan.packet.kmeta.zero_()
    plan.packet.vmeta.zero_()
    plan.run()
    plan.run()  # the statistics keys are left ready for the next run
    return codec, plan


def _pools(case, gen, layers):
    H, D, S, _, _, _, _, B = case
    return [torch.randn((2, 2 * B + 3, S, H, D), generator=gen, device="cuda").to(torch.bfloat16) for _ in range(layers)]


def _profiles(case, layers):
    H, bits = case[0], case[3]
    top, low = TOP[bits], max(2, TOP[bits] // 2)
    mixed = section_profile([h % 3 == 1 for h in range(H)], top, top, low, low)
    return [mixed if l % 2 == 0 else whole_layer_profile(H, top, low) for l in range(layers)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c[:5]) + "-" + "".join(a[1] for a in c[5]) + ("" if c[6] else "-plain") + f"-{c[7]}")
def test_tile_matches_rows(case):
    _tile_vs_rows(case)


@pytest.mark.parametrize("case,tiles,loops", LONG, ids=lambda c: "-".join(str(x) for x in c[:5]) if isinstance(c, tuple) else str(c))
def test_long_requests_match_rows(case, tiles, loops):
    H, D, S, bits, layout, axes, transform, B = case
    print(f"long request {case}", flush=True)
    for family, (tokens, image, run, parts) in _tile_vs_rows(case):
        assert (image, parts) == (tiles, 2) and run >= loops * 4 * tokens * image  # 4 waves a workgroup
        assert (B * S) % (4 * tokens * image) != 0


def _tile_vs_rows(case):
    H, D, S, bits, layout, axes, transform, B = case
    layers = 2
    gen = torch.Generator(device="cuda").manual_seed(3)
    pools = _pools(case, gen, layers)
    order = torch.randperm(2 * B + 3, generator=torch.Generator().manual_seed(4)).tolist()
    profiles = _profiles(case, layers)
    tile, a = _run(case, pools, order[:B], profiles, "mfma")
    rows, b = _run(case, pools, order[:B], profiles, "rows")
    assert a.error_code() == b.error_code()
    for x, y in zip(a.packet.streams, b.packet.streams):
        if transform:
            n = bad = 0
            for lo in range(16, x.numel(), bits << 21):  # whole symbols
                d = (_unpack(x[lo - 16:lo + (bits << 21)], bits) - _unpack(y[lo - 16:lo + (bits << 21)], bits)).abs()
                assert int(d.max()) <= 1
                n, bad = n + d.numel(), bad + int((d > 0).sum())
            assert bad <= 1e-4 * n
        else:
            assert torch.equal(x, y)
    for x, y in ((a.packet.kmeta, b.packet.kmeta), (a.packet.vmeta, b.packet.vmeta)):
        if transform and B > 64:
            d = (_bits(x) - _bits(y)).abs()
            assert int(d.max()) <= 2 and int((d > 0).sum()) <= 1e-3 * d.numel()
        else:
            assert torch.equal(x, y)
    out, shapes = [], [_kernels(a)]
    for codec, fwht in ((tile, "mfma"), (rows, "rows")):
        dst = [torch.full_like(p, 7.0) for p in pools]
        plan = codec.plan_decompress(b.packet, dst, order[-B:])
        assert _kernels(plan)[0] == FAMILY[fwht]
        if fwht == "mfma":
            shapes.append(_kernels(plan))
        plan.run()
        assert plan.error_code() == b.error_code()
        out.append(dst)
    for x, y in zip(*out):
        if transform:
            d = (_bits(x) - _bits(y)).abs()
            assert int(d.max()) <= 1 and int((d > 0).sum()) <= 1e-3 * d.numel()
        else:
            assert torch.equal(x, y)
    return shapes


@pytest.mark.parametrize("case", [c for c in CASES if c[7] >= 9], ids=lambda c: f"{c[0]}-{c[1]}-{c[3]}-{c[6]}")
def test_tile_special_values(case):
    """Zeros, constants, an infinity and a NaN in a row: the same symbols, metadata and caches
    as the row kernels (a NaN takes the top level, statistics pass it over)."""
    B, transform = case[7], case[6]
    gen = torch.Generator(device="cuda").manual_seed(5)
    pools = _pools(case, gen, 1)
    order = list(range(2 * B + 3))
    pools[0][:, 0] = 0.0
    pools[0][:, 1] = 1.5
    pools[0][:, 2, 0, 0, 5] = float("inf")
    pools[0][:, 3, 0, case[0] - 1, 8] = float("-inf")
    pools[0][:, 4, 0, 0, 17] = float("nan")
    profiles = _profiles(case, 1)
    tile, a = _run(case, pools, order[:B], profiles, "mfma")
    rows, b = _run(case, pools, order[:B], profiles, "rows")
    assert a.error_code() == b.error_code()
    same = lambda x, y: torch.equal(torch.nan_to_num(x.float(), nan=123.0), torch.nan_to_num(y.float(), nan=123.0))  # noqa: E731
    assert same(a.packet.kmeta, b.packet.kmeta) and same(a.packet.vmeta, b.packet.vmeta)
    d = (_unpack(a.packet.streams[0], case[3]) - _unpack(b.packet.streams[0], case[3])).abs()
    assert int((d > 0).sum()) <= (1e-4 * d.numel() if transform else 0)
    out = []
    for codec in (tile, rows):
        dst = [torch.zeros_like(p) for p in pools]
        codec.plan_decompress(b.packet, dst, order[:B]).run()
        out.append(dst[0])
    x, y = (torch.nan_to_num(t.float(), nan=123.0, posinf=1e9, neginf=-1e9) for t in out)
    close = (x - y).abs() <= (y.abs() * 2.0 ** -7 if transform else 0.0)
    assert bool(close.all())


@pytest.mark.parametrize("case", [(6, 96, 16, 8, "permuted", CT, True, 9), (8, 128, 16, 4, "native", ("token", "channel"), True, 33),
                                  (8, 64, 16, 4, "permuted", CT, False, 40)], ids=lambda c: f"{c[0]}-{c[1]}-{c[3]}-{c[6]}")
def test_tile_decode_reads_nothing_of_a_stream_whose_header_differs(case):
    """A stream of 1-bit symbols, as long as its own header says, in the place of a wider one:
    the error word is set, the caches keep their contents, and (by the order of the kernel's
    reads) nothing behind the short stream is touched."""
    H, D, S, bits, layout, axes, transform, B = case
    gen = torch.Generator(device="cuda").manual_seed(6)
    pools = _pools(case, gen, 2)
    codec, plan = _run(case, pools, list(range(B)), _profiles(case, 2), "mfma")
    narrow = FusedKVCodec(H, D, S, 1, 7, transform=transform, layout=layout, axes=axes, fwht="mfma")
    short = narrow.compress(pools, list(range(B)), [whole_layer_profile(H, 2, 2)] * 2)
    assert short.streams[0].numel() < plan.packet.streams[0].numel()
    dst = [torch.full_like(p, 7.0) for p in pools]
    back = codec.plan_decompress(plan.packet, dst, list(range(B)))
    back.jobs[:, 2] = short.streams[0].data_ptr()
    back.run()
    assert back.error_code() == _lib.ERR_BAD_HEADER
    assert all(bool((t == 7.0).all()) for t in dst)


@pytest.mark.parametrize("case", [(6, 96, 16, 4, "permuted", CT, True, 9), (5, 80, 16, 3, "permuted", ("token", "channel"), True, 20),
                                  (8, 128, 16, 4, "native", ("channel", "channel"), True, 33)], ids=lambda c: f"{c[0]}-{c[1]}-{c[3]}")
def test_tile_overflow_in_one_channel_leaves_its_neighbours(case):
    """A finite row of 2^122 in the signs of one row of the transform: the sum of that channel
    (2^128 over 64 channels) is infinite, every other channel of the row exactly 0.  Its symbols
    and metadata are those of the row kernels, bit for bit, and so is the decoded row where a
    scale's product overflows in one channel (an infinity of either sign, no NaN)."""
    H, D, S, bits, layout, axes, transform, B = case
    gen = torch.Generator(device="cuda").manual_seed(8)
    pools = _pools(case, gen, 1)
    chunk = 128 if D == 128 else 64
    order = list(range(B))
    profiles = [whole_layer_profile(H, TOP[bits], TOP[bits])]
    signs = torch.from_numpy(rademacher_sign_bits(7, 0, H, D).view("int32")).cuda().to(torch.int64)
    e = torch.arange(chunk, device="cuda")
    for h, f in ((0, 6), (H - 1, 17)):
        parity = sum((e & f) >> b & 1 for b in range(7)) & 1
        flip = (signs[h, e // 32] >> (e % 32)) & 1
        row = torch.where((parity ^ flip).bool(), -1.0, 1.0) * 2.0 ** (122 if chunk == 64 else 121)
        pools[0][:, 3, 2, h] = 0.0
        pools[0][:, 3, 2, h, :chunk] = row.to(torch.bfloat16)
    tile, a = _run(case, pools, order, profiles, "mfma")
    rows, b = _run(case, pools, order, profiles, "rows")
    assert torch.isinf(b.packet.kmeta.float()).any() or torch.isinf(b.packet.vmeta.float()).any()
    same = lambda x, y: torch.equal(torch.nan_to_num(x.float(), nan=123.0), torch.nan_to_num(y.float(), nan=123.0))  # noqa: E731
    assert same(a.packet.kmeta, b.packet.kmeta) and same(a.packet.vmeta, b.packet.vmeta)
    shape = (2, H, B * S, D) if layout == "permuted" else (2, B * S, H, D)
    sym = [_unpack(p.packet.streams[0], bits).view(shape) for p in (a, b)]
    if layout == "native":
        sym = [s.permute(0, 2, 1, 3) for s in sym]
    for h in (0, H - 1):
        x, y = (s[:, h, 3 * S + 2] for s in sym)
        assert torch.equal(x, y), (x, y)
    # decode: one channel whose scale makes its product infinite from symbol 2 on
    part = 0 if axes[0] == "channel" else 1
    meta = (b.packet.kmeta, b.packet.vmeta)[part]
    meta[:, 0], meta[:, 1] = 0.0, 1.0
    meta[:, 1, :, 10] = 3e38
    out = []
    for codec in (tile, rows):
        dst = [torch.zeros_like(pools[0])]
        codec.plan_decompress(b.packet, dst, order).run()
        out.append(dst[0][part, order].float())
    x, y = out
    assert torch.isinf(y).any() and torch.equal(torch.isinf(x), torch.isinf(y)) and torch.equal(torch.isnan(x), torch.isnan(y))
    assert torch.equal(x[torch.isinf(y)], y[torch.isinf(y)])
