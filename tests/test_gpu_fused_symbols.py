"""Symbols of the fused quantizer where its quotient lies on or beside a rounding boundary, byte
for byte against oracle/fused_v3.py, whose division is numpy's correctly rounded one: rows of
few small whole numbers, whose transforms put (y - min) / scale on halves and a rounding beside
them, over scales from 1e-30 to 1e30 and levels from 2 to 255.  The float16 tables are the float
ones rounded once, and a scale without a finite value gives symbol 0.  No tolerance: bytes."""

import ctypes

import numpy as np
import pytest
import torch

from kvserve_amd import _lib
from kvserve_amd.profiles import rademacher_sign_bits
from oracle import fused_v3 as fv
from oracle import kvpipe as kp

pytestmark = pytest.mark.gpu
SEED = 0xC0FEBABE


def _compress(dev, x, levels, vgroup, D, f16):
    lib = _lib.load()
    rows, H = x.shape[1], x.shape[2]
    signs = torch.from_numpy(rademacher_sign_bits(SEED, 1, H, D).view("int32")).to(dev)
    q = torch.empty((2, rows, H, D), dtype=torch.uint8, device=dev)
    k = torch.empty((2, H, D), dtype=torch.float32, device=dev)
    v = torch.empty((2, rows, H), dtype=torch.float32, device=dev)
    ws = torch.empty(int(lib.kvmi_v3_scratch_bytes(rows, H, D)), dtype=torch.uint8, device=dev)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    head = (x.data_ptr(), rows, H, D, signs.data_ptr(), levels.data_ptr(), vgroup.data_ptr(), q.data_ptr())
    if not f16:
        _lib.check(lib.kvmi_v3_compress(*head, k.data_ptr(), v.data_ptr(), ws.data_ptr(), stream), "compress")
        torch.cuda.synchronize()
        return q, k, v
    k16 = torch.empty((2, H, D), dtype=torch.float16, device=dev)
    v16 = torch.empty((2, rows, H), dtype=torch.float16, device=dev)
    _lib.check(lib.kvmi_v3_compress_f16(*head, k16[0].data_ptr(), k16[1].data_ptr(), v16[0].data_ptr(),
                                        v16[1].data_ptr(), k.data_ptr(), ws.data_ptr(), stream), "compress_f16")
    torch.cuda.synchronize()
    return q, k16, v16


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("exponent", [-100, -17, 0, 9, 100])
@pytest.mark.parametrize("levels", [(2, 3), (16, 12), (255, 100), (9, 6)])
def test_symbols_on_the_boundaries(cuda, D, exponent, levels):
    rows, H = 333, 4
    rng = np.random.default_rng([D, exponent + 200, levels[0]])
    x = rng.integers(-3, 4, (2, rows, H, D)) * (rng.random((2, rows, H, D)) < rng.choice([0.02, 0.1, 0.5, 1.0], (2, rows, 1, 1)))
    t = (torch.from_numpy(x.astype(np.float32)) * 2.0 ** exponent).to(torch.bfloat16)
    kl, vl = [float(levels[0])] * H, [float(levels[1]), float(levels[0])] * (H // 2)
    ref_q, ref_m = fv.compress_layer(t.view(torch.int16).numpy().view(np.uint16), kp.rademacher_signs(SEED, 1, H, D), kl, vl)
    lv = torch.tensor([kl, vl], dtype=torch.float32, device=cuda)
    group = torch.tensor([0, 1] * (H // 2), dtype=torch.int32, device=cuda)
    q, k, v = _compress(cuda, t.to(cuda), lv, group, D, False)
    assert np.array_equal(q.cpu().numpy(), ref_q)
    for got, want in ((k, ("kmin", "kscale")), (v, ("vmin", "vscale"))):
        for i, name in enumerate(want):
            assert np.array_equal(got[i].cpu().numpy(), ref_m[name]), name
    q16, k16, v16 = _compress(cuda, t.to(cuda), lv, group, D, True)
    assert torch.equal(q16, q) and torch.equal(k16, k.half()) and torch.equal(v16, v.half())


@pytest.mark.parametrize("rows,H,D", [(4111, 8, 128), (16391, 2, 64), (2049, 16, 128), (9031, 8, 128), (16403, 8, 64)])
def test_layers_of_several_passes_a_workgroup(cuda, rows, H, D):
    """More passes than workgroups (two or three each), or an odd number of them, the last one
    ragged."""
    t = torch.randn((2, rows, H, D), generator=torch.Generator().manual_seed(rows)).to(torch.bfloat16)
    kl, vl = [16.0] * H, [12.0, 6.0] * (H // 2)
    ref_q, ref_m = fv.compress_layer(t.view(torch.int16).numpy().view(np.uint16), kp.rademacher_signs(SEED, 1, H, D), kl, vl)
    lv = torch.tensor([kl, vl], dtype=torch.float32, device=cuda)
    group = torch.tensor([0, 1] * (H // 2), dtype=torch.int32, device=cuda)
    q, k, v = _compress(cuda, t.to(cuda), lv, group, D, False)
    assert np.array_equal(q.cpu().numpy(), ref_q)
    assert np.array_equal(v[1].cpu().numpy(), ref_m["vscale"]) and np.array_equal(k[1].cpu().numpy(), ref_m["kscale"])


def test_scales_without_a_finite_value_give_zero(cuda):
    """(y - min) over an infinite or undefined range is zero or undefined, and either is symbol 0."""
    H, D = 2, 128
    t = torch.randn((2, 8, H, D), generator=torch.Generator().manual_seed(2)).to(torch.bfloat16)
    t[:, 3, 0, 5], t[:, 5, 1, 7] = float("inf"), float("nan")
    lv = torch.full((2, H), 16.0, device=cuda)
    q, _, _ = _compress(cuda, t.to(cuda), lv, torch.tensor([0, 1], dtype=torch.int32, device=cuda), D, False)
    assert not q[1, 3, 0].any() and not q[1, 5, 1].any() and q[1, 3, 1].any() and q[1, 4].any()
    assert not q[0, :, 0].any()  # one infinity spreads over every channel of its head's row


@pytest.mark.parametrize("H,D", [(64, 128), (32, 64)])
def test_a_few_rows_of_many_heads_take_no_longer_than_a_pass_of_them(cuda, H, D):
    """K's passes are by head: one row of H heads is H passes, which run side by side.  The least
    of 20 timings of one row is within 1.5 times that of 64 rows, which have the same passes with
    every lane in use (one workgroup running them in turn took 5 to 8 times as long)."""
    lv, group = torch.full((2, H), 12.0, device=cuda), torch.zeros(H, dtype=torch.int32, device=cuda)
    lib, least = _lib.load(), {}
    for rows in (1, 64):
        x = torch.randn((2, rows, H, D), generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(cuda)
        signs = torch.zeros((H, D // 32), dtype=torch.int32, device=cuda)
        q, k = torch.empty_like(x, dtype=torch.uint8), torch.empty((2, H, D), device=cuda)
        v = torch.empty((2, rows, H), device=cuda)
        ws = torch.empty(int(lib.kvmi_v3_scratch_bytes(rows, H, D)), dtype=torch.uint8, device=cuda)
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        times = []
        for _ in range(20):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                _lib.check(lib.kvmi_v3_compress(x.data_ptr(), rows, H, D, signs.data_ptr(), lv.data_ptr(), group.data_ptr(),
                                                q.data_ptr(), k.data_ptr(), v.data_ptr(), ws.data_ptr(), stream), "compress")
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        least[rows] = min(times)
    assert least[1] <= 1.5 * least[64], least
