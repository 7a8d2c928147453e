"""rANS blocks over the whole range of symbol frequencies, byte-equal to oracle/rans.c.

The encoder divides by a symbol's frequency through a rounded reciprocal whose form differs for
one, for powers of two and for the rest, and the decoder's table has a symbol's slots in runs
that can begin anywhere; each block here has one symbol at a chosen share and one rare one, so
that the stream's tables hold small, large, odd and power-of-two frequencies.  No tolerance:
bytes."""

import numpy as np
import pytest
import torch

from kvserve_amd import ops
from oracle import crans

pytestmark = pytest.mark.gpu

SHARES = [0, 1, 2, 3, 5, 7, 8, 9, 31, 64, 97, 255, 256, 257, 1000, 1024, 1365, 2047, 2048, 2049, 3000, 4000, 4090,
          4094, 4095, 4096]


@pytest.mark.parametrize("w", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("tail", [0, 16383, 16385])
def test_every_kind_of_frequency(cuda, w, tail):
    rng = np.random.default_rng(97 * w + tail)
    A, parts = 1 << w, []
    for i, share in enumerate(SHARES):
        m = tail if tail and i == len(SHARES) - 1 else 65536
        heavy = rng.integers(0, A)
        other = (heavy + 1 + rng.integers(0, A - 1)) % A
        s = np.full(m, other, np.uint8)
        s[: m * share // 4096] = heavy
        if A > 2 and i % 2:  # the rest of the alphabet once each
            s[m - A :] = np.arange(A)
        parts.append(rng.permutation(s))
    s = np.concatenate(parts)
    body = crans.pack(s, w)
    ref = crans.encode_packed(body, s.size, w)
    st = ops.rans_encode(torch.from_numpy(body.copy()).to(cuda), s.size, w)
    assert np.array_equal(st.cpu().numpy(), ref)
    assert np.array_equal(ops.rans_decode(st, s.size, w).cpu().numpy(), body)


@pytest.mark.parametrize("extra", [0, 4, 7])
def test_first_two_steps_take_a_word_in_every_lane(cuda, extra):
    """Symbols of frequency one at steps 0 and 1 of every lane of a sub-block, so that these steps
    read 128 words, from unit 0 of the word region (an even count) or 1 (an odd one)."""
    s = np.zeros(65536, np.uint8)
    lanes = np.arange(64)
    s[lanes * 32] = 1 + lanes
    s[lanes * 32 + 1] = 65 + lanes
    late = 5 * 2048 + 7 * 32 + 3
    s[late : late + extra] = 200 + np.arange(extra)  # an odd number of further words in one lane
    body = crans.pack(s, 8)
    ref = crans.encode_packed(body, s.size, 8)
    count = int(ref[40:44].view(np.uint32)[0]) >> 1
    assert count >= 128 and count % 2 == (extra > 0)
    st = ops.rans_encode(torch.from_numpy(body.copy()).to(cuda), s.size, 8)
    assert np.array_equal(st.cpu().numpy(), ref)
    assert np.array_equal(ops.rans_decode(st, s.size, 8).cpu().numpy(), body)
