"""Row kernels of the fixed-profile runtime at the edges of their splits, bit for bit against
oracle/runtime_ref.py: head sizes whose lanes cross by each step, head counts that leave slots
empty or need two and four passes, column counts off the 64 of a reduction's workgroup, and row
counts off the rows of a wave and of a statistics workgroup.  No tolerance: the arithmetic is
defined rounding by rounding."""

import pytest

from tests.test_gpu_runtime import runtime_vs_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split,axis_v", [("layer", "token"), ("layer", "channel"), ("head", "token")])
@pytest.mark.parametrize("heads,dim,tokens", [(1, 8, 1), (5, 8, 33), (3, 16, 17), (7, 32, 15), (3, 64, 16), (9, 64, 49),
                                              (1, 128, 2), (7, 128, 63), (13, 128, 5), (3, 256, 66), (8, 256, 3)])
def test_rows_at_the_edges(tmp_path, split, axis_v, heads, dim, tokens):
    if split == "head" and heads == 1:
        pytest.skip("a head split needs two heads")
    print(f"runtime rows {split} {axis_v} heads={heads} dim={dim} tokens={tokens}", flush=True)
    runtime_vs_oracle(tmp_path, 2, heads, dim, 1, 1, tokens, {"split_type": split, "axis_value": axis_v})
