"""Which kernels a reference-rounding decode call runs (nie_paged_decode_kernel, the
decision that the call itself takes), checked without a GPU."""

from __future__ import annotations

import os
import subprocess
import sys

import pytest
import torch

from nano_infer_engine import _native

#: scores a wave of decode_ring_kernel keeps: 16-key tiles x query heads of a group
RING_SCORE_ROWS = {64: 128, 128: 256}


def _kernel(q_heads, kv_heads, head_dim, lens=None, batch=0, bound=0, block_size=16):
    """The kernel of a call with host lengths, or of a device-planned one within (batch, bound)."""
    if lens is not None:
        return _native.decode_kernel(torch.bfloat16, q_heads, kv_heads, head_dim, block_size, len(lens), max(lens),
                                     sum(lens), seq_lens_host=lens)
    return _native.decode_kernel(torch.bfloat16, q_heads, kv_heads, head_dim, block_size, batch, bound, batch * bound,
                                 device_planned=True)


_FORCED = """
import sys
sys.path.insert(0, sys.argv[1])
import torch
from nano_infer_engine import _native
for arg in sys.argv[2:]:
    q_heads, kv_heads, head_dim, batch, bound = map(int, arg.split(","))
    print(_native.decode_kernel(torch.bfloat16, q_heads, kv_heads, head_dim, 16, batch, bound, batch * bound,
                                device_planned=True))
"""


@pytest.mark.parametrize("forced", [8, 33, 64, 128])
def test_forced_split_length_fits_the_ring(forced):
    """With the split length forced, every table of a device-planned call has
    it: a call whose scores would not fit a wave's region of the ring kernel
    (which then writes no output) takes another kernel."""
    shapes = [(32, 8, 64, 4, 512), (32, 8, 64, 16, 4096), (8, 8, 64, 4, 512), (16, 1, 64, 2, 1024),
              (32, 8, 128, 4, 512), (16, 8, 128, 4, 512), (64, 8, 128, 3, 2048)]
    package = os.path.dirname(os.path.dirname(os.path.abspath(_native.__file__)))
    out = subprocess.run([sys.executable, "-c", _FORCED, package] + [",".join(map(str, s)) for s in shapes],
                         env=dict(os.environ, NIE_DECODE_TILES_PER_SPLIT=str(forced)), capture_output=True, text=True,
                         check=True, timeout=300)
    kernels = out.stdout.split()
    assert len(kernels) == len(shapes)
    for (q_heads, kv_heads, head_dim, *_), kernel in zip(shapes, kernels):
        assert kernel in ("passes", "fused", "ring")
        if kernel == "ring":
            assert forced * (q_heads // kv_heads) <= RING_SCORE_ROWS[head_dim]
