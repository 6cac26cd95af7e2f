"""Which kernels a reference-rounding decode call runs (nie_paged_decode_kernel, the
decision that the call itself takes), checked without a GPU."""

from __future__ import annotations

import os
import random
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


@pytest.mark.parametrize("q_heads,kv_heads,head_dim,lens,kernel", [
    # the shares that one wave of the ring sums, against the sum's launch
    (16, 1, 64, [100] * 7 + [4000], "passes"),  # 125 splits of 16 rows: 54.5 us on the ring, 17.3 here
    (16, 1, 64, [1000] * 4, "passes"),
    (8, 1, 128, [2000] * 4, "passes"),
    (14, 2, 64, [2000] * 4, "passes"),
    (64, 8, 128, [1000] * 4, "passes"),  # 32 splits of 2 tiles, 8 rows
    (64, 8, 128, [1000] * 16, "ring"),  # 8 splits of 8 tiles
    (32, 8, 128, [100] * 15 + [3000], "passes"),  # 63 splits of 3 tiles
    (32, 8, 128, [1000] * 8 + [3000], "ring"),  # 32 splits of 6 tiles
    (32, 8, 128, [30000], "passes"),
    (24, 8, 128, [2047, 331, 1200, 77, 905, 1618], "ring"),
    # against decode_fused_kernel's sum
    (32, 8, 64, [1000] * 4, "fused"),  # 32 splits of 2 tiles
    (32, 8, 64, [100] * 15 + [2000], "fused"),
    (32, 8, 64, [2000] * 16, "ring"),  # 16 splits of 8 tiles
    (32, 8, 64, [1000] * 8 + [3000], "fused"),  # 63 splits of 3 tiles
    (32, 8, 64, [90] * 33, "ring"),  # 3 splits of 2 tiles
    (32, 32, 64, [2000], "fused"),
    (32, 32, 64, [600] * 16, "ring"),
    (8, 8, 64, [3000] * 8, "fused"),  # 32 splits of 6 tiles
    # a sequence's splits in one workgroup
    (32, 8, 64, [17, 64, 129, 500], "short"),
    (32, 8, 64, [17, 64, 129, 513], "fused"),
    (32, 8, 64, [60] * 32, "short"),
    (32, 8, 64, [60] * 33, "ring"),  # more (sequence, KV head) pairs than CUs
])
def test_kernel_of_host_planned_calls(q_heads, kv_heads, head_dim, lens, kernel):
    assert _kernel(q_heads, kv_heads, head_dim, lens) == kernel


def test_shapes_outside_the_one_launch_kernels():
    assert _kernel(32, 8, 64, [500] * 4, block_size=8) == "passes"  # tiles over several blocks
    assert _kernel(32, 1, 64, [500] * 4) == "none"  # 32 rows: the generic kernel
    assert _kernel(8, 8, 32, [500] * 4) == "none"
    assert _native.decode_kernel(torch.float32, 32, 8, 64, 16, 4, 500, 2000, seq_lens_host=[500] * 4) == "none"


@pytest.mark.parametrize("q_heads,kv_heads,head_dim,batch,bound,kernel", [
    (32, 8, 64, 4, 512, "fused"),  # a captured step of short sequences
    (32, 8, 64, 16, 2048, "fused"),  # any of 2,000 tokens each, and one of them among short ones
    (32, 8, 64, 16, 11776, "fused"),
    (16, 1, 64, 8, 1024, "passes"),
    (64, 8, 128, 8, 2048, "passes"),
    (32, 8, 128, 16, 3072, "passes"),
    (32, 8, 128, 43, 1024, "passes"),  # tables of 215 items in two rounds of 128
    (32, 8, 128, 4, 512, "ring"),
    (16, 8, 128, 4, 1024, "ring"),
])
def test_kernel_of_device_planned_calls(q_heads, kv_heads, head_dim, batch, bound, kernel):
    assert _kernel(q_heads, kv_heads, head_dim, batch=batch, bound=bound) == kernel


@pytest.mark.parametrize("q_heads,kv_heads,head_dim", [(32, 8, 128), (16, 8, 128), (8, 8, 128), (32, 32, 128), (4, 2, 128),
                                                       (24, 8, 128), (64, 8, 128), (32, 8, 64), (32, 32, 64), (40, 5, 64)])
def test_device_planned_ring_holds_for_every_table(q_heads, kv_heads, head_dim):
    """A device-planned call on the ring: whatever lengths within its bounds
    the table is written for, the host-planned call of these lengths runs on
    the ring or in one workgroup per sequence and head, too."""
    rng = random.Random(5)
    rings = 0
    for _ in range(300):
        batch, bound = rng.choice([1, 2, 3, 4, 6, 8, 12, 16, 24, 40, 43, 64, 100]), rng.choice([64, 128, 192, 256, 512, 1024, 1536])
        if _kernel(q_heads, kv_heads, head_dim, batch=batch, bound=bound) != "ring":
            continue
        rings += 1
        low = rng.choice([1, bound // 2, bound - 20])
        lens = [rng.randint(low, bound) if rng.random() < rng.choice([0.1, 0.9]) else rng.randint(1, 32)
                for _ in range(batch)]
        lens[0] = rng.choice([bound, lens[0]])
        if not _native.decode_plan_fits(torch.bfloat16, q_heads, kv_heads, head_dim, 16, lens):
            continue  # (no table: planned on the device)
        assert _kernel(q_heads, kv_heads, head_dim, lens) in ("ring", "short"), (batch, bound, lens)
    assert rings or q_heads // kv_heads > 4
