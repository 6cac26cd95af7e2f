"""The decode of short host-planned calls in one workgroup per (sequence, KV
head) (decode_short_kernel) against the pass launches it replaces: outputs
and cache writes bit for bit around the edges of its tiles and splits."""

from __future__ import annotations

import pytest
import torch

from nano_infer_engine import _native
from tests import test_gpu_decode_ring as ring
from tests.test_gpu_decode_fused import _decode_oracle, _gave_up_counts, _reference_rounding  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = {  # q_heads, kv_heads, head_dim, block_size, contexts
    # a split of one key, a whole tile, a whole step, one key past each, 16 splits
    "edges64": (32, 8, 64, 16, [0, 14, 15, 16, 30, 31, 32, 33, 63, 64, 480, 511]),
    "edges128": (32, 8, 128, 16, [0, 14, 15, 16, 30, 31, 32, 33, 63, 64, 480, 511]),
    "one_token": (32, 8, 64, 16, [0]),
    "one_split": (8, 8, 128, 32, [31, 7]),  # no sum over splits
    "group16": (16, 1, 64, 64, [511, 257, 3]),  # every query row of the tile
    "group16_dim128": (16, 1, 128, 16, [400, 5]),
    "group3": (24, 8, 128, 16, [330, 77]),
    "group7": (14, 2, 64, 32, [500, 128, 129]),
    "many_rows": (12, 2, 128, 16, [i % 40 for i in range(120)]),
}


@pytest.fixture(autouse=True)
def _cases(monkeypatch):
    monkeypatch.setattr(ring, "CASES", CASES)
    monkeypatch.setattr(ring, "KERNEL", "short")


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("append", ["none", "append", "rope"])
def test_matches_pass_launches(name, append):
    print(f"short decode: {name} {append}", flush=True)
    wl, kc, vc, q, run = ring._run(name, append)
    run()  # creates the cached workspace
    torch.cuda.synchronize()
    before = sum(_gave_up_counts())
    _native.set_decode_fused_spin(0)  # nothing of the call waits (the imported fixture puts it back)
    out = ring._check(run)
    assert sum(_gave_up_counts()) == before
    if append == "none":
        err = (out.cpu().float() - _decode_oracle(wl, kc, vc, q).float()).abs().max().item()
        print(f"  max_abs_err={err:.3e}", flush=True)
        assert err <= 2e-2  # the bf16 bar of the other decode tests
