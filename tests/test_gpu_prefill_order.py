"""Prefill calls too large for the host's item table whose query tiles are one
piece each: the workgroups take the tiles in the order of the keys they see
(up to 16 requests), in request order otherwise.  Every row is written, with
the result that the request alone gives."""

from __future__ import annotations

import pytest
import torch

from nano_infer_engine import _native, workloads
from tests.test_gpu_kernels import TOL, _prefill_case, rounding  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = {  # contexts, queries
    "equal": ([0] * 4, [560] * 4),
    "ragged": ([0, 40, 7, 0, 300, 0], [1200, 1, 700, 33, 64, 515]),
    "contexts_above": ([3000, 0, 2968, 1500], [31, 2048, 64, 500]),  # equal levels of different requests
    "contexts_near": ([700, 0, 668, 500], [531, 1200, 764, 900]),
    "empty_requests": ([0, 5, 0, 64, 9], [900, 0, 1111, 0, 513]),  # (with cached tokens only)
    "sixteen": ([0] * 16, [130 + 17 * i for i in range(16)]),
    "seventeen": ([0] * 17, [130 + 17 * i for i in range(17)]),
}


@pytest.mark.parametrize("q_heads,kv_heads,head_dim,host_plan,name,order", [
    # 16 query heads per KV head: tiles of 8 tokens
    (64, 4, 64, True, "equal", "sorted"),
    (64, 4, 64, True, "ragged", "sorted"),
    (64, 4, 64, True, "contexts_above", "sorted"),
    (64, 4, 64, True, "empty_requests", "sorted"),
    (64, 4, 64, True, "sixteen", "sorted"),
    (64, 4, 64, True, "seventeen", "requests"),
    # tiles of 40 tokens (a padding row per row block), and of 16 (two)
    (24, 8, 128, True, "contexts_near", "sorted"),
    (24, 8, 128, True, "sixteen", "sorted"),
    (24, 8, 128, True, "equal", "table"),
    (24, 8, 128, True, "ragged", "requests"),  # (tiles of several pieces)
    (28, 4, 128, True, "sixteen", "sorted"),
    # planned from bounds
    (64, 4, 64, False, "sixteen", "sorted"),
    (64, 4, 64, False, "equal", "requests"),
    (128, 8, 64, False, "equal", "sorted"),
    (128, 8, 64, False, "ragged", "sorted"),
    (128, 8, 64, False, "empty_requests", "sorted"),
])
def test_sorted_items(q_heads, kv_heads, head_dim, host_plan, name, order, rounding):  # noqa: F811
    print(f"prefill order {name} {q_heads}/{kv_heads} d={head_dim} host={host_plan}", flush=True)
    contexts, queries = CASES[name]
    assert _native.prefill_order(queries, contexts, q_heads, kv_heads, head_dim, host_plan) == order
    wl = workloads.ragged(contexts, queries, seed=31, pool_factor=1.2, q_heads=q_heads, kv_heads=kv_heads,
                          head_dim=head_dim, block_size=16)
    got, want = _prefill_case(wl, torch.bfloat16, host_plan)
    err = (got.float() - want.float()).abs().max().item()
    print(f"  max_abs_err={err:.3e}", flush=True)
    assert err <= TOL[torch.bfloat16]  # the bf16 bar of the other prefill tests
