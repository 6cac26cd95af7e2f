"""Varlen prefill with the reference rounding on scores that other tests do not
draw: maxima that rise late, large common offsets, -inf, +inf and NaN scores,
over one and several pieces of a query tile.  q and K hold small whole
numbers, so that every product of a row pair is exact and the scores, and
their rounding to bf16, are the oracle's; column 0 carries the rest."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from nano_infer_engine import _native, workloads
from oracle import reference_ops
from tests.test_gpu_kernels import TOL

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _column(kind: str, position: np.ndarray, length: int) -> np.ndarray:
    """K[..., 0] by position; q[..., 0] is 2."""
    if kind == "rising":  # by 40 per 64 keys, the maximum near each row's last key
        return np.floor(position / 64) * 160.0
    if kind == "falling":
        return np.floor((length - position) / 64) * 160.0
    if kind == "spikes":  # a new maximum at keys far apart, on one lane each
        return np.where(position % 389 == 388, position // 389 * 400.0 + 400.0, 0.0)
    if kind == "offset":
        return np.full(position.shape, -4096.0)
    if kind == "minus_inf":  # rows 0 and 1 of a fresh prompt see nothing else
        return np.where(position % 3 < 2, -3e38, 0.0)
    if kind == "plus_inf":
        return np.where(position == 100, 3e38, 0.0)
    assert kind == "nan"
    return np.where(position == 100, np.nan, 0.0)


@pytest.mark.parametrize("kind", ["rising", "falling", "spikes", "offset", "minus_inf", "plus_inf", "nan"])
@pytest.mark.parametrize("q_heads,kv_heads,head_dim", [(8, 2, 64), (8, 2, 128), (6, 2, 128)])
@pytest.mark.parametrize("host_plan", [True, False])
def test_scores(kind, q_heads, kv_heads, head_dim, host_plan):
    print(f"prefill scores {kind} {q_heads}/{kv_heads} d={head_dim} host={host_plan}", flush=True)
    contexts, queries = [0, 700, 2000], [130, 65, 40]
    wl = workloads.ragged(contexts, queries, seed=37, pool_factor=1.2, q_heads=q_heads, kv_heads=kv_heads,
                          head_dim=head_dim, block_size=16)
    rng = np.random.default_rng(7)
    kc, vc = wl.pool(torch.bfloat16)
    q, k, v = wl.new_tokens(torch.bfloat16)
    for t in (kc, q, k):
        t.copy_(torch.from_numpy(rng.integers(-1, 2, t.shape)))
    q[..., 0] = 2
    flat, at = kc.view(-1, kv_heads, head_dim), 0
    for table, c, n in zip(wl.tables, contexts, queries):
        column = torch.from_numpy(_column(kind, np.arange(c + n, dtype=np.float64), c + n)).to(kc.dtype)[:, None]
        pos = np.arange(c)
        flat[torch.from_numpy(np.asarray(table)[pos // 16] * 16 + pos % 16), :, 0] = column[:c]
        k[at : at + n, :, 0] = column[c:]
        at += n
    want = reference_ops.ragged_attention_reference(q, k, v, kc, vc, 0, wl.tables, contexts, queries,
                                                    head_dim**-0.5).float()  # (writes k and v into the pools)
    cu = np.concatenate([[0], np.cumsum(queries)]).astype(np.int64)
    host = dict(cu_seqlens_host=cu.tolist(), context_lens_host=contexts) if host_plan else {}
    got = _native.varlen_prefill(q.to(DEV), torch.from_numpy(cu).to(DEV),
                                 torch.tensor(contexts, dtype=torch.int32, device=DEV), kc.to(DEV), vc.to(DEV), 0,
                                 torch.from_numpy(wl.table_array()).to(DEV), max(queries), max(wl.seq_lens),
                                 head_dim**-0.5, **host).float().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    if kind in ("minus_inf", "plus_inf", "nan"):
        assert torch.isnan(want).any() and not torch.isnan(want).all()
    err = (got - want).nan_to_num(0.0).abs().max().item()
    print(f"  max_abs_err={err:.3e}", flush=True)
    assert err <= TOL[torch.bfloat16]  # the bf16 bar of the other prefill tests
