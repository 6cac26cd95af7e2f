"""GQA groups that do not divide an MFMA's 16 rows (3, 5, 6, 7, 12 query heads
per KV head, ...) run on the MFMA kernels at head_dim 64 and 128: decode,
the fused append (+ RoPE), varlen prefill and device-planned decode, both
bf16 rounding points; calls whose alignment or workspace keeps them from those
kernels run on the generic one.  Bars as for the other shapes: fp32 max-abs
<= 1e-4 and bf16 <= 2e-2 against the oracle, fused calls bit-identical to
the separate ones.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from nano_infer_engine import _native, workloads
from tests.test_gpu_kernels import (  # noqa: F401
    TOL, _append_decode_pair, _decode_hip, _decode_oracle, _prefill_case, rounding)

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")

SHAPES = [  # (q_heads, kv_heads, head_dim, block_size)
    (24, 8, 128, 16),  # 3: 5 tokens and one padding row per row block
    (24, 8, 64, 16),   # 3 in the one-launch decode
    (10, 2, 64, 8),    # 5, blocks smaller than a tile
    (12, 2, 128, 32),  # 6
    (14, 2, 64, 16),   # 7
    (12, 1, 128, 12),  # 12: one token per row block, a block size that is no power of two
]


def _err(got, want) -> float:
    err = (got.float() - want.float()).abs().max().item()
    print(f"  max_abs_err={err:.3e}", flush=True)
    return err


@pytest.mark.parametrize("q_heads,kv_heads,head_dim,block_size", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("host_plan", [True, False])
def test_decode_matches_oracle(q_heads, kv_heads, head_dim, block_size, dtype, host_plan, rounding):  # noqa: F811
    print(f"group decode {q_heads}/{kv_heads} d={head_dim} bs={block_size} {dtype} host={host_plan}", flush=True)
    wl = workloads.ragged([0, 14, 15, 16, 300, 1500], [1] * 6, seed=61, pool_factor=1.5, q_heads=q_heads,
                          kv_heads=kv_heads, head_dim=head_dim, block_size=block_size)
    kc, vc = wl.pool(dtype)
    q, _, _ = wl.new_tokens(dtype)
    got = _decode_hip(wl, kc.to(DEV), vc.to(DEV), q, dtype, host_plan=host_plan)
    assert _native.decode_last_path() not in ("none", "generic")
    assert _err(got, _decode_oracle(wl, kc, vc, q)) <= TOL[dtype]


@pytest.mark.parametrize("q_heads,kv_heads,head_dim,block_size", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_decode_append_matches_separate_calls(q_heads, kv_heads, head_dim, block_size, dtype, rounding):  # noqa: F811
    print(f"group decode_append {q_heads}/{kv_heads} d={head_dim} bs={block_size} {dtype}", flush=True)
    wl = workloads.ragged([0, 4, 15, 16, 70, 300], [1] * 6, seed=47, pool_factor=1.5, q_heads=q_heads,
                          kv_heads=kv_heads, head_dim=head_dim, block_size=block_size)
    _append_decode_pair(wl, dtype, True, layer=1, rope=True)


@pytest.mark.parametrize("q_heads,kv_heads,head_dim,block_size", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("host_plan", [True, False])
def test_varlen_prefill_matches_oracle(q_heads, kv_heads, head_dim, block_size, dtype, host_plan, rounding):  # noqa: F811
    print(f"group prefill {q_heads}/{kv_heads} d={head_dim} bs={block_size} {dtype} host={host_plan}", flush=True)
    # one token, tiles that end inside a row block, a tile split over several pieces
    wl = workloads.ragged([0, 3, 700, 0, 17], [19, 1, 45, 130, 40], seed=43, pool_factor=1.5, q_heads=q_heads,
                          kv_heads=kv_heads, head_dim=head_dim, block_size=block_size)
    got, want = _prefill_case(wl, dtype, host_plan)
    assert _err(got, want) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_unaligned_rows_run_on_the_generic_kernel(dtype):
    """Rows at element alignment are accepted as before, and give the same results."""
    wl = workloads.ragged([0, 15, 300], [1] * 3, seed=53, pool_factor=1.5, q_heads=6, kv_heads=2, head_dim=64)
    kc, vc = wl.pool(dtype)
    q, _, _ = wl.new_tokens(dtype)
    flat = torch.empty(q.numel() + 1, dtype=dtype, device=DEV)
    rows = flat[1:].view(q.shape)
    rows.copy_(q)
    tables = torch.from_numpy(wl.table_array()).to(DEV)
    lens = torch.tensor(wl.seq_lens, dtype=torch.int32, device=DEV)
    decode = _native.PreparedDecode(kc.to(DEV), vc.to(DEV), tables, lens, max(wl.seq_lens), sum(wl.seq_lens), 6,
                                    wl.head_dim**-0.5, seq_lens_host=list(wl.seq_lens))
    want = _decode_oracle(wl, kc, vc, q)
    got = torch.empty_like(q, device=DEV)
    decode(rows, 0, got)
    assert _native.decode_last_path() == "generic"
    assert _err(got.cpu(), want) <= TOL[dtype]
    decode(rows.clone(), 0, got)
    assert _native.decode_last_path() != "generic"
    assert _err(got.cpu(), want) <= TOL[dtype]


def _attention_64(q, keys, values, scale, last):
    """q (n, heads, dim), key and value rows of each query head's KV head, in 64 bits."""
    seen = torch.arange(keys.shape[0], device=DEV)[None, :] <= last[:, None]
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    for h in range(q.shape[1]):
        k, v = (t[:, h * keys.shape[1] // q.shape[1]].double().contiguous() for t in (keys, values))
        scores = (q[:, h].double() @ k.t().contiguous()) * scale
        out[:, h] = torch.softmax(scores.masked_fill(~seen, -torch.inf), dim=-1) @ v
    return out


@pytest.mark.parametrize("q_heads,kv_heads,head_dim", [(6, 2, 64), (24, 8, 128), (14, 2, 128), (26, 2, 128)])
@pytest.mark.parametrize("contexts,queries", [([4000, 15, 700, 2000], [1] * 4), ([0, 200, 1500], [300, 128, 77])])
def test_fp32_is_as_exact_as_the_generic_kernel(q_heads, kv_heads, head_dim, contexts, queries):
    """Relative error against 64 bits, of the MFMA kernels and of the generic
    ones (rows at element alignment) on the same numbers, over three draws."""
    print(f"group fp32 error {q_heads}/{kv_heads} d={head_dim} {queries}", flush=True)
    total = {"mfma": 0.0, "generic": 0.0}
    for seed in (3, 4, 5):
        wl = workloads.ragged(contexts, queries, seed=seed, pool_factor=1.2, q_heads=q_heads, kv_heads=kv_heads,
                              head_dim=head_dim)
        kc, vc = (t.to(DEV) for t in wl.pool(torch.float32))
        q = wl.new_tokens(torch.float32)[0].to(DEV)
        tables = torch.from_numpy(wl.table_array()).to(DEV)
        scale, lens = head_dim**-0.5, list(wl.seq_lens)
        want, at = torch.empty(q.shape, dtype=torch.float64, device=DEV), 0
        for b, (n, m) in enumerate(zip(lens, queries)):
            pos = torch.arange(n, device=DEV)
            slots = tables[b][pos // wl.block_size].long() * wl.block_size + pos % wl.block_size
            keys, values = (t[0].reshape(-1, kv_heads, head_dim)[slots] for t in (kc, vc))
            want[at : at + m] = _attention_64(q[at : at + m], keys, values, scale, pos[n - m :])
            at += m
        if max(queries) == 1:
            call = _native.PreparedDecode(kc, vc, tables, torch.tensor(lens, dtype=torch.int32, device=DEV), max(lens),
                                          sum(lens), q_heads, scale, seq_lens_host=lens)
        else:
            cu = np.concatenate([[0], np.cumsum(queries)]).astype(np.int64)
            call = _native.PreparedPrefill(kc, vc, torch.from_numpy(cu).to(DEV),
                                           torch.tensor(contexts, dtype=torch.int32, device=DEV), tables, sum(queries),
                                           max(queries), max(lens), q_heads, scale, cu_seqlens_host=cu.tolist(),
                                           context_lens_host=contexts)
        off = torch.empty(q.numel() + 1, device=DEV)[1:].view(q.shape).copy_(q)  # 4 bytes off 16
        for name, rows in (("mfma", q), ("generic", off)):
            out = torch.empty_like(q)
            call(rows, 0, out)
            total[name] += ((out.double() - want).norm() / want.norm()).item()
    print(f"  {total}", flush=True)
    assert total["mfma"] <= total["generic"]


@pytest.mark.parametrize("q_heads,head_dim", [(6, 64), (6, 128)])
def test_device_planned_decode_equals_host_planned(q_heads, head_dim, rounding):  # noqa: F811
    dtype = torch.bfloat16
    wl = workloads.ragged([0, 15, 700], [1] * 3, seed=59, pool_factor=1.5, q_heads=q_heads, kv_heads=2,
                          head_dim=head_dim)
    kc, vc = (t.to(DEV) for t in wl.pool(dtype))
    q, k, v = (t.to(DEV) for t in wl.new_tokens(dtype))
    bound = 1024
    tables = torch.zeros((3, bound // wl.block_size), dtype=torch.int32, device=DEV)
    arr = torch.from_numpy(wl.table_array()).to(DEV)
    tables[:, : arr.shape[1]] = arr
    lens = torch.tensor(wl.seq_lens, dtype=torch.int32, device=DEV)
    host = np.asarray(wl.seq_lens, dtype=np.int32)
    plan = np.zeros(-(-_native.decode_plan_bytes() // 4), dtype=np.int32)
    _native.write_decode_plan(plan.ctypes.data, plan.nbytes, dtype, q_heads, 2, head_dim, wl.block_size, host,
                              int(host.max()), int(host.sum()))
    assert plan[0] > 0
    planned = _native.PreparedDecode(kc, vc, tables, lens, bound, 3 * bound, q_heads, wl.head_dim**-0.5,
                                     device_plan=torch.from_numpy(plan).to(DEV))
    direct = _native.PreparedDecode(kc, vc, tables, lens, int(host.max()), int(host.sum()), q_heads,
                                    wl.head_dim**-0.5, seq_lens_host=host.tolist())
    a, b = torch.empty_like(q), torch.empty_like(q)
    planned.append_decode(q, k, v, 0, a)
    direct.append_decode(q, k, v, 0, b)
    assert torch.equal(a, b)
