"""The one-launch decode of host-planned calls (decode_ring_kernel) against
the pass launches it replaces: outputs and cache writes bit for bit, control
region zero afterwards, at head_dim 64 and 128 and GQA groups up to 16,
around the edges of its tiles, steps, splits and score regions."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from nano_infer_engine import _native, workloads
from tests.test_gpu_decode_fused import (  # noqa: F401
    _control_regions_zero, _decode_oracle, _fused_and_passes, _gave_up_counts, _reference_rounding, _same_bits)

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
KERNEL = "ring"  # what every case but the last runs on

CASES = {  # q_heads, kv_heads, head_dim, block_size, contexts
    # a split of one key, a whole tile, a whole step, one key past each
    "edges64": (32, 8, 64, 16, [0, 15, 16, 31, 32, 47, 64, 700] + [1190] * 14),
    "edges128": (32, 8, 128, 16, [0, 15, 16, 31, 32, 47, 64, 700] + [600] * 12),
    "four_head_group": (16, 4, 64, 32, [i % 97 for i in range(100)]),
    "two_head_group": (4, 2, 128, 16, [1000, 33, 15, 777]),
    "one_head_group": (2, 1, 128, 32, [1000, 33, 15, 777]),
    "group1_dim128": (8, 8, 128, 16, [2000, 15, 640, 100, 1990, 1500, 1200]),
    "group8_dim128": (64, 8, 128, 64, [700, 15, 640, 100] + [650] * 12),
    "group3": (24, 8, 128, 16, [2047, 331, 1200, 77, 905, 1618]),
    "group12": (48, 4, 128, 32, [7 * i % 311 for i in range(100)]),
    "group16": (64, 4, 128, 16, [800 - i for i in range(40)]),  # every query row of the tile
    "many_splits": (32, 8, 64, 16, [7990, 20, 8000, 8000, 8000]),  # 63 splits: two polls, several rounds of the sum
    "longest_splits": (32, 8, 64, 16, [8100] * 16),  # 32 tiles: the scores fill their region
    "past_the_ring": (32, 8, 64, 16, [9000] * 16),  # longer: decode_fused_kernel
}


def _run(name: str, append: str):
    q_heads, kv_heads, head_dim, block_size, contexts = CASES[name]
    wl = workloads.ragged(contexts, [1] * len(contexts), seed=83, pool_factor=1.2, q_heads=q_heads, kv_heads=kv_heads,
                          head_dim=head_dim, block_size=block_size)
    dtype = torch.bfloat16
    kc, vc = wl.pool(dtype)
    q, k_new, v_new = wl.new_tokens(dtype)
    if append != "none":
        # the new rows' slots hold NaN until the call writes them
        for pool in (kc, vc):
            flat = pool.view(-1, kv_heads, head_dim)
            flat[torch.from_numpy(wl.slots())] = float("nan")
    tables = torch.from_numpy(wl.table_array()).to(DEV)
    lens = torch.tensor(wl.seq_lens, dtype=torch.int32, device=DEV)
    rope = None
    if append == "rope":
        from nano_infer_engine.layers.rope import RopeScale

        rope = RopeScale(head_dim).tables(DEV, dtype, max(wl.seq_lens))
    dq = q.to(DEV)
    kernel = _native.decode_kernel(dtype, q_heads, kv_heads, head_dim, block_size, len(contexts), max(wl.seq_lens),
                                   sum(wl.seq_lens), seq_lens_host=list(wl.seq_lens))
    assert kernel == ("fused" if name == "past_the_ring" else KERNEL), kernel

    def run():
        k, v = kc.to(DEV), vc.to(DEV)
        kw = {} if append == "none" else dict(new_kv=(k_new.to(DEV), v_new.to(DEV)), rope_tables=rope)
        out = _native.paged_decode(dq, k, v, 0, tables, lens, max(wl.seq_lens), sum(wl.seq_lens), head_dim**-0.5,
                                   seq_lens_host=list(wl.seq_lens), **kw)
        return out, k, v

    return wl, kc, vc, q, run


def _check(run):
    (o1, k1, v1), (o2, k2, v2), p1, p2 = _fused_and_passes(run)
    assert p1 == "fused" and p2 == "passes", (p1, p2)
    assert not torch.isnan(o1).any()
    assert _same_bits(o1, o2), "one-launch output differs from the pass launches"
    assert _same_bits(k1, k2) and _same_bits(v1, v2), "one-launch cache writes differ from the pass launches"
    assert _control_regions_zero()
    return o1


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("append", ["none", "append", "rope"])
def test_matches_pass_launches(name, append):
    print(f"ring decode: {name} {append}", flush=True)
    wl, kc, vc, q, run = _run(name, append)
    out = _check(run)
    if append == "none":
        err = (out.cpu().float() - _decode_oracle(wl, kc, vc, q).float()).abs().max().item()
        print(f"  max_abs_err={err:.3e}", flush=True)
        assert err <= 2e-2  # the bf16 bar of the other decode tests


@pytest.mark.parametrize("name", ["edges128", "group12", "many_splits"])
@pytest.mark.parametrize("append", ["none", "rope"])
def test_waits_that_give_up(name, append):
    """With a poll limit of 0 every split forms the others' pairs from K."""
    print(f"ring decode, waits give up: {name} {append}", flush=True)
    *_, run = _run(name, append)
    run()  # creates the cached workspace
    torch.cuda.synchronize()
    before = sum(_gave_up_counts())
    _native.set_decode_fused_spin(0)
    _check(run)
    assert sum(_gave_up_counts()) > before


def test_back_to_back_calls():
    """Calls of several shapes in turn on one stream: each finds the records clear."""
    runs = [_run(name, "rope")[-1] for name in ("edges128", "group3", "many_splits", "edges64")]
    single = []
    for run in runs:
        single.append(run()[0])
        torch.cuda.synchronize()
    outs = [runs[i % len(runs)]()[0] for i in range(16)]
    torch.cuda.synchronize()
    for i, out in enumerate(outs):
        assert _same_bits(out, single[i % len(runs)]), i
    assert _control_regions_zero()


@pytest.mark.parametrize("q_heads,kv_heads,head_dim,bound,kernel", [
    (32, 8, 128, 512, "ring"), (16, 8, 128, 1024, "ring"), (24, 8, 128, 512, "ring"), (32, 8, 64, 512, "fused")])
def test_replays_of_a_device_planned_call(q_heads, kv_heads, head_dim, bound, kernel):
    """One captured launch, replayed with tables of even, ragged and skewed
    lengths (and none): each replay equals the eager call planned from the
    host lengths bit for bit, cache included."""
    print(f"device-planned replays: {q_heads}/{kv_heads} x {head_dim}, bound {bound}", flush=True)
    dtype, batch, bs = torch.bfloat16, 4, 16
    assert _native.decode_kernel(dtype, q_heads, kv_heads, head_dim, bs, batch, bound, batch * bound,
                                 device_planned=True) == kernel
    wl = workloads.ragged([bound - 1] * batch, [1] * batch, seed=29, pool_factor=1.2, q_heads=q_heads,
                          kv_heads=kv_heads, head_dim=head_dim, block_size=bs)
    kc, vc = wl.pool(dtype)
    q, k_new, v_new = (t.to(DEV) for t in wl.new_tokens(dtype))
    tables = torch.from_numpy(wl.table_array()).to(DEV)
    lens = torch.zeros(batch, dtype=torch.int32, device=DEV)
    plan = torch.zeros(-(-_native.decode_plan_bytes() // 4), dtype=torch.int32, device=DEV)
    k, v, out = kc.to(DEV), vc.to(DEV), torch.empty_like(q)
    scale = head_dim**-0.5

    def host_plan(host):
        buf = np.zeros(plan.numel(), dtype=np.int32)
        _native.write_decode_plan(buf.ctypes.data, buf.nbytes, dtype, q_heads, kv_heads, head_dim, bs,
                                  np.asarray(host, dtype=np.int32), max(host), sum(host))
        assert buf[0] > 0
        return torch.from_numpy(buf).to(DEV)

    lens.copy_(torch.tensor([bound] * batch, dtype=torch.int32))
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        call = _native.PreparedDecode(k, v, tables, lens, bound, batch * bound, q_heads, scale, device_plan=plan)
        call.append_decode(q, k_new, v_new, 0, out)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            call.append_decode(q, k_new, v_new, 0, out)
    for host, table in [([bound] * batch, True), ([1, 17, 40, bound], True), ([bound - 1, 33, 250, 16], True),
                        ([5, 100, 64, 31], True), ([bound, 3, 200, 77], False), ([1, 2, 1, 1], True)]:
        with torch.cuda.stream(stream):
            k.copy_(kc)
            v.copy_(vc)
            lens.copy_(torch.tensor(host, dtype=torch.int32))
            plan.copy_(host_plan(host)) if table else plan.zero_()
            graph.replay()
            stream.synchronize()
        k2, v2 = kc.to(DEV), vc.to(DEV)
        want = torch.empty_like(q)
        _native.PreparedDecode(k2, v2, tables, lens, max(host), sum(host), q_heads, scale,
                               seq_lens_host=host).append_decode(q, k_new, v_new, 0, want)
        torch.cuda.synchronize()
        if table:
            assert _same_bits(out, want), host
        else:  # (other splits)
            assert (out.float() - want.float()).abs().max().item() <= 2e-2
        assert _same_bits(k, k2) and _same_bits(v, v2), host
    assert _control_regions_zero()
