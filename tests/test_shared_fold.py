"""The shared fold: a unit's workgroups each fold a slice of its output.

GPU: split counts that divide the output and that do not, the smallest and
the largest that share, ragged lengths whose last split is short, every
element format, against the fp32 oracle; the counters are zero again after
each launch, and launches that compete for the chip on several streams (whose
workgroups may give up waiting) write the bits of a launch alone.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle.reference import decode_fp16_protocol
from paged_attention_decode_amd import _native, heuristics
from tests.helpers import make_cache, shuffled_table

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}

CASES = [
    # (lengths, kv heads, group, head_dim, page size, q, kv)
    ([8192] * 8, 1, 16, 256, 16, "bf16", "bf16"),
    ([8192, 8191, 4097, 8000, 1, 0, 8177, 8192], 1, 16, 256, 16, "fp16", "fp16"),
    ([4096] * 10, 1, 13, 256, 16, "fp16", "e4m3"),  # 25 splits of 832 elements
    ([16384] * 2, 1, 16, 256, 32, "fp16", "fp16"),  # 64 splits
    ([16384, 9000, 100, 16000, 12345, 16384, 1, 7], 1, 16, 128, 16, "bf16", "e5m2"),
    ([4096, 4000, 17, 4096, 2048, 4095], 2, 16, 256, 1, "fp16", "fp16"),
    ([2000] * 16, 1, 16, 256, 24, "fp16", "fp16"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"b{len(c[0])}-{'-'.join(map(str, c[1:]))}")
def test_shared_fold_against_oracle(case):
    import paged_attention_decode_amd as pad

    lens, hkv, group, d, ps, qt, kvt = case
    bt, num_pages = shuffled_table(lens, ps, spare_pages=2, extra_cols=0, seed=d)
    k, v = make_cache(num_pages, ps, hkv, d, seed=len(lens))
    q = torch.randn(len(lens), hkv * group, d, generator=torch.Generator().manual_seed(ps)).to(DTYPES[qt])
    k, v, sl = k.to(DTYPES[kvt]), v.to(DTYPES[kvt]), torch.tensor(lens, dtype=torch.int32)
    expected = decode_fp16_protocol(q.float(), k.float(), v.float(), bt, sl)
    q, k, v, bt, sl = q.cuda(), k.cuda(), v.cuda(), bt.cuda(), sl.cuda()
    decode = pad.paged_attention_decode_fp8 if kvt in ("e4m3", "e5m2") else pad.paged_attention_decode_ex
    out = decode(q, k, v, bt, sl)
    # bfloat16: P and the output are rounded to 8 bits, as in tests/test_bf16.py
    tol = 2e-3 if qt == "fp16" else 1e-2
    got = out.float().cpu()
    assert torch.isfinite(got).all()
    assert torch.allclose(got, expected, rtol=tol, atol=tol), (got - expected).abs().max().item()
    for _ in range(3):  # the counters are back at zero
        assert torch.equal(out, decode(q, k, v, bt, sl))
    streams = [torch.cuda.Stream() for _ in range(4)]
    torch.cuda.synchronize()
    outs = []
    for _ in range(5):
        for s in streams:
            with torch.cuda.stream(s):
                outs.append(decode(q, k, v, bt, sl))
    torch.cuda.synchronize()
    assert all(torch.equal(out, o) for o in outs)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[i] for i in (0, 1, 3, 5)], ids=lambda c: f"b{len(c[0])}-{'-'.join(map(str, c[1:]))}")
def test_workgroups_that_give_up_leave_the_same_bits(case):
    """In the measurement library with one poll: a unit's early workgroups give up, and its last arrival folds it."""
    import paged_attention_decode_amd as pad

    lens, hkv, group, d, ps, qt, kvt = case
    bt, num_pages = shuffled_table(lens, ps, spare_pages=2, extra_cols=0, seed=d)
    k, v = make_cache(num_pages, ps, hkv, d, seed=len(lens))
    q = torch.randn(len(lens), hkv * group, d, generator=torch.Generator().manual_seed(ps)).to(DTYPES[qt]).cuda()
    k, v, bt = k.to(DTYPES[kvt]).cuda(), v.to(DTYPES[kvt]).cuda(), bt.cuda()
    sl = torch.tensor(lens, dtype=torch.int32).cuda()
    expected = pad.paged_attention_decode_ex(q, k, v, bt, sl)
    lib = _native.timeline()
    out = torch.empty_like(q)
    dm = _native.dims_for(q, k, v, bt, sl, out)
    ws, n = ctypes.c_size_t(), ctypes.c_int64()
    assert lib.pad_decode_workspace_bytes(ctypes.byref(dm), 0, 0, ctypes.byref(ws)) == 0
    assert lib.pad_decode_counters_needed(ctypes.byref(dm), 0, 0, ctypes.byref(n)) == 0
    workspace = torch.empty(ws.value, dtype=torch.uint8, device="cuda")
    counters = torch.zeros(n.value, dtype=torch.int32, device="cuda")
    c = _native.PadCall()
    c.q, c.k_cache, c.v_cache, c.out = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr()
    c.block_table, c.seq_lens = bt.data_ptr(), sl.data_ptr()
    c.workspace, c.workspace_bytes = workspace.data_ptr(), ws.value
    c.counters, c.num_counters = counters.data_ptr(), n.value
    c.scale, c.k_scale, c.v_scale, c.kv_format = d ** -0.5, 1.0, 1.0, 3 if qt == "bf16" else 0
    shape = (_native.TL_LAUNCHES, _native.TL_MAX_GROUPS, _native.TL_SLOTS)
    buf = np.zeros(shape, dtype=np.uint64)

    def run(polls):
        out.zero_()
        assert lib.pad_timeline_reset() == 0 and lib.pad_timeline_set_fold_polls(polls) == 0
        try:
            st = lib.pad_decode_launch_call(ctypes.byref(c), ctypes.byref(dm), torch.cuda.current_stream().cuda_stream)
        finally:
            lib.pad_timeline_set_fold_polls(0)
        assert st == 0
        torch.cuda.synchronize()
        assert torch.equal(out, expected)
        assert int(counters.abs().sum()) == 0
        assert lib.pad_timeline_read(buf.ctypes.data, buf.nbytes) == 0
        rows = buf[0].astype(np.int64)
        flags = rows[:, _native.TL_INFO] >> 40 & 0xFF
        arrived = rows[:, _native.TL_ARRIVED] != 0
        folded = (flags & _native.TL_F_MERGER) != 0
        return int((arrived & folded).sum()), int((arrived & ~folded).sum())

    for _ in range(3):
        folded, gave_up = run(1)
        assert folded > 0 and gave_up > 0, (folded, gave_up)
    folded, gave_up = run(0)
    assert folded > gave_up, (folded, gave_up)


def test_split_counts_of_shared_folds():
    plan = heuristics.plan_units
    assert plan(8, 16, 1, 256, 16, 512).num_splits == 32  # all CUs: 21.0 us against 23.4 us at 16 splits
    assert plan(6, 32, 2, 256, 16, 256).num_splits == 16  # what 16-block splits allow of 21
    assert plan(8, 8, 1, 128, 16, 512).num_splits == 16  # half the CUs: 8192 elements a unit
    assert plan(4, 16, 1, 256, 16, 1024).num_splits == 32  # half the CUs: 64 splits would not share
