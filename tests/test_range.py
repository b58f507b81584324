"""The range kernel (csrc/pa_range.hip): equal page ranges, head groups.

GPU: every element format, page-size mode, head_dim and head-group size that
a launch takes to it, at the edges of its ranges (ragged lengths with empty
sequences at both ends, one-token sequences, lengths around page and block
ends; equal lengths cut alike, in whole units per workgroup, and in whole
units with batches past one register of the table), through the dense table,
the CSR index and a work list, against the fp32 oracle (bfloat16 and fp8 with
bfloat16 q at the bfloat16 tolerance).  A launch with the per-unit kernel's
scratch runs that kernel.

CPU: which shapes take it, and that its scratch is in the plan's.
"""

from __future__ import annotations

import ctypes
import random

import pytest
import torch

from oracle.reference import decode_fp16_protocol
from paged_attention_decode_amd import _native, heuristics
from tests.helpers import make_cache, shuffled_table

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}


def _lens(kind, batch, cap, ps, seed):
    rng = random.Random(seed)
    if kind == "equal":
        return [cap] * batch
    if kind == "equal_pages":  # the same page count, last pages partly filled
        return [cap - rng.randint(0, ps - 1) for _ in range(batch)]
    lens = [rng.choice([rng.randint(1, cap), rng.randint(1, min(cap, 40)), cap]) for _ in range(batch)]
    lens[0] = lens[-1] = lens[batch // 2] = lens[batch // 2 + 1] = 0
    lens[1], lens[2], lens[3] = 1, cap, min(cap, 17)
    return lens


CASES = [
    # (lengths, batch, kv heads, group, head_dim, page size, table tokens, q, kv)
    ("ragged", 40, 4, 4, 128, 16, 2048, "fp16", "fp16"),
    ("ragged", 40, 4, 3, 128, 32, 2048, "bf16", "bf16"),
    ("ragged", 70, 8, 2, 128, 1, 1024, "bf16", "bf16"),
    ("ragged", 40, 4, 4, 128, 2, 2048, "fp16", "fp16"),
    ("ragged", 40, 4, 4, 128, 4, 2048, "fp16", "e5m2"),
    ("ragged", 40, 4, 4, 128, 8, 2048, "bf16", "e4m3"),
    ("ragged", 40, 4, 4, 128, 12, 2048, "fp16", "e4m3"),
    ("ragged", 40, 8, 1, 128, 3, 1000, "fp16", "fp16"),
    ("ragged", 40, 8, 4, 64, 16, 2048, "fp16", "fp16"),
    ("ragged", 40, 8, 16, 64, 24, 2048, "bf16", "e5m2"),
    ("ragged", 40, 8, 3, 96, 16, 1500, "fp16", "fp16"),
    ("ragged", 70, 4, 4, 32, 16, 4096, "bf16", "bf16"),
    ("ragged", 33, 4, 16, 256, 16, 1024, "bf16", "bf16"),
    ("ragged", 33, 4, 2, 256, 5, 1024, "fp16", "e4m3"),
    ("ragged", 70, 6, 2, 128, 16, 2048, "fp16", "fp16"),  # two kv heads per workgroup
    ("ragged", 300, 1, 8, 128, 16, 4096, "fp16", "fp16"),  # past the per-unit planner's batch
    ("ragged", 512, 1, 2, 128, 64, 3200, "fp16", "fp16"),
    ("ragged", 140, 1, 16, 256, 1, 2048, "fp16", "fp16"),
    ("equal", 40, 8, 4, 128, 16, 1040, "fp16", "fp16"),
    ("equal_pages", 33, 4, 8, 128, 16, 2048, "bf16", "e4m3"),
    ("equal", 140, 8, 1, 64, 16, 2048, "fp16", "fp16"),  # 280 head groups: two whole units per workgroup
    ("equal_pages", 260, 4, 1, 32, 8, 3072, "fp16", "fp16"),
]


def _inputs(case):
    kind, batch, hkv, group, d, ps, room, qt, kvt = case
    lens = _lens(kind, batch, room, ps, seed=batch + d)
    width = -(-room // ps)
    used = max(-(-n // ps) for n in lens)
    bt, num_pages = shuffled_table(lens, ps, spare_pages=2, extra_cols=width - used, seed=d)
    k, v = make_cache(num_pages, ps, hkv, d, seed=batch)
    q = torch.randn(batch, hkv * group, d, generator=torch.Generator().manual_seed(ps)).to(DTYPES[qt])
    k, v = k.to(DTYPES[kvt]), v.to(DTYPES[kvt])
    return lens, q, k, v, bt, torch.tensor(lens, dtype=torch.int32)


def _check(out, expected, qt):
    # bfloat16: P and the output are rounded to 8 bits, as in tests/test_bf16.py
    tol = 2e-3 if qt == "fp16" else 1e-2
    got = out.float().cpu()
    assert torch.isfinite(got).all()
    assert torch.allclose(got, expected, rtol=tol, atol=tol), (got - expected).abs().max().item()


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_range_kernel_against_oracle(case):
    import paged_attention_decode_amd as pad

    kind, batch, hkv, group, d, ps, room, qt, kvt = case
    lens, q, k, v, bt, sl = _inputs(case)
    hq = hkv * group
    assert heuristics.range_launch(batch, hq, hkv, d, ps, bt.shape[1]) is not None
    expected = decode_fp16_protocol(q.float(), k.float(), v.float(), bt, sl)
    qd, kd, vd, btd, sld = q.cuda(), k.cuda(), v.cuda(), bt.cuda(), sl.cuda()
    fp8 = kvt in ("e4m3", "e5m2")
    dense = pad.paged_attention_decode_fp8 if fp8 else pad.paged_attention_decode_ex
    out = dense(qd, kd, vd, btd, sld)
    _check(out, expected, qt)
    assert torch.equal(out, dense(qd, kd, vd, btd, sld))  # the same bits again
    w = pad.BatchDecodeWrapper()
    types = dict(q_data_type=DTYPES[qt], kv_data_type=DTYPES[kvt])
    w.plan_block_table(btd, sld, hq, hkv, d, ps, **types)
    assert torch.equal(out, w.run(qd, (kd, vd)))
    indptr, indices, last = pad.paged_kv_indices(btd, sld, ps)
    csr = pad.paged_attention_decode_csr(qd, kd, vd, indptr, indices, last)
    _check(csr, expected, qt)
    w.plan(indptr, indices, last, hq, hkv, d, ps, **types)
    assert torch.equal(csr, w.run(qd, (kd, vd)))


@pytest.mark.gpu
def test_least_scratch_runs_the_per_unit_kernel():
    lib = _native.capi()
    case = CASES[0]
    lens, q, k, v, bt, sl = _inputs(case)
    expected = decode_fp16_protocol(q.float(), k.float(), v.float(), bt, sl)
    qd, kd, vd, btd, sld = q.cuda(), k.cuda(), v.cuda(), bt.cuda(), sl.cuda()
    out = torch.empty_like(qd)
    dm = _native.dims_for(qd, kd, vd, btd, sld, out)
    full, least, n, least_n = ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_int64(), ctypes.c_int64()
    assert lib.pad_decode_workspace_bytes(ctypes.byref(dm), 0, 0, ctypes.byref(full)) == 0
    assert lib.pad_decode_counters_needed(ctypes.byref(dm), 0, 0, ctypes.byref(n)) == 0
    assert lib.pad_decode_least_scratch(ctypes.byref(dm), 0, 0, 0, ctypes.byref(least), ctypes.byref(least_n)) == 0
    assert least.value <= full.value and least_n.value <= n.value
    counters = torch.zeros(n.value, dtype=torch.int32, device="cuda")
    ws = torch.empty(full.value, dtype=torch.uint8, device="cuda")
    for nbytes in (full.value, least.value):
        out.zero_()
        st = lib.pad_decode_launch(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), btd.data_ptr(), sld.data_ptr(),
                                   out.data_ptr(), ws.data_ptr(), nbytes, counters.data_ptr(), n.value,
                                   ctypes.byref(dm), ctypes.c_float(128 ** -0.5), 0,
                                   torch.cuda.current_stream().cuda_stream)
        assert st == 0
        torch.cuda.synchronize()
        _check(out, expected, "fp16")
        assert int(counters.abs().sum()) == 0


# fp8 calls whose own grid has fewer workgroups than the range launch.
SHORT_LISTS = [(129, 1, 8, 128, 16, 4096), (12, 8, 4, 128, 16, 4096)]  # batch, kv heads, group, head_dim, page size, table


def _fp8_records(batch, hkv, group, d, ps, room):
    return heuristics.plan_units(batch, hkv * group, hkv, d, ps, room // ps, kv_bytes=1).num_splits * batch * hkv


@pytest.mark.parametrize("shape", SHORT_LISTS)
def test_fp8_grids_smaller_than_the_range_launch(shape):
    batch, hkv, group, d, ps, room = shape
    groups, _, _ = heuristics.range_launch(batch, hkv * group, hkv, d, ps, room // ps, kv_bytes=1)
    assert _fp8_records(*shape) < groups


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHORT_LISTS)
def test_worklist_of_the_fp8_grids_size_is_not_overrun(shape):
    """A list with room for the per-unit grid only is planned and run per unit; a shorter one is refused."""
    batch, hkv, group, d, ps, room = shape
    lib = _native.capi()
    lens, q, k, v, bt, sl = _inputs(("ragged", batch, hkv, group, d, ps, room, "fp16", "e4m3"))
    expected = decode_fp16_protocol(q.float(), k.float(), v.float(), bt, sl)
    q, k, v, bt, sl = q.cuda(), k.cuda(), v.cuda(), bt.cuda(), sl.cuda()
    out = torch.empty_like(q)
    dm = _native.dims_for(q, k, v, bt, sl, out)
    ws, n = ctypes.c_size_t(), ctypes.c_int64()
    assert lib.pad_decode_workspace_bytes(ctypes.byref(dm), 0, 0, ctypes.byref(ws)) == 0
    assert lib.pad_decode_counters_needed(ctypes.byref(dm), 0, 0, ctypes.byref(n)) == 0
    workspace = torch.empty(ws.value, dtype=torch.uint8, device="cuda")
    counters = torch.zeros(n.value, dtype=torch.int32, device="cuda")
    full, least = ctypes.c_size_t(), 128 * (1 + _fp8_records(*shape))
    assert lib.pad_decode_worklist_bytes(ctypes.byref(dm), 0, 0, 0, ctypes.byref(full)) == 0
    assert least < full.value
    worklist = torch.empty(full.value, dtype=torch.uint8, device="cuda")
    c = _native.PadCall()
    c.q, c.k_cache, c.v_cache, c.out = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr()
    c.block_table, c.seq_lens = bt.data_ptr(), sl.data_ptr()
    c.workspace, c.workspace_bytes = workspace.data_ptr(), ws.value
    c.counters, c.num_counters = counters.data_ptr(), n.value
    c.scale, c.kv_format, c.k_scale, c.v_scale = d ** -0.5, 1, 1.0, 1.0
    c.worklist = worklist.data_ptr()
    stream = torch.cuda.current_stream().cuda_stream

    def plan(nbytes):
        return lib.pad_decode_plan_worklist_call(ctypes.byref(c), ctypes.byref(dm), worklist.data_ptr(), nbytes, stream)

    for nbytes in (least, least + 128, full.value):
        worklist.fill_(0x5A)
        out.zero_()
        assert plan(nbytes) == 0
        c.worklist_bytes = nbytes
        assert lib.pad_decode_launch_call(ctypes.byref(c), ctypes.byref(dm), stream) == 0
        torch.cuda.synchronize()
        assert bool((worklist[nbytes:] == 0x5A).all())
        _check(out, expected, "fp16")
        assert int(counters.abs().sum()) == 0
    c.worklist_bytes = least - 1
    assert plan(least - 1) == 7  # PAD_ERR_WORKSPACE
    assert lib.pad_decode_launch_call(ctypes.byref(c), ctypes.byref(dm), stream) == 7


@pytest.mark.gpu
def test_noalloc_runs_per_unit_where_the_range_scratch_does_not_fit():
    """65790 units: the range launch would count past the static counters, the per-unit kernel needs none."""
    batch, heads, d, ps, width = 510, 129, 32, 16, 768
    lib = _native.capi()
    p = heuristics.plan(batch, heads, heads, d, ps, width)
    assert p.counters > 65536 and heuristics.plan_units(batch, heads, heads, d, ps, width).single_pass
    rng = random.Random(5)
    lens = [rng.choice([0, 1, 15, 16, 17, 40]) for _ in range(batch)]
    bt, num_pages = shuffled_table([16 * 8], ps, spare_pages=0, extra_cols=width - 8, seed=1)
    bt = bt.expand(batch, width).contiguous()
    k, v = make_cache(num_pages, ps, heads, d, seed=2)
    q = torch.randn(batch, heads, d, generator=torch.Generator().manual_seed(3)).half()
    k, v, sl = k.half(), v.half(), torch.tensor(lens, dtype=torch.int32)
    expected = decode_fp16_protocol(q.float(), k.float(), v.float(), bt, sl)
    q, k, v, bt, sl = q.cuda(), k.cuda(), v.cuda(), bt.cuda(), sl.cuda()
    out = torch.full_like(q, float("nan"))
    dm = _native.dims_for(q, k, v, bt, sl, out)
    assert lib.pad_decode_launch_noalloc(q.data_ptr(), k.data_ptr(), v.data_ptr(), bt.data_ptr(), sl.data_ptr(),
                                         out.data_ptr(), ctypes.byref(dm), ctypes.c_float(d ** -0.5), 0,
                                         torch.cuda.current_stream().cuda_stream) == 0
    _check(out, expected, "fp16")


@pytest.mark.gpu
@pytest.mark.parametrize("ps", [16, 12, 1])
def test_lengths_far_past_the_table_are_clipped_to_it(ps):
    """Lengths up to 2^31 - 1 name every page of their row, in the range kernel and in the per-unit kernel."""
    import paged_attention_decode_amd as pad

    batch, hkv, group, d, room = 40, 4, 4, 128, 2048
    lens, q, k, v, bt, _ = _inputs(("ragged", batch, hkv, group, d, ps, room, "fp16", "fp16"))
    cap = bt.shape[1] * ps
    given = list(lens)
    for b, n in ((2, 2**31 - 1), (5, 2**31 - ps), (9, 2**31 - ps - 1), (30, cap + 1)):
        lens[b], given[b] = cap, n
    expected = decode_fp16_protocol(q.float(), k.float(), v.float(), bt, torch.tensor(lens, dtype=torch.int32))
    q, k, v, bt, sl = q.cuda(), k.cuda(), v.cuda(), bt.cuda(), torch.tensor(given, dtype=torch.int32).cuda()
    assert heuristics.range_launch(batch, hkv * group, hkv, d, ps, bt.shape[1]) is not None
    for splits in (None, 3):  # 3: the per-unit kernel
        _check(pad.paged_attention_decode_ex(q, k, v, bt, sl, num_splits=splits), expected, "fp16")


# Equal lengths whose units do not divide the grid: cut alike, or in whole units, up to half of it would be idle.
EQUAL_SHAPES = [(65, 8, 1024), (72, 8, 1024), (129, 8, 768), (140, 8, 768), (257, 1, 3072), (64, 8, 1024), (33, 8, 1024),
                (200, 4, 1024)]  # batch, kv heads, tokens; the last three are cut alike


@pytest.mark.gpu
@pytest.mark.parametrize("shape", EQUAL_SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_equal_lengths_keep_the_grid_busy(shape):
    """Read from the work list: no range is more than 1.6 times as long as an equal share of the positions."""
    import paged_attention_decode_amd as pad

    batch, hkv, tokens = shape
    group, d, ps = 2, 128, 16
    pages = tokens // ps
    groups, heads, _ = heuristics.range_launch(batch, hkv * group, hkv, d, ps, pages)
    lens, q, k, v, bt, sl = _inputs(("equal", batch, hkv, group, d, ps, tokens, "fp16", "fp16"))
    expected = decode_fp16_protocol(q.float(), k.float(), v.float(), bt, sl)
    q, k, v, bt, sl = q.cuda(), k.cuda(), v.cuda(), bt.cuda(), sl.cuda()
    w = pad.BatchDecodeWrapper()
    w.plan_block_table(bt, sl, hkv * group, hkv, d, ps)
    records = w._plan[2].view(torch.int32)[32:32 + 32 * groups].view(groups, 32).cpu()
    T, P = int(records[0, 11]), int(records[0, 12])
    units = batch * hkv // heads
    extra = -(-160 * 1024 // (ps * d * 4 * heads))  # positions of a unit beyond its pages
    assert int((records[:, 8] != 0).sum()) == -(-P // T) <= groups
    assert 5 * T <= 8 * -(-units * (pages + extra) // groups)
    _check(w.run(q, (k, v)), expected, "fp16")
    _check(pad.paged_attention_decode(q, k, v, bt, sl), expected, "fp16")


def _widest(lens, hkv, heads, groups, d, ps, kv_bytes=2):
    """Ranges that the longest sequence's first head group spans, in a call of unequal lengths (pa_range.hip's plan)."""
    page_bytes = ps * d * kv_bytes * 2 * heads
    extra, least = -(-160 * 1024 // page_bytes), -(-192 * 1024 // page_bytes)
    pages = [-(-n // ps) for n in lens]
    assert len({p for p in pages if p}) > 1
    size = [(p + extra) * (hkv // heads) if p else 0 for p in pages]
    T = max(-(-sum(size) // groups), least)
    b = max(range(len(lens)), key=lambda i: pages[i])
    first = sum(size[:b]) + extra
    return (first + pages[b] - 1) // T - first // T + 1


# One long sequence among empty and one-token ones: its ranges merge in two levels (more than 48), the last of the first
# level's groups of 16 not full.
SKEWED = [
    # (batch, kv heads, group, head_dim, page size, q, kv)
    (65, 1, 8, 128, 16, "fp16", "fp16"),
    (33, 8, 4, 128, 16, "bf16", "bf16"),  # four kv heads per workgroup
    (65, 6, 2, 128, 1, "fp16", "fp16"),  # two
    (33, 4, 16, 256, 16, "bf16", "bf16"),  # a thread folds several elements
    (33, 8, 4, 128, 16, "bf16", "e4m3"),
]


def _skewed(case):
    batch, hkv, group, d, ps, qt, kvt = case
    lens = [(0, 1, 1)[b % 3] for b in range(batch)]
    lens[batch // 3] = 32768
    bt, num_pages = shuffled_table(lens, ps, spare_pages=1, extra_cols=0, seed=d)
    k, v = make_cache(num_pages, ps, hkv, d, seed=batch)
    q = torch.randn(batch, hkv * group, d, generator=torch.Generator().manual_seed(ps)).to(DTYPES[qt])
    return lens, q, k.to(DTYPES[kvt]), v.to(DTYPES[kvt]), bt, torch.tensor(lens, dtype=torch.int32)


@pytest.mark.parametrize("case", SKEWED, ids=lambda c: "-".join(map(str, c)))
def test_skewed_calls_merge_in_two_levels(case):
    batch, hkv, group, d, ps, _, kvt = case
    lens = [(0, 1, 1)[b % 3] for b in range(batch)]
    lens[batch // 3] = 32768
    es = 1 if kvt == "e4m3" else 2
    groups, heads, _ = heuristics.range_launch(batch, hkv * group, hkv, d, ps, 32768 // ps, kv_bytes=es)
    n = _widest(lens, hkv, heads, groups, d, ps, es)
    assert n > heuristics.TWO_LEVEL_SPLITS and n % 16


@pytest.mark.gpu
@pytest.mark.parametrize("case", SKEWED, ids=lambda c: "-".join(map(str, c)))
def test_two_level_fold_against_oracle(case):
    import paged_attention_decode_amd as pad

    batch, hkv, group, d, ps, qt, kvt = case
    lens, q, k, v, bt, sl = _skewed(case)
    expected = decode_fp16_protocol(q.float(), k.float(), v.float(), bt, sl)
    q, k, v, bt, sl = q.cuda(), k.cuda(), v.cuda(), bt.cuda(), sl.cuda()
    call = pad.paged_attention_decode_fp8 if kvt == "e4m3" else pad.paged_attention_decode_ex
    out = call(q, k, v, bt, sl)
    _check(out, expected, qt)
    for _ in range(3):  # the group and unit counters are back at zero
        assert torch.equal(out, call(q, k, v, bt, sl))
    w = pad.BatchDecodeWrapper()
    types = dict(q_data_type=DTYPES[qt], kv_data_type=DTYPES[kvt])
    w.plan_block_table(bt, sl, hkv * group, hkv, d, ps, **types)
    assert torch.equal(out, w.run(q, (k, v)))
    indptr, indices, last = pad.paged_kv_indices(bt, sl, ps)
    csr = pad.paged_attention_decode_csr(q, k, v, indptr, indices, last)
    _check(csr, expected, qt)
    w.plan(indptr, indices, last, hkv * group, hkv, d, ps, **types)
    assert torch.equal(csr, w.run(q, (k, v)))
    # With counters of its own: zero afterwards.
    lib = _native.capi()
    dm = _native.dims_for(q, k, v, bt, sl, out)
    ws, n = ctypes.c_size_t(), ctypes.c_int64()
    assert lib.pad_decode_workspace_bytes(ctypes.byref(dm), 0, 0, ctypes.byref(ws)) == 0
    assert lib.pad_decode_counters_needed(ctypes.byref(dm), 0, 0, ctypes.byref(n)) == 0
    workspace = torch.empty(ws.value, dtype=torch.uint8, device="cuda")
    counters = torch.zeros(n.value, dtype=torch.int32, device="cuda")
    again = torch.empty_like(out)
    c = _native.PadCall()
    c.q, c.k_cache, c.v_cache, c.out = q.data_ptr(), k.data_ptr(), v.data_ptr(), again.data_ptr()
    c.block_table, c.seq_lens = bt.data_ptr(), sl.data_ptr()
    c.workspace, c.workspace_bytes = workspace.data_ptr(), ws.value
    c.counters, c.num_counters = counters.data_ptr(), n.value
    c.scale, c.k_scale, c.v_scale = d ** -0.5, 1.0, 1.0
    c.kv_format = {("fp16", "fp16"): 0, ("bf16", "bf16"): 3, ("bf16", "e4m3"): 4}[qt, kvt]
    assert lib.pad_decode_launch_call(ctypes.byref(c), ctypes.byref(dm), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    assert int(counters.abs().sum()) == 0


# What the per-unit kernel is tested on, in shapes that take the range kernel: one of each way to address a block.
FORMS = [("ragged", 40, 4, 4, 128, 16, 2048, "fp16", "fp16"), ("ragged", 40, 4, 4, 128, 12, 2048, "bf16", "bf16"),
         ("ragged", 40, 4, 4, 128, 4, 2048, "fp16", "e4m3"), ("ragged", 33, 4, 2, 256, 32, 1024, "bf16", "e4m3"),
         ("ragged", 70, 8, 2, 128, 1, 1024, "bf16", "e5m2"), ("ragged", 70, 6, 2, 96, 16, 2800, "fp16", "fp16")]


def _decode(kvt):
    import paged_attention_decode_amd as pad

    return pad.paged_attention_decode_fp8 if kvt in ("e4m3", "e5m2") else pad.paged_attention_decode_ex


def _bits(x):
    return x.view(torch.uint8) if x.dtype.itemsize == 1 else x


@pytest.mark.gpu
@pytest.mark.parametrize("case", FORMS, ids=lambda c: "-".join(map(str, c)))
def test_strided_views(case):
    """q, out and both caches as slices of wider tensors, K unlike V, a table and lengths with strides of their own."""
    kind, batch, hkv, group, d, ps, room, qt, kvt = case
    lens, q, k, v, bt, sl = _inputs(case)
    assert heuristics.range_launch(batch, hkv * group, hkv, d, ps, bt.shape[1]) is not None
    expected = decode_fp16_protocol(q.float(), k.float(), v.float(), bt, sl)
    dense = _decode(kvt)(q.cuda(), k.cuda(), v.cuda(), bt.cuda(), sl.cuda())
    qw = torch.zeros(batch, hkv * group, d + 128, dtype=q.dtype, device="cuda")
    qw[:, :, 64:64 + d] = q.cuda()
    n = k.shape[0]
    kw = torch.zeros(n, ps, hkv + 1, d + 8, dtype=k.dtype, device="cuda")
    _bits(kw)[:, :, :hkv, :d] = _bits(k).cuda()
    vw = torch.zeros(n, hkv, ps, d + 16, dtype=v.dtype, device="cuda")  # head-major pages
    _bits(vw)[..., :d] = _bits(v).cuda().transpose(1, 2)
    btw = torch.full((batch, 2 * bt.shape[1] + 1), -1, dtype=torch.int32, device="cuda")
    btw[:, :2 * bt.shape[1]:2] = bt.cuda()
    slw = torch.full((2 * batch,), 1 << 30, dtype=torch.int32, device="cuda")
    slw[::2] = sl.cuda()
    out = _decode(kvt)(qw[:, :, 64:64 + d], kw[:, :, :hkv, :d], vw[..., :d].transpose(1, 2),
                       btw[:, :2 * bt.shape[1]:2], slw[::2])
    _check(out, expected, qt)
    assert torch.equal(out, dense)


@pytest.mark.gpu
@pytest.mark.parametrize("case", FORMS, ids=lambda c: "-".join(map(str, c)))
def test_nan_in_slots_without_a_token(case):
    kind, batch, hkv, group, d, ps, room, qt, kvt = case
    lens, q, k, v, bt, sl = _inputs(case)
    expected = _decode(kvt)(q.cuda(), k.cuda(), v.cuda(), bt.cuda(), sl.cuda())
    used = torch.zeros(k.shape[0], ps, dtype=torch.bool)
    for b, n in enumerate(lens):
        for p in range(-(-n // ps)):
            used[int(bt[b, p]), :n - p * ps] = True
    bad = 0x7F if kvt == "e4m3" else 0x7E if kvt == "e5m2" else float("nan")
    for x in (k, v):
        _bits(x)[~used] = bad
    assert not bool(used.all()) and not bool(torch.isfinite(k.float()).all())
    assert torch.equal(_decode(kvt)(q.cuda(), k.cuda(), v.cuda(), bt.cuda(), sl.cuda()), expected)


@pytest.mark.gpu
@pytest.mark.parametrize("case", FORMS[:5], ids=lambda c: "-".join(map(str, c)))
def test_page_ids_outside_the_cache_read_page_zero(case):
    kind, batch, hkv, group, d, ps, room, qt, kvt = case
    lens, q, k, v, bt, sl = _inputs(case)
    wild, zero = bt.clone(), bt.clone()
    for i, bad in enumerate((-1, k.shape[0], 2**31 - 1, -2**31)):
        for b in range(1 + i, batch, 9):
            col = (7 * b) % bt.shape[1]
            wild[b, col], zero[b, col] = bad, 0
    q, k, v, sl = q.cuda(), k.cuda(), v.cuda(), sl.cuda()
    out = _decode(kvt)(q, k, v, wild.cuda(), sl)
    assert torch.equal(out, _decode(kvt)(q, k, v, zero.cuda(), sl))


@pytest.mark.gpu
def test_list_of_other_lengths_keeps_the_scratch_consistent():
    """A range launch's list run with other lengths: rows of the planned items, and the next launches are right."""
    import paged_attention_decode_amd as pad

    case = FORMS[0]
    kind, batch, hkv, group, d, ps, room, qt, kvt = case
    lens, q, k, v, _, _ = _inputs(case)
    bt, num_pages = shuffled_table([room] * batch, ps, spare_pages=1, extra_cols=0, seed=2)
    k, v = make_cache(num_pages, ps, hkv, d, seed=3, dtype=torch.float16)
    other = lens[::-1]
    sla, slb = (torch.tensor(x, dtype=torch.int32).cuda() for x in (lens, other))
    qc, kc, vc, btc = q.cuda(), k.cuda(), v.cuda(), bt.cuda()
    w = pad.BatchDecodeWrapper()
    w.plan_block_table(btc, sla, hkv * group, hkv, d, ps)
    stale = pad.ops.ext().forward_worklist(qc, kc, vc, btc, slb, w._plan[2], d ** -0.5, 0)
    planned = w.run(qc, (kc, vc))
    assert torch.equal(stale, planned)  # every length comes from the list
    _check(planned, decode_fp16_protocol(q.float(), k.float(), v.float(), bt, torch.tensor(lens)), qt)
    out = pad.paged_attention_decode(qc, kc, vc, btc, slb)
    _check(out, decode_fp16_protocol(q.float(), k.float(), v.float(), bt, torch.tensor(other)), qt)


@pytest.mark.gpu
@pytest.mark.parametrize("scratch", ["planned", "least"])
def test_graph_capture_replays(scratch):
    """Replays equal the eager call's bits; with scratch for the per-unit kernel only, that kernel is captured."""
    import paged_attention_decode_amd as pad

    # 300 sequences: the per-unit kernel needs no scratch, so a stream without any captures it.
    batch, hkv, group, d, ps, room = 300, 1, 8, 128, 16, 4096
    lens, q, k, v, bt, sl = _inputs(("ragged", batch, hkv, group, d, ps, room, "fp16", "fp16"))
    assert heuristics.plan_units(batch, hkv * group, hkv, d, ps, bt.shape[1]).single_pass
    assert heuristics.range_launch(batch, hkv * group, hkv, d, ps, bt.shape[1]) is not None
    expected = decode_fp16_protocol(q.float(), k.float(), v.float(), bt, sl)
    dev = [k.cuda(), v.cuda(), bt.cuda(), sl.cuda()]
    qs = [q.cuda(), q.flip(0).contiguous().cuda()]
    q_static = qs[0].clone()
    eager = [pad.paged_attention_decode(x, *dev) for x in qs]
    per_unit = [pad.paged_attention_decode_ex(x, *dev, num_splits=1) for x in qs]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    if scratch == "planned":
        with torch.cuda.stream(s):
            pad.paged_attention_decode(q_static, *dev)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        out = pad.paged_attention_decode(q_static, *dev)
    for _ in range(3):
        for i, x in enumerate(qs):
            q_static.copy_(x)
            graph.replay()
            torch.cuda.synchronize()
            # (the runtime hands out streams again: one of an earlier test may hold more than the least)
            assert torch.equal(out, eager[i]) or (scratch == "least" and torch.equal(out, per_unit[i]))
            pad.paged_attention_decode(x, *dev)
            torch.cuda.synchronize()
            if i == 0:
                _check(out, expected, "fp16")


def test_plans_describe_one_kernel():
    """Splits, pages and waves of a plan are the per-unit kernel's; its scratch covers the range kernel too."""
    lib = _native.capi()
    taken = 0
    for batch, hq, hkv, d, ps, pages in ((64, 32, 8, 128, 16, 512), (70, 32, 8, 64, 16, 512), (300, 8, 1, 128, 16, 256),
                                         (33, 64, 4, 256, 16, 64), (100, 24, 6, 96, 16, 400), (8, 32, 8, 128, 16, 512)):
        u = heuristics.plan_units(batch, hq, hkv, d, ps, pages)
        m = heuristics.plan(batch, hq, hkv, d, ps, pages)
        r = heuristics.range_launch(batch, hq, hkv, d, ps, pages)
        taken += r is not None and r[2] != u.waves_per_group
        q, k = torch.empty(batch, hq, d, dtype=torch.float16), torch.empty(1, ps, hkv, d, dtype=torch.float16)
        index = torch.zeros(batch, pages, dtype=torch.int32)
        p = _native.PadPlan()
        dm = _native.dims_for(q, k, k, index, index[:, 0], q)
        assert lib.pad_decode_plan(ctypes.byref(dm), 0, 256, ctypes.byref(p)) == 0
        assert (p.num_splits, p.pages_per_split, p.waves_per_group) == (
            u.num_splits, u.pages_per_split, u.waves_per_group) == (m.num_splits, m.pages_per_split, m.waves_per_group)
        assert (bool(p.single_pass), p.workspace_bytes, p.counters) == (m.single_pass, m.workspace_bytes, m.counters)
    assert taken >= 1


def test_few_units_of_four_heads_stay_per_unit():
    r = heuristics.range_launch
    assert r(10, 64, 8, 128, 16, 208) is None and r(11, 64, 8, 128, 16, 202) is None  # 0.7 of the per-unit kernel's speed
    assert r(9, 32, 8, 128, 16, 4096) is None and r(24, 16, 4, 256, 16, 256) is None
    assert r(16, 32, 8, 128, 16, 512) is None and r(17, 32, 8, 128, 16, 512) == (256, 4, 4)
    assert r(9, 32, 8, 128, 16, 512, kv_bytes=1) is None and r(12, 32, 8, 128, 16, 256, kv_bytes=1) is not None
    assert r(9, 32, 8, 64, 16, 512) is not None  # 128-byte rows
    assert r(12, 24, 6, 128, 16, 288) is not None and r(70, 8, 1, 128, 16, 296) is not None  # one and two heads
    # the fp8 launch's scratch is in the 16-bit plan that sizes it
    for group in (1, 4, 16):
        plan = heuristics.plan(12, 8 * group, 8, 128, 16, 256)
        assert plan.workspace_bytes >= 256 + 2 * 256 * 4 * group * (128 * 4 + 8) and plan.counters >= 24 + 2 * 256


def test_shapes_that_take_the_range_kernel():
    r = heuristics.range_launch
    assert r(256, 64, 8, 128, 16, 2048) == (256, 4, 4)
    assert r(64, 32, 8, 128, 16, 512, kv_bytes=1) == (256, 4, 8)
    assert r(300, 8, 1, 128, 16, 256) == (256, 1, 4)
    assert r(70, 12, 6, 128, 16, 128) == (256, 2, 4)
    assert r(64, 12, 2, 128, 16, 256) is None  # two kv heads
    assert r(1, 32, 8, 128, 16, 8192) is None  # few units: the per-unit kernel's shorter merge
    assert r(200, 64, 8, 128, 16, 8) is None  # short rows
    assert r(43, 32, 8, 64, 16, 96) == (256, 4, 8) and r(42, 32, 8, 64, 16, 96) is None  # few bytes in all
    assert r(513, 8, 1, 128, 16, 4096) is None
    for batch, hq, hkv, d, ps, pages in ((256, 64, 8, 128, 16, 2048), (300, 8, 1, 128, 16, 256), (33, 64, 4, 256, 16, 64)):
        p = heuristics.plan(batch, hq, hkv, d, ps, pages)
        u = heuristics.plan_units(batch, hq, hkv, d, ps, pages)
        groups, heads, _ = r(batch, hq, hkv, d, ps, pages)
        rows = 2 * groups * heads * (hq // hkv)
        assert p.workspace_bytes >= max(u.workspace_bytes, rows * (d * 4 + 8)) and not p.single_pass
        assert p.counters >= max(u.counters, batch * hkv // heads + 2 * groups)
