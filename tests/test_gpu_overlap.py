"""Runs of one plan that overlap on the GPU (the layers of one forward share a
plan, src/models/llama.py:212-245; here two streams run it at once): plans that
cut KV ranges take their partials from scratch of the run's own, so each run
gives the bits it gives alone.  Without scratch the plan's whole form runs."""

import math

import pytest
import torch

import pagedattn
from pagedattn import _lib

from paged_cases import decode_case, i32, prefill_case, workspace

pytestmark = pytest.mark.gpu

HQ, HKV, D = 16, 2, 128


@pytest.fixture(autouse=True)
def _default_planner(monkeypatch):
    for var in ("PAGEDATTN_PREFILL_SPLIT", "PAGEDATTN_DECODE_SHARED",
                "PAGEDATTN_DECODE_SHARED_SLACK_KB", "PAGEDATTN_DECODE_DETERMINISTIC"):
        monkeypatch.delenv(var, raising=False)


def _wrapper(gpu, kind, ws=None):
    """A planned wrapper, the pool, a q and the kernel-facing metadata."""
    ws = workspace(gpu) if ws is None else ws
    if kind == "decode":
        meta, pool, q = decode_case(gpu, [9001, 8990], HQ, HKV, D, seed=1)
        w = pagedattn.BatchDecodeWithPagedKVCacheWrapper(ws, "HND")
        args = [i32(meta.kv_indptr, gpu), i32(meta.kv_indices, gpu),
                i32(meta.kv_last_page_len, gpu)]
        w.plan(*args, HQ, HKV, D, 16, q_data_type=q.dtype)
    else:
        meta, pool, q = prefill_case(gpu, [6000, 500], [90, 64], HQ, HKV, D, seed=2)
        w = pagedattn.BatchPrefillWithPagedKVCacheWrapper(ws, "HND")
        args = [i32(meta.qo_indptr, gpu), i32(meta.kv_indptr, gpu), i32(meta.kv_indices, gpu),
                i32(meta.kv_last_page_len, gpu)]
        device = dict(device_plan=True, max_qo_tokens=meta.nnz) if kind == "device" else {}
        w.plan(*args, HQ, HKV, D, 16, causal=True, q_data_type=q.dtype, **device)
        w.update_plan()
    return w, pool, q, args


def _scratch_bytes(w):
    return _lib.lib().pagedattn_plan_scratch_bytes(w._plan.handle, 1)


@pytest.mark.parametrize("kind", ["decode", "host", "device"])
@pytest.mark.parametrize("native", [True, False])
def test_overlapping_runs_of_one_plan(gpu, monkeypatch, kind, native):
    if not native:
        monkeypatch.setattr(pagedattn.ops, "_native", lambda *a: NotImplemented)
    w, pool, q, _ = _wrapper(gpu, kind)
    assert _scratch_bytes(w) > 0
    qs = [q, q.flip(0).contiguous()]
    want = [w.run(x, pool, return_lse=True) for x in qs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in qs]
    got = [[], []]
    for _ in range(20):
        for s, x, g in zip(streams, qs, got):
            with torch.cuda.stream(s):
                g.append(w.run(x, pool, return_lse=True))
    torch.cuda.synchronize()
    for (o, l), g in zip(want, got):
        assert all(torch.equal(o, a) and torch.equal(l, b) for a, b in g)


@pytest.mark.parametrize("kind", ["host", "device"])
def test_prefill_calls_without_scratch_run_whole_tiles(gpu, monkeypatch, kind):
    # the C call without scratch: the bits of a plan that may not cut
    w, pool, q, (qo, indptr, ind, last) = _wrapper(gpu, kind)
    cut, _ = w.run(q, pool, return_lse=True)
    lib = _lib.lib()
    out = torch.empty_like(cut)
    head = (w._plan.handle, q.data_ptr(), q.stride(0), q.stride(1), _lib.BF16, qo.data_ptr(),
            pool.data_ptr(), _lib.BF16, None, pool.shape[0], ind.data_ptr(), ind.numel(),
            indptr.data_ptr(), last.data_ptr(), out.data_ptr(), None, 1, 1.0 / math.sqrt(D))
    assert lib.pagedattn_prefill_run(*head, _lib.stream_of(gpu)) == 0
    small = torch.empty(_scratch_bytes(w) - 256, dtype=torch.uint8, device=gpu)
    assert lib.pagedattn_prefill_run_scratch(*head, small.data_ptr(), small.numel(),
                                             _lib.stream_of(gpu)) == 3
    assert lib.pagedattn_prefill_run_scratch(*head, small.data_ptr() + 16, small.numel(),
                                             _lib.stream_of(gpu)) == 1
    monkeypatch.setenv("PAGEDATTN_PREFILL_SPLIT", "0")
    w2, _, _, _ = _wrapper(gpu, kind)
    assert _scratch_bytes(w2) == 0
    assert torch.equal(out, w2.run(q, pool)) and not torch.equal(out, cut)


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("kind", ["decode", "host", "device"])
def test_runs_without_memory_for_scratch(gpu, monkeypatch, kind, native):
    # no memory for the scratch: the whole form, as with a workspace too small
    # for the partials
    if not native:
        monkeypatch.setattr(pagedattn.ops, "_native", lambda *a: NotImplemented)
    small = torch.zeros(1 << 18 if kind != "decode" else 1 << 13, dtype=torch.uint8, device=gpu)
    w0, pool, q, _ = _wrapper(gpu, kind, ws=small)
    assert _scratch_bytes(w0) == 0
    want = w0.run(q, pool)
    w, _, _, _ = _wrapper(gpu, kind)
    cut, out = w.run(q, pool), torch.empty_like(want)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    hold = []
    try:
        # what is left of the blocks in use, then no more from the device
        torch.cuda.set_per_process_memory_fraction(1e-9)
        for size in (16 << 20, 2 << 20, (1 << 20) + 512, 1 << 18, 1 << 14, 512):
            while True:
                try:
                    hold.append(torch.empty(size, dtype=torch.uint8, device=gpu))
                except torch.OutOfMemoryError:
                    break
        w.run(q, pool, out=out)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    torch.cuda.synchronize()
    assert torch.equal(out, want) and not torch.equal(out, cut)
