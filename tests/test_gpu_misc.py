"""GPU parity of the small kernels: batch positions, page append (bf16,
fp16, e4m3), the e4m3 pool builder and RoPE, against the CPU oracle.
Integer and byte results must be bit-exact."""

import numpy as np
import pytest
import torch

import oracle as O
import pagedattn
from pagedattn import _lib
from pagedattn.metadata import decode_metadata, prefill_metadata

from paged_cases import i32, random_tables, strided_rows

pytestmark = pytest.mark.gpu


def test_one_hip_runtime(gpu):
    # the library must bind to torch's HIP runtime, not load a second one
    assert len(_lib.loaded_hip_runtimes()) == 1, _lib.loaded_hip_runtimes()
    assert _lib.lib().pagedattn_device_cu_count() > 0


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_batch_indices_positions(gpu, seed):
    rng = np.random.default_rng(seed)
    bsz = int(rng.integers(1, 40))
    counts = rng.integers(0, 600, size=bsz)
    counts[0] = 0  # an empty append range
    indptr = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    lens = (counts + rng.integers(0, 5000, size=bsz)).astype(np.int32)
    nnz = int(indptr[-1])
    bi, pos = pagedattn.get_batch_indices_positions(i32(indptr, gpu), i32(lens, gpu), nnz)
    ebi, epos = O.batch_indices_positions(indptr, lens, nnz)
    assert np.array_equal(bi.cpu().numpy(), ebi)
    assert np.array_equal(pos.cpu().numpy(), epos)


def _append_case(gpu, dtype, seed, prefill):
    rng = np.random.default_rng(seed)
    hkv, d = 4, 64
    if prefill:
        computed = [0, 16, 35, 100]
        chunks = [17, 1, 64, 29]
        lens = [c + n for c, n in zip(computed, chunks)]
        tables, num_pages = random_tables(rng, lens, extra_pages=5)
        meta = prefill_metadata(tables, computed, chunks)
    else:
        lens = rng.integers(1, 300, size=37).tolist()
        tables, num_pages = random_tables(rng, lens, extra_pages=5)
        meta = decode_metadata(tables, lens)
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    pool = torch.randn((num_pages, 2, hkv, 16, d), generator=g, device=gpu,
                       dtype=torch.float32).to(dtype)
    nnz = meta.nnz
    # k and v are strided views of one fused projection, as in the engine
    qkv = torch.randn((nnz, (8 + 2 * hkv) * d), generator=g, device=gpu,
                      dtype=torch.float32).to(dtype)
    k = qkv[:, 8 * d:(8 + hkv) * d].view(nnz, hkv, d)
    v = qkv[:, (8 + hkv) * d:].view(nnz, hkv, d)
    return meta, pool, k, v


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("prefill", [False, True])
def test_append_bit_exact(gpu, dtype, prefill):
    meta, pool, k, v = _append_case(gpu, dtype, 3, prefill)
    before = O.to_bits(pool)
    err = torch.zeros(1, dtype=torch.int32, device=gpu)
    pagedattn.append_paged_kv_cache(k, v, i32(meta.batch_indices, gpu), i32(meta.positions, gpu),
                                    pool, i32(meta.kv_indices, gpu), i32(meta.kv_indptr, gpu),
                                    i32(meta.kv_last_page_len, gpu), kv_layout="HND",
                                    error_flag=err)
    want, skipped = O.append_pages(before, O.to_bits(k), O.to_bits(v), meta.batch_indices,
                                   meta.positions, meta.kv_indices, meta.kv_indptr)
    assert skipped == 0 and int(err.item()) == 0
    assert np.array_equal(O.to_bits(pool), want)


def test_append_bad_metadata_is_skipped_and_counted(gpu):
    meta, pool, k, v = _append_case(gpu, torch.bfloat16, 4, False)
    bi = meta.batch_indices.copy()
    pos = meta.positions.copy()
    bi[0] = 1000  # no such sequence
    pos[1] = pos[1] + 16 * 50  # past the end of its table
    pos[2] = -3
    before = O.to_bits(pool)
    err = torch.zeros(1, dtype=torch.int32, device=gpu)
    pagedattn.append_paged_kv_cache(k, v, i32(bi, gpu), i32(pos, gpu), pool,
                                    i32(meta.kv_indices, gpu), i32(meta.kv_indptr, gpu),
                                    i32(meta.kv_last_page_len, gpu), kv_layout="HND",
                                    error_flag=err)
    want, skipped = O.append_pages(before, O.to_bits(k), O.to_bits(v), bi, pos,
                                   meta.kv_indices, meta.kv_indptr)
    assert skipped == 3 and int(err.item()) == 3
    assert np.array_equal(O.to_bits(pool), want)


def test_quantize_pages_bit_exact(gpu):
    g = torch.Generator(device=gpu)
    g.manual_seed(5)
    for d in (64, 128):
        pool = torch.randn((50, 2, 8, 16, d), generator=g, device=gpu).to(torch.bfloat16)
        pool[3, 1, 2] = 0
        pool[7, 0, 0, 3, 5] = 200.0  # an outlier sets the block scale
        q8, scales = pagedattn.quantize_pages_e4m3(pool)
        bits, ref_scales = O.quantize_pages(pool.cpu())
        assert torch.equal(scales.cpu(), ref_scales)
        assert np.array_equal(O.to_bits(q8), bits)


@pytest.mark.parametrize("src", [torch.bfloat16, torch.float16])
def test_append_e4m3_bit_exact(gpu, src):
    meta, pool, k, v = _append_case(gpu, src, 6, True)
    q8, scales = pagedattn.quantize_pages_e4m3(pool)
    # scale some rows up so the clamp at +-448 is exercised
    k = k * 40
    before = O.to_bits(q8)
    pagedattn.append_paged_kv_cache(k, v, i32(meta.batch_indices, gpu), i32(meta.positions, gpu),
                                    q8, i32(meta.kv_indices, gpu), i32(meta.kv_indptr, gpu),
                                    i32(meta.kv_last_page_len, gpu), kv_layout="HND",
                                    kv_scales=scales)
    want, skipped = O.append_pages_e4m3(before, scales.cpu(), k.cpu(), v.cpu(),
                                        meta.batch_indices, meta.positions, meta.kv_indices,
                                        meta.kv_indptr)
    assert skipped == 0
    assert np.array_equal(O.to_bits(q8), want)


@pytest.mark.parametrize("src", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("with_rope", [False, True])
def test_append_e4m3_fixed_scale_counts(gpu, src, with_rope):
    # fixed-scale e4m3 appends (stand-alone and RoPE-fused) count every
    # skipped token in error_flag[0] and every clamped 8-element piece in
    # error_flag[1]; blocks with a zero or infinite scale get zero codes and
    # are counted as clamped too
    meta, pool, k, v = _append_case(gpu, src, 16, True)
    q8, scales = pagedattn.quantize_pages_e4m3(pool)
    pages = meta.kv_indices
    scales[int(pages[0]), 0, 1] = 0.0
    scales[int(pages[3]), 1, 2] = float("inf")
    k = (k.float() * 40).to(src)
    bi = meta.batch_indices.copy()
    pos = meta.positions.copy()
    bi[5] = 999
    pos[7] = -1
    g = torch.Generator(device=gpu)
    g.manual_seed(17)
    q = torch.randn((meta.nnz, 8, k.shape[2]), generator=g, device=gpu).to(src)
    before = O.to_bits(q8)
    ka = k.clone()
    if with_rope:
        qa = q.clone()
        pagedattn.apply_rope_pos_ids_inplace(qa, ka, i32(pos, gpu), rope_theta=1e4,
                                             rope_scale=1.0)
    want, skipped = O.append_pages_e4m3(before, scales.cpu(), ka.cpu().float(), v.cpu().float(),
                                        bi, pos, meta.kv_indices, meta.kv_indptr)
    clamped = O.e4m3_clamped_pieces(ka.cpu().float(), v.cpu().float(), scales.cpu(), bi, pos,
                                    meta.kv_indices, meta.kv_indptr, q8.shape[0])
    assert skipped == 2 and clamped > 2 * (k.shape[2] // 8)
    err = torch.zeros(2, dtype=torch.int32, device=gpu)
    args = (i32(bi, gpu), i32(pos, gpu), q8, i32(meta.kv_indices, gpu),
            i32(meta.kv_indptr, gpu), i32(meta.kv_last_page_len, gpu))
    if with_rope:
        pagedattn.rope_append_paged_kv_cache(q, k, v, *args, kv_layout="HND", rope_scale=1.0,
                                             rope_theta=1e4, kv_scales=scales, error_flag=err)
    else:
        pagedattn.append_paged_kv_cache(k, v, *args, kv_layout="HND", kv_scales=scales,
                                        error_flag=err)
    torch.cuda.synchronize()
    assert np.array_equal(O.to_bits(q8), want)
    assert err.tolist() == [skipped, clamped]


def _bf16_ulp(x: torch.Tensor) -> torch.Tensor:
    e = torch.floor(torch.log2(x.abs().clamp_min(2.0 ** -100)))
    return torch.pow(2.0, e - 7)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("theta,scale,interleave", [(10000.0, 1.0, False),
                                                    (500000.0, 1.0, False),
                                                    (10000.0, 4.0, True)])
def test_rope(gpu, dtype, theta, scale, interleave):
    g = torch.Generator(device=gpu)
    g.manual_seed(7)
    n, hq, hkv, d = 300, 32, 8, 128
    qkv = torch.randn((n, (hq + 2 * hkv) * d), generator=g, device=gpu).to(dtype)
    q = qkv[:, :hq * d].view(n, hq, d)
    k = qkv[:, hq * d:(hq + hkv) * d].view(n, hkv, d)
    pos = torch.randint(0, 131072, (n,), generator=g, device=gpu, dtype=torch.int32)
    q0, k0 = q.float().cpu(), k.float().cpu()
    v_before = qkv[:, (hq + hkv) * d:].clone()
    pagedattn.apply_rope_pos_ids_inplace(q, k, pos, interleave=interleave, rope_scale=scale,
                                         rope_theta=theta)
    rq = O.rope(q0, pos.cpu().numpy(), theta, scale, interleave=interleave)
    rk = O.rope(k0, pos.cpu().numpy(), theta, scale, interleave=interleave)
    # within one ulp of the 16-bit result (fp32 sin/cos vs fp64 angles)
    tol = (_bf16_ulp(rq) if dtype == torch.bfloat16 else rq.abs() * 2.0 ** -10) + 1e-5
    assert bool(((q.float().cpu() - rq).abs() <= tol).all())
    tolk = (_bf16_ulp(rk) if dtype == torch.bfloat16 else rk.abs() * 2.0 ** -10) + 1e-5
    assert bool(((k.float().cpu() - rk).abs() <= tolk).all())
    assert torch.equal(qkv[:, (hq + hkv) * d:], v_before)  # v untouched


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("prefill", [False, True])
@pytest.mark.parametrize("fp8", [False, True])
def test_rope_append_equals_separate(gpu, dtype, prefill, fp8):
    # one launch == apply_rope_pos_ids_inplace then append_paged_kv_cache,
    # bit for bit: rotated q and k in place and the pool
    meta, pool, k, v = _append_case(gpu, dtype, 5, prefill)
    hq = 8
    g = torch.Generator(device=gpu)
    g.manual_seed(6)
    q = strided_rows(meta.nnz, hq, pool.shape[-1], dtype, gpu, g, lead=0, tail=8)
    scales = None
    if fp8:
        pool, scales = pagedattn.quantize_pages_e4m3(pool)
    pos = meta.positions.copy()
    bi = meta.batch_indices.copy()
    bi[0] = 1000  # a token the append must skip (and count); RoPE still rotates it
    args = dict(kv_layout="HND", kv_scales=scales)
    q_a, k_a, pool_a = q.clone(), k.clone(), pool.clone()
    err_a = torch.zeros(2, dtype=torch.int32, device=gpu)
    pagedattn.apply_rope_pos_ids_inplace(q_a, k_a, i32(pos, gpu), rope_theta=500000.0,
                                         rope_scale=2.0)
    pagedattn.append_paged_kv_cache(k_a, v, i32(bi, gpu), i32(pos, gpu), pool_a,
                                    i32(meta.kv_indices, gpu), i32(meta.kv_indptr, gpu),
                                    i32(meta.kv_last_page_len, gpu), error_flag=err_a, **args)
    q_b, k_b, pool_b = q.clone(), k.clone(), pool.clone()
    err_b = torch.zeros(2, dtype=torch.int32, device=gpu)
    pagedattn.rope_append_paged_kv_cache(q_b, k_b, v, i32(bi, gpu), i32(pos, gpu), pool_b,
                                         i32(meta.kv_indices, gpu), i32(meta.kv_indptr, gpu),
                                         i32(meta.kv_last_page_len, gpu), rope_scale=2.0,
                                         rope_theta=500000.0, error_flag=err_b, **args)
    torch.cuda.synchronize()
    assert torch.equal(q_a, q_b)
    assert torch.equal(k_a, k_b)
    assert np.array_equal(O.to_bits(pool_a), O.to_bits(pool_b))
    # the skipped token, plus (e4m3) the 8-element pieces clamped at +-448:
    # new rows are not bounded by the pool's per-page amax scales
    clamped = 0
    if fp8:
        clamped = O.e4m3_clamped_pieces(k_a.cpu().float(), v.cpu().float(), scales.cpu(), bi,
                                        pos, meta.kv_indices, meta.kv_indptr, pool.shape[0])
    assert err_a.tolist() == err_b.tolist() == [1, clamped]


@pytest.mark.parametrize("d,hq,hkv,nnz", [
    (16, 1, 1, 1),      # one chunk pair a head, one token
    (48, 3, 1, 7),      # pairs not a power of two, tokens not a multiple of the workgroup's
    (64, 32, 4, 33),
    (128, 8, 1, 5),     # few heads: four tokens a workgroup
    (128, 64, 8, 18),   # more units than one batch of loads
    (160, 2, 2, 9),     # two frequency blocks, the second partial
    (256, 16, 16, 3),
    (48, 1, 1, 17001),  # few heads, many tokens: 16 tokens a workgroup, the last one's partial
    (64, 4, 1, 5131),   # 5 tokens a workgroup, more than its waves
    (128, 4, 4, 8197),  # 8 tokens a workgroup, the most lanes a token for that
])
def test_rope_append_shapes_equal_separate(gpu, d, hq, hkv, nnz):
    # the workgroup split of the fused launch at its edges: same bits as the
    # two calls, for every head of q, k and v and every page slot
    g = torch.Generator(device=gpu)
    g.manual_seed(d + hq)
    n_pages = -(-nnz // 16) + 1
    pool = torch.randn((n_pages, 2, hkv, 16, d), generator=g, device=gpu).to(torch.bfloat16)
    qkv = torch.randn((nnz, (hq + 2 * hkv) * d), generator=g, device=gpu).to(torch.bfloat16)
    ind = i32(np.arange(n_pages)[::-1].copy(), gpu)
    indptr, last = i32([0, n_pages], gpu), i32([nnz % 16 + 1], gpu)
    bi, pos = i32(np.zeros(nnz), gpu), i32(np.arange(1, nnz + 1), gpu)

    def views(x):
        q, k, v = x.split([hq * d, hkv * d, hkv * d], dim=-1)
        return q.view(nnz, hq, d), k.view(nnz, hkv, d), v.view(nnz, hkv, d)

    a, b, pool_a, pool_b = qkv.clone(), qkv.clone(), pool.clone(), pool.clone()
    q, k, v = views(a)
    pagedattn.apply_rope_pos_ids_inplace(q, k, pos, rope_theta=500000.0)
    pagedattn.append_paged_kv_cache(k, v, bi, pos, pool_a, ind, indptr, last, kv_layout="HND")
    q, k, v = views(b)
    pagedattn.rope_append_paged_kv_cache(q, k, v, bi, pos, pool_b, ind, indptr, last,
                                         kv_layout="HND", rope_theta=500000.0)
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    assert torch.equal(pool_a, pool_b)


@pytest.mark.parametrize("dtype,fp8", [(torch.bfloat16, False), (torch.float16, False),
                                       (torch.bfloat16, True)])
def test_native_calls_equal_the_general_path(gpu, monkeypatch, dtype, fp8):
    # every per-layer call through the extension, which takes all of them, and,
    # with it switched off, through the general path: same bits; calls with int64
    # metadata go the general way
    hq, hkv, d = 8, 2, 64
    g = torch.Generator(device=gpu)
    g.manual_seed(3)
    meta = prefill_metadata([[3, 1], [0, 4, 2]], [10, 20], [9, 20])
    pool0 = torch.randn((6, 2, hkv, 16, d), generator=g, device=gpu).to(dtype)
    scales0 = None
    if fp8:
        pool0, scales0 = pagedattn.quantize_pages_e4m3(pool0)
        scales0 = torch.exp2(torch.ceil(torch.log2(scales0)))
    qkv0 = torch.randn((meta.nnz, (hq + 2 * hkv) * d), generator=g, device=gpu).to(dtype)
    ind, indptr = i32(meta.kv_indices, gpu), i32(meta.kv_indptr, gpu)
    last, qo = i32(meta.kv_last_page_len, gpu), i32(meta.qo_indptr, gpu)
    bi, pos = i32(meta.batch_indices, gpu), i32(meta.positions, gpu)
    ws = torch.zeros(1 << 24, dtype=torch.uint8, device=gpu)

    def step(cast):
        pool, qkv = pool0.clone(), qkv0.clone()
        scales = None if scales0 is None else scales0.clone()
        q, k, v = (x.view(meta.nnz, -1, d) for x in
                   qkv.split([hq * d, hkv * d, hkv * d], dim=-1))
        flag = torch.zeros(2, dtype=torch.int32, device=gpu)
        m = (cast(bi), cast(pos), pool, cast(ind), cast(indptr), last)
        res = []
        pagedattn.append_paged_kv_cache(k, v, *m, kv_layout="HND", kv_scales=scales,
                                        error_flag=flag)
        res += [pool.clone(), flag.clone()]
        pagedattn.rope_append_paged_kv_cache(q, k, v, *m, kv_layout="HND", kv_scales=scales,
                                             rope_theta=5e5)
        res += [pool.clone(), qkv.clone()]
        if fp8:
            pagedattn.append_paged_kv_cache_e4m3_amax(k, v, *m, scales, kv_layout="HND")
            res += [pool.clone(), scales.clone()]
        pw = pagedattn.BatchPrefillWithPagedKVCacheWrapper(ws, "HND")
        pw.plan(qo, indptr, ind, last, hq, hkv, d, 16, causal=True, q_data_type=dtype)
        res += [pw.run(q, pool, kv_scales=scales)]
        res += list(pw.run(q, pool, kv_scales=scales, causal=False, sm_scale=0.2,
                           out=torch.empty_like(res[-1]), return_lse=True))
        dw = pagedattn.BatchDecodeWithPagedKVCacheWrapper(ws, "HND")
        dw.plan(indptr, ind, last, hq, hkv, d, 16, q_data_type=dtype)
        q2, k2, v2 = (x[:2] for x in (q, k, v))
        lse = torch.empty((2, hq), device=gpu)
        res += [dw.run(q2, pool, kv_scales=scales)]
        res += list(dw.run(q2, pool, kv_scales=scales, lse=lse, return_lse=True))
        assert res[-1] is lse
        res += [dw.run(q2, pool, kv_scales=scales, append_key=k2, append_value=v2)]
        res += [dw.run(q2, pool, kv_scales=scales, append_key=k2, append_value=v2,
                       rope=(1.0, 5e5), positions=cast(last * 0 + 17)), pool]
        torch.cuda.synchronize()
        return res

    took = []
    native = pagedattn.ops._native

    def record(fn, *args):
        r = native(fn, *args)
        took.append((fn, r is not NotImplemented))
        return r

    monkeypatch.setattr(pagedattn.ops, "_native", record)
    want = step(lambda t: t)
    writes = ["append", "rope_append"] + ["append_amax"] * fp8
    assert took == [(fn, True) for fn in writes + ["prefill_run"] * 2 + ["decode_run"] * 4]
    took.clear()
    wide = step(lambda t: t.long())
    assert took == ([(fn, False) for fn in writes] + [("prefill_run", True)] * 2
                    + [("decode_run", True)] * 3 + [("decode_run", False)])
    monkeypatch.setattr(pagedattn.ops, "_native", lambda *a: NotImplemented)
    general = step(lambda t: t)
    for x, y, z in zip(want, wide, general):
        x, y, z = (t.view(torch.uint8) if t.dtype == torch.float8_e4m3fn else t
                   for t in (x, y, z))
        assert torch.equal(x, y) and torch.equal(x, z)


@pytest.mark.parametrize("native", [True, False])
def test_runs_refuse_outputs_they_would_overrun(gpu, monkeypatch, native):
    # out and lse are written through raw pointers: anything but q's dtype (lse:
    # float32), enough entries in order and q's device is refused before a launch
    if not native:
        monkeypatch.setattr(pagedattn.ops, "_native", lambda *a: NotImplemented)
    hq, hkv, d = 8, 2, 64
    meta = prefill_metadata([[0, 1], [2, 3]], [10, 20], [2, 3])
    pool = torch.zeros((4, 2, hkv, 16, d), dtype=torch.bfloat16, device=gpu)
    args = [i32(a, gpu) for a in (meta.kv_indptr, meta.kv_indices, meta.kv_last_page_len)]
    ws = torch.zeros(1 << 20, dtype=torch.uint8, device=gpu)
    dw = pagedattn.BatchDecodeWithPagedKVCacheWrapper(ws, "HND")
    dw.plan(*args, hq, hkv, d, 16, q_data_type=torch.bfloat16)
    pw = pagedattn.BatchPrefillWithPagedKVCacheWrapper(ws.clone(), "HND")
    pw.plan(i32(meta.qo_indptr, gpu), *args, hq, hkv, d, 16, q_data_type=torch.bfloat16)
    for w, n in ((dw, 2), (pw, meta.nnz)):
        q = torch.ones((n, hq, d), dtype=torch.bfloat16, device=gpu)
        for out in (torch.empty((n, hq, d), dtype=torch.uint8, device=gpu),
                    torch.empty((n, hq, d), dtype=torch.float16, device=gpu),
                    torch.empty((n, hq, d), dtype=q.dtype)):
            with pytest.raises(ValueError, match="out must be"):
                w.run(q, pool, out=out)
        for lse in (torch.empty((n, hq)), torch.empty((n, hq), dtype=q.dtype, device=gpu),
                    torch.empty((n, hq - 1), device=gpu),
                    torch.empty((n, 2 * hq), device=gpu)[:, ::2]):
            with pytest.raises(ValueError, match="lse must be"):
                w.run(q, pool, lse=lse, return_lse=True)
        # more room than needed, in any shape, is taken as it was
        big = torch.full((n * hq + 3,), -1.0, device=gpu)
        out, lse = w.run(q, pool, lse=big, return_lse=True)
        assert lse is big and torch.equal(big[n * hq:], torch.full((3,), -1.0, device=gpu))
        assert torch.equal(big[:n * hq].view(n, hq), w.run(q, pool, return_lse=True)[1])


def test_native_calls_refuse_what_the_general_path_refuses(gpu, monkeypatch):
    # the extension repeats the general path's checks: bad device arguments end
    # in the same errors with it and without it
    n, hq, hkv, d = 2, 8, 2, 64
    dev = dict(device=gpu)
    bf = dict(dtype=torch.bfloat16, **dev)
    meta = prefill_metadata([[0], [1]], [3, 4], [1, 1])
    ind, indptr = i32(meta.kv_indices, gpu), i32(meta.kv_indptr, gpu)
    last, qo = i32(meta.kv_last_page_len, gpu), i32(meta.qo_indptr, gpu)
    bi, pos = i32(meta.batch_indices, gpu), i32(meta.positions, gpu)
    pool, q = torch.zeros((2, 2, hkv, 16, d), **bf), torch.ones((n, hq, d), **bf)
    k = torch.ones((n, hkv, d), **bf)
    pool8 = torch.zeros(pool.shape, dtype=torch.uint8, **dev).view(torch.float8_e4m3fn)
    scales = torch.ones((2, 2, hkv), **dev)
    ws = torch.zeros(1 << 20, dtype=torch.uint8, device=gpu)
    dw = pagedattn.BatchDecodeWithPagedKVCacheWrapper(ws, "HND")
    dw.plan(indptr, ind, last, hq, hkv, d, 16, q_data_type=torch.bfloat16)
    pw = pagedattn.BatchPrefillWithPagedKVCacheWrapper(ws.clone(), "HND")
    pw.plan(qo, indptr, ind, last, hq, hkv, d, 16, q_data_type=torch.bfloat16)
    bad_q = [q[:, :4], q[..., :32], q[:1], q.float(), q.to(torch.float16), q[0],
             torch.ones((n, hq, 2 * d), **bf)[..., ::2]]
    bad_pool = [pool[:, :1], pool[:, :, :1], pool[..., :32], pool.float(), pool.to(torch.float16),
                pool[:, :, :, :8], pool[0], torch.zeros((2, 2, hkv, 16, 2 * d), **bf)[..., ::2]]
    bad_scales = [None, scales[:1], scales.half(), scales.cpu()]
    bad_rows = [k[:, :1], k[:1], k[..., :32], k.float(), k.to(torch.float16)]
    meta_args = (bi, pos, pool, ind, indptr, last)
    rope = dict(rope=(1.0, 1e4))
    calls = [lambda w=w, x=x: w.run(x, pool) for w in (dw, pw) for x in bad_q]
    calls += [lambda w=w, x=x: w.run(q, x) for w in (dw, pw) for x in bad_pool]
    calls += [lambda w=w, x=x: w.run(q, pool8, kv_scales=x) for w in (dw, pw) for x in bad_scales]
    calls += [lambda x=x, r=r: dw.run(q, pool, append_key=x, append_value=k, **r)
              for x in bad_rows for r in ({}, rope)]
    calls += [lambda x=x: dw.run(q, pool, append_key=k, append_value=x) for x in [None] + bad_rows]
    calls += [lambda: dw.run(q, pool, append_value=k),
              lambda: dw.run(q, pool, append_key=k, append_value=k, positions=pos),
              lambda: dw.run(q, pool, append_key=k, append_value=k, positions=pos[:1], **rope),
              lambda: dw.run(q, pool, append_key=k, append_value=k, rope=(0.0, 1e4)),
              lambda: pw.run(q, pool, sm_scale=-1.0)]
    hnd = dict(kv_layout="HND")
    for x in bad_rows:
        calls += [lambda x=x: pagedattn.append_paged_kv_cache(x, k, *meta_args, **hnd),
                  lambda x=x: pagedattn.append_paged_kv_cache(k, x, *meta_args, **hnd),
                  lambda x=x: pagedattn.rope_append_paged_kv_cache(q, x, k, *meta_args, **hnd),
                  lambda x=x: pagedattn.append_paged_kv_cache_e4m3_amax(
                      x if x.dtype != torch.float16 else x[:1], k, bi, pos, pool8, ind, indptr,
                      last, scales)]
    for x in (bi[:1], torch.cat([bi, bi])):
        calls += [lambda x=x: pagedattn.append_paged_kv_cache(k, k, x, *meta_args[1:], **hnd),
                  lambda x=x: pagedattn.rope_append_paged_kv_cache(q, k, k, bi, x, *meta_args[2:],
                                                                   **hnd)]
    for x in bad_scales:
        calls += [lambda x=x: pagedattn.append_paged_kv_cache(k, k, bi, pos, pool8, ind, indptr,
                                                              last, kv_scales=x, **hnd)]
    flag = torch.zeros(1, dtype=torch.int32, **dev)
    calls += [lambda f=f: pagedattn.append_paged_kv_cache(k, k, bi, pos, pool8, ind, indptr, last,
                                                          kv_scales=scales, error_flag=f, **hnd)
              for f in (flag, flag.long(), flag.cpu())]

    def errors():
        got = []
        for i, call in enumerate(calls):
            with pytest.raises((ValueError, NotImplementedError, RuntimeError, TypeError)) as e:
                call()
                pytest.fail(f"call {i} was taken")
            got.append((type(e.value), str(e.value)))
        return got

    with_native = errors()
    monkeypatch.setattr(pagedattn.ops, "_native", lambda *a: NotImplemented)
    assert errors() == with_native
