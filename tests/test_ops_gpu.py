"""GPU numerics: every HIP kernel vs its plain-PyTorch fp32 reference
(tests run on a real MI355X via gpurun; marked gpu)."""
import math
import os

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.gpu

import rbg_amd.ops as ops
from rbg_amd.ops import reference as ref


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available()
    torch.manual_seed(1234)
    return torch.device("cuda:0")


def test_hip_extension_loaded(dev):
    # on a GPU box the native extension must be the path that runs
    ops.require("_hip_ops")


def test_mfma_fragment_layout(dev):
    """Empirically identify the v_mfma_f32_16x16x32_bf16 operand layout
    (guide §3: asymmetric operands, transpose-detecting)."""
    a = torch.randn(16, 32, dtype=torch.bfloat16, device=dev)
    b = torch.randn(32, 16, dtype=torch.bfloat16, device=dev)
    want = a.float() @ b.float()
    results = {}
    for a_s in (0, 1):
        for b_s in (0, 1):
            d = ops._hip.mfma_probe(a.contiguous(), b.contiguous(), a_s, b_s)
            results[(a_s, b_s)] = (d - want).abs().max().item()
    best = min(results, key=results.get)
    assert results[best] < 0.1, f"no layout matched: {results}"
    # the kernels assume contiguous-8 per lane (0,0); fail loudly otherwise
    assert best == (0, 0), (
        f"MFMA layout is {best}, kernels assume (0,0); errors={results}")


def test_rmsnorm(dev):
    for T, H in ((1, 4096), (17, 4096), (256, 8192), (64, 1024)):
        x = torch.randn(T, H, dtype=torch.bfloat16, device=dev)
        w = torch.randn(H, dtype=torch.bfloat16, device=dev)
        got = ops.rmsnorm(x, w, 1e-5).float()
        want = ref.rmsnorm(x, w, 1e-5).float()
        assert torch.allclose(got, want, atol=2e-2, rtol=2e-2), \
            (T, H, (got - want).abs().max().item())


def test_fused_add_rmsnorm(dev):
    T, H = 33, 4096
    x = torch.randn(T, H, dtype=torch.bfloat16, device=dev)
    res = torch.randn(T, H, dtype=torch.bfloat16, device=dev)
    w = torch.randn(H, dtype=torch.bfloat16, device=dev)
    x2, res2 = x.clone(), res.clone()
    ops.fused_add_rmsnorm(x, res, w, 1e-5)
    ref.fused_add_rmsnorm(x2, res2, w, 1e-5)
    assert torch.allclose(res.float(), res2.float(), atol=2e-2, rtol=2e-2)
    assert torch.allclose(x.float(), x2.float(), atol=2e-2, rtol=2e-2)


def test_silu_mul(dev):
    T, I = 129, 14336
    x = torch.randn(T, 2 * I, dtype=torch.bfloat16, device=dev)
    got = ops.silu_mul(x).float()
    want = ref.silu_mul(x).float()
    assert torch.allclose(got, want, atol=2e-2, rtol=2e-2)


def _mk_cache(dev, pages=64, kvh=8, page=16, d=128):
    kc = torch.zeros(pages, kvh, page, d, dtype=torch.bfloat16, device=dev)
    vc = torch.zeros_like(kc)
    return kc, vc


def test_rope_store_kv(dev):
    T, QH, KVH, D, page = 37, 32, 8, 128, 16
    q = torch.randn(T, QH, D, dtype=torch.bfloat16, device=dev)
    k = torch.randn(T, KVH, D, dtype=torch.bfloat16, device=dev)
    v = torch.randn(T, KVH, D, dtype=torch.bfloat16, device=dev)
    cos_sin = ref.build_cos_sin_table(D, 4096, device=dev)
    positions = torch.randint(0, 4096, (T,), dtype=torch.int32, device=dev)
    slots = torch.randperm(64 * page, device=dev)[:T].to(torch.int32)
    kc, vc = _mk_cache(dev)
    kc2, vc2 = _mk_cache(dev)
    q2, k2, v2 = q.clone(), k.clone(), v.clone()
    ops.rope_store_kv(q, k, v, kc, vc, cos_sin, positions, slots)
    ref.rope_store_kv(q2, k2, v2, kc2, vc2, cos_sin, positions, slots)
    assert torch.allclose(q.float(), q2.float(), atol=2e-2, rtol=2e-2)
    assert torch.allclose(k.float(), k2.float(), atol=2e-2, rtol=2e-2)
    assert torch.allclose(kc.float(), kc2.float(), atol=2e-2, rtol=2e-2)
    assert torch.allclose(vc.float(), vc2.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("qpg,splits", [(4, 1), (4, 4), (8, 1), (1, 2)])
def test_decode_attention(dev, qpg, splits):
    KVH, D, page = 8, 128, 16
    QH = KVH * qpg
    S = 5
    ctx_lens = torch.tensor([1, 16, 57, 300, 777], dtype=torch.int32,
                            device=dev)
    max_pages = (int(ctx_lens.max()) + page - 1) // page
    total_pages = int((torch.div(ctx_lens + page - 1, page,
                                 rounding_mode="floor")).sum())
    kc = torch.randn(total_pages + 1, KVH, page, D, dtype=torch.bfloat16,
                     device=dev)
    vc = torch.randn_like(kc)
    bt = torch.zeros(S, max_pages, dtype=torch.int32, device=dev)
    nxt = 0
    for s in range(S):
        n = (int(ctx_lens[s]) + page - 1) // page
        bt[s, :n] = torch.arange(nxt, nxt + n, dtype=torch.int32, device=dev)
        nxt += n
    q = torch.randn(S, QH, D, dtype=torch.bfloat16, device=dev)
    scale = 1.0 / math.sqrt(D)
    got = ops._hip.decode_attention(q, kc, vc, bt, ctx_lens, scale, splits, 0)
    got_w = ops._hip.decode_attention(q, kc, vc, bt, ctx_lens, scale, splits, 1)
    want = ref.decode_attention(q, kc, vc, bt, ctx_lens, scale)
    err = (got.float() - want.float()).abs().max().item()
    assert err < 3e-2, f"qpg={qpg} splits={splits} err={err}"
    err_w = (got_w.float() - want.float()).abs().max().item()
    assert err_w < 3e-2, f"WIDE qpg={qpg} splits={splits} err={err_w}"


@pytest.mark.parametrize("lens", [[128], [64, 200, 1], [2048], [33, 129]])
def test_prefill_attention(dev, lens):
    QH, KVH, D = 32, 8, 128
    T = sum(lens)
    q = torch.randn(T, QH, D, dtype=torch.bfloat16, device=dev)
    k = torch.randn(T, KVH, D, dtype=torch.bfloat16, device=dev)
    v = torch.randn(T, KVH, D, dtype=torch.bfloat16, device=dev)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)),
                      dtype=torch.int32, device=dev)
    scale = 1.0 / math.sqrt(D)
    got = ops.prefill_attention(q, k, v, cu, scale)
    want = ref.prefill_attention(q, k, v, cu, scale)
    err = (got.float() - want.float()).abs().max().item()
    assert err < 3e-2, f"lens={lens} err={err}"


def test_prefill_attention_spiked_scores(dev):
    """Force large per-tile max jumps (rule 26: exercise the rescale path)."""
    QH, KVH, D = 4, 4, 128
    L = 512
    q = torch.randn(L, QH, D, dtype=torch.bfloat16, device=dev)
    k = torch.randn(L, KVH, D, dtype=torch.bfloat16, device=dev)
    # spike one late key against everything
    k[400] *= 30.0
    v = torch.randn(L, KVH, D, dtype=torch.bfloat16, device=dev)
    cu = torch.tensor([0, L], dtype=torch.int32, device=dev)
    got = ops.prefill_attention(q, k, v, cu, 1.0 / math.sqrt(D))
    want = ref.prefill_attention(q, k, v, cu, 1.0 / math.sqrt(D))
    err = (got.float() - want.float()).abs().max().item()
    assert err < 5e-2, f"spiked err={err}"


@pytest.mark.parametrize("lens", [[(96, 32)], [(200, 80), (64, 64), (40, 1)]])
def test_prefill_attention_with_prefix(dev, lens):
    """Extended kernel: q rows are the LAST Lq positions of an Lk-token KV
    (prefix caching / chunked prefill)."""
    QH, KVH, D = 32, 8, 128
    Tk = sum(lk for lk, _ in lens)
    Tq = sum(lq for _, lq in lens)
    k = torch.randn(Tk, KVH, D, dtype=torch.bfloat16, device=dev)
    v = torch.randn(Tk, KVH, D, dtype=torch.bfloat16, device=dev)
    q = torch.randn(Tq, QH, D, dtype=torch.bfloat16, device=dev)
    cu_q = [0]
    cu_k = [0]
    for lk, lq in lens:
        cu_q.append(cu_q[-1] + lq)
        cu_k.append(cu_k[-1] + lk)
    cu_q = torch.tensor(cu_q, dtype=torch.int32, device=dev)
    cu_k = torch.tensor(cu_k, dtype=torch.int32, device=dev)
    scale = 1.0 / math.sqrt(D)
    got = ops.prefill_attention(q, k, v, cu_q, scale, cu_k)
    want = ref.prefill_attention(q, k, v, cu_q, scale, cu_k)
    err = (got.float() - want.float()).abs().max().item()
    assert err < 3e-2, f"lens={lens} err={err}"


@pytest.mark.gpu
def test_skinny_gemm_matches_fp32():
    """skinny_gemm vs fp32 matmul on every decode projection shape of
    llama-3-8b plus edge batches (M=1, 7, 33, 128) and all split picks."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    H, I, QH, KVH, D = 4096, 14336, 32, 8, 128
    shapes = [(H, (QH + 2 * KVH) * D), (QH * D, H), (H, 2 * I), (I, H)]
    torch.manual_seed(7)
    for M in (1, 7, 33, 64, 128, 192, 256):
        for (k, n) in shapes:
            x = torch.randn(M, k, dtype=torch.bfloat16, device=dev) * 0.5
            w = torch.randn(n, k, dtype=torch.bfloat16, device=dev) * 0.05
            got = ops._hip.skinny_gemm(x, w).float()
            ref = x.float() @ w.float().t()
            # bf16 inputs, f32 accumulate: error comes from input rounding
            tol = ref.abs().max().item() * 3e-2 + 0.02
            assert (got - ref).abs().max().item() < tol, \
                (M, k, n, (got - ref).abs().max().item(), tol)


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [4, 5, 6])
def test_decode_attention_mfma_variant4(variant):
    """MFMA-tiled decode (variant 4, register-diet 5, producer/consumer
    6) vs fp32 reference, including ragged contexts, multiple splits,
    odd page tails."""
    import torch
    from rbg_amd import ops
    from rbg_amd.ops import reference
    dev = torch.device("cuda:0")
    torch.manual_seed(3)
    B, KVH, QH, D, page = 5, 8, 32, 128, 16
    ctxs = [1, 17, 33, 256, 2048]
    max_pages = (max(ctxs) + page - 1) // page
    npages = sum((c + page - 1) // page for c in ctxs) + 1
    kc = torch.randn(npages, KVH, page, D, dtype=torch.bfloat16, device=dev)
    vc = torch.randn_like(kc)
    bt = torch.zeros(B, max_pages, dtype=torch.int32, device=dev)
    nxt = 1
    for i, c in enumerate(ctxs):
        n = (c + page - 1) // page
        bt[i, :n] = torch.arange(nxt, nxt + n, dtype=torch.int32)
        nxt += n
    ctx = torch.tensor(ctxs, dtype=torch.int32, device=dev)
    q = torch.randn(B, QH, D, dtype=torch.bfloat16, device=dev)
    ref = reference.decode_attention(
        q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(), ctx.cpu(), 0.088).to(dev)
    for splits in (1, 2, 4):
        got = ops._hip.decode_attention(q, kc, vc, bt, ctx, 0.088, splits,
                                        variant)
        assert torch.allclose(got.float(), ref.float(), atol=2e-2,
                              rtol=2e-2), \
            (splits, (got.float() - ref.float()).abs().max().item())


@pytest.mark.gpu
def test_strided_qkv_slices_match_contiguous():
    """rope + both attention kernels accept fused-QKV slices (wide row
    stride): results must equal the contiguous-copy path exactly."""
    import torch
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    torch.manual_seed(11)
    T, QH, KVH, D, page = 32, 32, 8, 128, 16
    width = (QH + 2 * KVH) * D
    kv_pages = 16
    for mode in ("prefill", "decode"):
        qkv = torch.randn(T, width, dtype=torch.bfloat16, device=dev)
        qkv2 = qkv.clone()
        kc1 = torch.zeros(kv_pages, KVH, page, D, dtype=torch.bfloat16,
                          device=dev)
        vc1 = torch.zeros_like(kc1)
        kc2, vc2 = kc1.clone(), vc1.clone()
        cs = ops.build_cos_sin_table(D, 4096, 5e5, device=dev)
        pos = torch.arange(T, dtype=torch.int32, device=dev)
        slots = torch.arange(16, 16 + T, dtype=torch.int32, device=dev)
        # strided path
        q = qkv[:, :QH * D]
        k = qkv[:, QH * D:(QH + KVH) * D]
        v = qkv[:, (QH + KVH) * D:]
        ops._hip.rope_store_kv(q, k, v, kc1, vc1, cs, pos, slots)
        # contiguous path
        q2 = qkv2[:, :QH * D].contiguous()
        k2 = qkv2[:, QH * D:(QH + KVH) * D].contiguous()
        v2 = qkv2[:, (QH + KVH) * D:].contiguous()
        ops._hip.rope_store_kv(q2, k2, v2, kc2, vc2, cs, pos, slots)
        assert torch.equal(kc1, kc2) and torch.equal(vc1, vc2)
        assert torch.equal(q.contiguous(), q2)
        if mode == "prefill":
            from rbg_amd.ops import reference
            cu = torch.tensor([0, T], dtype=torch.int32)
            bi, sl = reference.prefill_block_info(cu, qtile=128)
            o1 = ops._hip.prefill_attention(
                q.view(T, QH, D), k.view(T, KVH, D), v.view(T, KVH, D),
                bi.to(dev), sl.to(dev), 0.088, 6)
            o2 = ops._hip.prefill_attention(
                q2.view(T, QH, D), k2.view(T, KVH, D), v2.view(T, KVH, D),
                bi.to(dev), sl.to(dev), 0.088, 6)
            assert torch.equal(o1, o2)
        else:
            bt = torch.arange(1, 3, dtype=torch.int32,
                              device=dev).repeat(T, 1)
            bt = torch.arange(1, 1 + 2, dtype=torch.int32,
                              device=dev).unsqueeze(0).repeat(T, 1)
            ctx = torch.full((T,), 2, dtype=torch.int32, device=dev)
            o1 = ops._hip.decode_attention(q.view(T, QH, D), kc1, vc1, bt,
                                           ctx, 0.088, 1, 4)
            o2 = ops._hip.decode_attention(q2.view(T, QH, D), kc2, vc2, bt,
                                           ctx, 0.088, 1, 4)
            assert torch.equal(o1, o2)


@pytest.mark.gpu
def test_xgmi_allreduce_pair_protocol():
    """Full one-shot all-reduce protocol on ONE device: two in-process
    'ranks' launched on separate streams spin-satisfy each other's start/
    end flags; results must equal the elementwise sum.  Repeated calls
    prove the epoch counters advance (the graph-replay property)."""
    import torch

    from rbg_amd import ops
    from rbg_amd.parallel.xgmi_allreduce import XgmiAllReduce
    dev = torch.device("cuda", 0)
    a, b = XgmiAllReduce.for_test_pair(dev)
    torch.manual_seed(11)
    sa = torch.cuda.Stream(dev)
    sb = torch.cuda.Stream(dev)
    for round_ in range(3):
        xa = torch.randn(1024, 512, dtype=torch.bfloat16, device=dev)
        xb = torch.randn(1024, 512, dtype=torch.bfloat16, device=dev)
        torch.cuda.synchronize()
        with torch.cuda.stream(sa):
            oa = a.all_reduce(xa)
        with torch.cuda.stream(sb):
            ob = b.all_reduce(xb)
        torch.cuda.synchronize()
        a.check()
        b.check()
        want = (xa.float() + xb.float()).bfloat16()
        assert torch.equal(oa, want), round_
        assert torch.equal(ob, want), round_


@pytest.mark.gpu
def test_xgmi_allreduce_graph_capture():
    """Both ranks capture their all-reduce into hipGraphs and 3 replays
    with changing inputs produce exact sums (epochs advance in device
    memory).  Runs tools/xgmi_graph_debug.py in a FRESH subprocess: the
    protocol is order-sensitive to unrelated prior GPU state in the same
    process (pair-test-then-capture interleaving flaked), and production
    TP engines are fresh processes."""
    import subprocess
    import sys
    out = subprocess.run(
        [sys.executable, os.path.join(ROOT, "tools", "xgmi_graph_debug.py")],
        capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout[-2000:] + out.stderr[-2000:]
    for round_ in range(3):
        want = float(round_ + 1) + 10 * (round_ + 1)
        assert f"want {want}" in out.stdout
        assert f"oa uniq [{want}] ob uniq [{want}]" in out.stdout,             out.stdout[-1500:]
    assert "err=0" in out.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("swz", [8, 9, 10])
@pytest.mark.parametrize("lens", [[128], [64, 200, 1], [1024], [33, 129]])
def test_prefill_attention_32x32(dev, lens, swz, monkeypatch):
    """32x32x16 MFMA prefill (swz bit 3; 9 = +XCD swizzle, 10 = +DB) vs
    fp32 reference across ragged/causal shapes."""
    monkeypatch.setattr(ops, "PREFILL_SWZ", swz)
    QH, KVH, D = 32, 8, 128
    T = sum(lens)
    torch.manual_seed(5)
    q = torch.randn(T, QH, D, dtype=torch.bfloat16, device=dev)
    k = torch.randn(T, KVH, D, dtype=torch.bfloat16, device=dev)
    v = torch.randn(T, KVH, D, dtype=torch.bfloat16, device=dev)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)),
                      dtype=torch.int32, device=dev)
    scale = 1.0 / math.sqrt(D)
    got = ops.prefill_attention(q, k, v, cu, scale)
    want = ref.prefill_attention(q, k, v, cu, scale)
    err = (got.float() - want.float()).abs().max().item()
    assert err < 3e-2, f"swz={swz} lens={lens} err={err}"


@pytest.mark.gpu
@pytest.mark.parametrize("swz", [8])
def test_prefill_attention_32x32_with_prefix(dev, swz, monkeypatch):
    """Chunked-prefill path (q_offset > 0) on the 32x32 kernel."""
    monkeypatch.setattr(ops, "PREFILL_SWZ", swz)
    QH, KVH, D = 32, 8, 128
    torch.manual_seed(6)
    past, new = 192, 160
    kv_total = past + new
    q = torch.randn(new, QH, D, dtype=torch.bfloat16, device=dev)
    k = torch.randn(kv_total, KVH, D, dtype=torch.bfloat16, device=dev)
    v = torch.randn(kv_total, KVH, D, dtype=torch.bfloat16, device=dev)
    cu_q = torch.tensor([0, new], dtype=torch.int32, device=dev)
    cu_k = torch.tensor([0, kv_total], dtype=torch.int32, device=dev)
    scale = 1.0 / math.sqrt(D)
    got = ops.prefill_attention(q, k, v, cu_q, scale, cu_k)
    want = ref.prefill_attention(q, k, v, cu_q, scale, cu_k)
    err = (got.float() - want.float()).abs().max().item()
    assert err < 3e-2, err


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 4, 5, 16, 17, 32, 33, 48, 49, 65, 97, 129,
                               193, 256])
@pytest.mark.parametrize("n,k", [(32, 256), (160, 768), (8224, 512),
                                 (2048, 5632), (1312, 2048), (33024, 256)])
def test_skinny_gemm_edges(m, n, k):
    """Row tiles of every kernel, columns that leave waves idle, splits of
    unequal length, fewer chunks of k than are in flight.  f32 sums of bf16
    products, rounded once: half an ulp of the result (2^-9) and k roundings
    of 2^-24 of the sums of magnitudes."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(m * 1000003 + n + k)
    x = torch.randn(m, k, device=dev, generator=gen).bfloat16()
    w = torch.randn(n, k, device=dev, generator=gen).bfloat16()
    want = x.double() @ w.double().t().contiguous()
    bound = want.abs() * 2 ** -8 + \
        (x.double().abs() @ w.double().abs().t().contiguous()) * k * 2 ** -24
    got = ops._hip.skinny_gemm(x, w).double()
    assert ((got - want).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [0, 1, 128, 129])
@pytest.mark.parametrize("n,k", [(6144, 2048), (12320, 2048), (64, 96)])
def test_linear_any_shape(rows, n, k):
    """Both routes of linear, no rows at all among them."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    x = torch.randn(rows, k, device=dev).bfloat16()
    w = torch.randn(n, k, device=dev).bfloat16()
    got = ops.linear(x, w)
    want = x.float() @ w.float().t()
    assert got.shape == want.shape
    assert ((got.float() - want).abs() <= want.abs() * 2 ** -7 + 0.05).all()


@pytest.mark.gpu
@pytest.mark.parametrize("qpg,kvh,lens,splits", [
    (4, 8, [1, 15, 16, 17, 31, 32, 33, 127, 128, 129, 2080], 1),
    (1, 3, [1, 128, 129, 255, 257, 640], 5),
    (8, 2, [700, 1, 500, 384, 385], 4),
    (2, 1, [2048], 40),                     # more parts than steps
    (4, 3, [1 + 37 * i % 300 for i in range(97)], 3),   # XCD groups, a rest
    (4, 8, [2 + 29 * i % 200 for i in range(96)], 1),
])
def test_decode_pages(qpg, kvh, lens, splits):
    """Parts of the table's capacity: ends inside a page, a step and a part,
    empty parts, sequences of one part beside others of many; spread pages;
    values far outside the softmax's weights; capture.  Weights are rounded to
    bf16 (2^-9 of a weighted mean of |v|) and so is the result."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(len(lens) * 100 + splits)
    pages = [(n + 15) // 16 for n in lens]
    total = sum(pages) + 1
    kc = torch.randn(total, kvh, 16, 128, device=dev, generator=gen).bfloat16()
    vc = torch.randn(total, kvh, 16, 128, device=dev, generator=gen).bfloat16()
    perm = (torch.randperm(total - 1, device=dev, generator=gen) + 1).int()
    bt = torch.zeros(len(lens), max(pages) + 3, dtype=torch.int32, device=dev)
    at = 0
    for i, n in enumerate(pages):
        bt[i, :n] = perm[at:at + n]
        at += n
    cl = torch.tensor(lens, dtype=torch.int32, device=dev)
    fused = torch.randn(len(lens), (qpg + 2) * kvh * 128, device=dev,
                        generator=gen).bfloat16()
    q = fused[:, :qpg * kvh * 128].view(len(lens), qpg * kvh, 128)
    def call():
        return ops._hip.decode_attention(q, kc, vc, bt, cl, 0.4, splits, 7)
    got = call().double()
    for i, n in enumerate(lens):
        rows = [t[bt[i, :pages[i]].long()].transpose(0, 1).reshape(
            kvh, -1, 128)[:, :n].double() for t in (kc, vc)]
        for h in range(kvh):
            w = (q[i, h * qpg:(h + 1) * qpg].double() @
                 rows[0][h].t().contiguous() * 0.4).softmax(-1)
            want = w @ rows[1][h]
            bound = want.abs() * 2 ** -8 + (w @ rows[1][h].abs()) * 2 ** -7
            err = (got[i, h * qpg:(h + 1) * qpg] - want).abs()
            assert (err <= bound + 1e-5).all(), (i, n, h)
    g = torch.cuda.CUDAGraph()
    with torch.inference_mode(), torch.cuda.graph(g):
        out = call()
    for _ in range(3):
        with torch.inference_mode():
            out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.double(), got)


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [0, 1, 5, 16])
@pytest.mark.parametrize("rows,hidden", [(1, 4096), (7, 256), (3, 20),
                                         (130, 5120), (2, 16384)])
def test_add_rmsnorm_rows(parts, rows, hidden):
    """Both sources, rows that leave threads idle.  The residual is one
    rounding of the sum, the result another two (2^-8 each, generously)."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(rows * hidden + parts)
    def rnd(*shape):
        return torch.randn(*shape, device=dev, generator=gen)
    x = rnd(parts, rows, hidden) if parts else rnd(rows, hidden).bfloat16()
    res, w = rnd(rows, hidden).bfloat16(), rnd(hidden).bfloat16()
    total = (x.double().sum(0) if parts else x.double()) + res.double()
    want = total * torch.rsqrt(total.square().mean(-1, keepdim=True) + 1e-5) \
        * w.double()
    got = ops._hip.add_rmsnorm(x, res, w, 1e-5)
    assert ((res.double() - total).abs() <= total.abs() * 2 ** -8 +
            1e-5).all()
    assert ((got.double() - want).abs() <= want.abs() * 2 ** -7 + 1e-5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [0, 1, 6])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("tokens,heads,kvh", [(1, 2, 1), (5, 32, 8),
                                              (37, 6, 3), (87, 32, 8)])
def test_rope_heads(parts, norm, tokens, heads, kvh):
    """Head norms, rotation and store from bf16 rows (in place) and from the
    sums of a split GEMM, with a skipped slot; one rounding of the result."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(tokens * 100 + parts)
    def rnd(*shape):
        return torch.randn(*shape, device=dev, generator=gen)
    width, pages = (heads + 2 * kvh) * 128, max(4, tokens // 8)
    proj = (rnd(parts, tokens, width) if parts
            else rnd(tokens, width).bfloat16())
    x = (proj.double().sum(0) if parts else proj.double()).view(
        tokens, heads + 2 * kvh, 128)
    norms = [rnd(128).bfloat16() for _ in range(2)] if norm else [None, None]
    table = ref.build_cos_sin_table(128, 512, device=dev)
    pos = torch.randint(0, 512, (tokens,), device=dev, generator=gen).int()
    slots = torch.randperm(pages * 16, device=dev,
                           generator=gen)[:tokens].int()
    if tokens > 1:
        slots[1] = -1
    kc = torch.zeros(pages, kvh, 16, 128, dtype=torch.bfloat16, device=dev)
    vc = torch.zeros_like(kc)
    want = x.clone()
    for part, w in zip((want[:, :heads], want[:, heads:heads + kvh]), norms):
        if norm:
            part *= torch.rsqrt(part.square().mean(-1, keepdim=True) +
                                1e-6) * w.double()
        cs = table[pos.long()].double()[:, None]
        a, b = part[..., :64].clone(), part[..., 64:].clone()
        part[..., :64] = a * cs[..., :64] - b * cs[..., 64:]
        part[..., 64:] = b * cs[..., :64] + a * cs[..., 64:]
    got = ops.rope_heads(proj, heads, *norms, 1e-6, kc, vc, table, pos, slots)
    assert got.dtype == torch.bfloat16
    bound = want.abs() * 2 ** -8 + 2e-5
    assert ((got.double().view_as(want) - want).abs() <= bound).all()
    for cache, at in ((kc, heads), (vc, heads + kvh)):
        held = torch.zeros_like(cache)
        for t, s in enumerate(slots.tolist()):
            if s >= 0:
                held[s // 16, :, s % 16] = got.view(
                    tokens, -1, 128)[t, at:at + kvh]
        assert torch.equal(cache, held)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 4, 5, 17, 33, 64, 65])
@pytest.mark.parametrize("f,k", [(32, 512), (36, 4096), (5632, 2048),
                                 (8224, 2048)])
def test_linear_swiglu(m, f, k):
    """Gate and up tiles of every kernel, columns that leave waves idle; error
    of the f32 sums through silu and one rounding (the separate kernels round
    gate and up as well)."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(m * 7 + f)
    x = torch.randn(m, k, device=dev, generator=gen).bfloat16()
    w = (torch.randn(2 * f, k, device=dev, generator=gen) / k ** 0.5
         ).bfloat16()
    full = x.double() @ w.double().t().contiguous()
    want = torch.nn.functional.silu(full[:, :f]) * full[:, f:]
    bound = 2 ** -7 * (full[:, :f].abs() + 1) * (full[:, f:].abs() + 1)
    if f % 32:
        with pytest.raises(RuntimeError):
            ops._hip.skinny_swiglu(x, w)
        w = torch.cat([w[:32], w[f:f + 32]])    # 1 to 16 parts
        full, f = torch.cat([full[:, :32], full[:, f:f + 32]], 1), 32
        want, bound = want[:, :32], bound[:, :32]
    for got in (ops._hip.skinny_swiglu(x, w), ops.linear_swiglu(x, w),
                ops.silu_mul(ops.linear_parts(x, w))):
        assert ((got.double() - want).abs() <= bound).all()
    got = ops._hip.skinny_swiglu(x, w).double()
    assert (got - want).norm() <= 2 ** -8 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kvh", [(4, 1), (8, 8), (6, 2), (16, 2),
                                       (32, 8), (5, 5)])
@pytest.mark.parametrize("news,pasts", [
    ([1], [0]), ([1, 63, 64, 65, 129], [0] * 5),
    ([31, 33, 1, 200], [1, 64, 500, 63]), ([300], [0])])
def test_prefill_flash(heads, kvh, news, pasts):
    """Ends of tiles, waves and blocks, pasts of any length, groups that do
    not divide 128, key heads in and out of step with the XCDs; rows beside
    pages, scale of either sign, scores large enough to move the maximum, and
    sums that a capture replays.  Weights are rounded to bf16 (2^-9 of a
    weighted mean of |v|) and so is the result."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(heads * 1000 + sum(news))
    cu = [0] + torch.tensor(news).cumsum(0).tolist()
    cu_k = [0] + (torch.tensor(news) + torch.tensor(pasts)).cumsum(0).tolist()
    q = torch.randn(cu[-1], heads, 128, device=dev, generator=gen).bfloat16()
    rows = torch.randn(cu_k[-1], 2 * kvh, 128, device=dev,
                       generator=gen).bfloat16()
    rows[::50] *= 4
    rows = rows.view(cu_k[-1], -1)
    k = rows[:, :kvh * 128].view(-1, kvh, 128)
    v = rows[:, kvh * 128:].view(-1, kvh, 128)
    n = cu_k[-1] // 32 + 1
    slots = torch.randperm(n * 32, device=dev, generator=gen)[:cu_k[-1]]
    pages = torch.zeros(2, n, kvh, 32, 128, dtype=torch.bfloat16, device=dev)
    pages[0, slots // 32, :, slots % 32] = k
    pages[1, slots // 32, :, slots % 32] = v
    cut = torch.tensor(cu, dtype=torch.int32, device=dev)
    cut_k = torch.tensor(cu_k, dtype=torch.int32, device=dev)
    for scale in (0.3, -0.09, 0.0):
        got = ops.prefill_attention(q, k, v, cut, scale, cut_k)
        for b, past in enumerate(pasts):
            kb, vb = (t[cu_k[b]:cu_k[b + 1]].double() for t in (k, v))
            at = past + torch.arange(news[b], device=dev)
            hide = torch.arange(len(kb), device=dev)[None] > at[:, None]
            for h in range(heads):
                g = h // (heads // kvh)
                qb = q[cu[b]:cu[b + 1], h].double()
                s = (qb @ kb[:, g].t().contiguous() * scale).masked_fill(
                    hide, -math.inf)
                w = s.softmax(-1)
                want = w @ vb[:, g]
                bound = want.abs() * 2 ** -8 + (w @ vb[:, g].abs()) * 2 ** -7
                err = (got[cu[b]:cu[b + 1], h].double() - want).abs()
                assert (err <= bound + 1e-5).all(), (scale, b, h)
        paged = ops.prefill_attention(q, pages[0], pages[1], cut, scale,
                                      cut_k, slots=slots.int())
        assert torch.equal(paged, got)
    plan = ops.prefill_plan(cu, cu_k, heads, kvh, dev)
    g = torch.cuda.CUDAGraph()
    with torch.inference_mode(), torch.cuda.graph(g):
        out = ops.prefill_attention(q, k, v, cut, 0.0, cut_k, plan)
    for _ in range(3):
        with torch.inference_mode():
            out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, got)


@pytest.mark.gpu
@pytest.mark.parametrize("kvh", [1, 8])
@pytest.mark.parametrize("rows,past", [(1, 62), (64, 64), (65, 63), (200, 1000),
                                       (3, 9000)])
def test_prefill_flash_pages_of_any_pool(kvh, rows, past):
    """Whole and ragged last tiles of rows, of pages in a pool whose offsets are 32
    bits and in one beyond 4 GB, at both ends of it: the same bits."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(rows + past + kvh)
    n = rows + past
    q = torch.randn(rows, 4 * kvh, 128, device=dev, generator=gen).bfloat16()
    k, v = (torch.randn(n, kvh, 128, device=dev, generator=gen).bfloat16()
            for _ in range(2))
    cut = torch.tensor([0, rows], dtype=torch.int32, device=dev)
    cut_k = torch.tensor([0, n], dtype=torch.int32, device=dev)
    want = ops.prefill_attention(q, k, v, cut, 0.1, cut_k)
    used = n // 16 + 1
    for pages in (used, 2 ** 24 // (16 * kvh), 2 ** 24 // (16 * kvh) + 1):
        # the sequence's pages from both ends, the others without numbers
        mine = torch.arange(used, device=dev)
        mine = torch.where(mine % 2 == 0, mine // 2, pages - 1 - mine // 2)
        at = torch.arange(n, device=dev)
        page, place = mine[at // 16], at % 16
        pool = [torch.empty(pages, kvh, 16, 128, dtype=torch.bfloat16,
                            device=dev) for _ in range(2)]
        for p, rows_of in zip(pool, (k, v)):
            p[page, :, place] = rows_of
        got = ops.prefill_attention(q, *pool, cut, 0.1, cut_k,
                                    slots=(page * 16 + place).int())
        assert torch.equal(got, want), pages
        del pool


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kvh", [(5, 1), (18, 2), (127, 1), (128, 1)])
@pytest.mark.parametrize("rows", [1, 32, 33, 70])
def test_prefill_flash_rows_of_q(heads, kvh, rows):
    """Query rows of any group, as slices of wider rows and off 16 bytes, against rows
    by themselves; and those against softmax in 64 bits."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(heads + rows)
    k, v = (torch.randn(rows, kvh, 128, device=dev, generator=gen).bfloat16()
            for _ in range(2))
    cut = torch.tensor([0, rows], dtype=torch.int32, device=dev)
    first = None
    for pad, begin in ((0, 0), (8, 8), (8, 4), (6, 2)):
        wide = torch.zeros(rows, heads * 128 + pad, device=dev,
                           dtype=torch.bfloat16)
        q = wide[:, begin:begin + heads * 128].view(rows, heads, 128)
        gen.manual_seed(rows)
        q.copy_(torch.randn(rows, heads, 128, device=dev, generator=gen))
        got = ops.prefill_attention(q, k, v, cut, 0.2)
        if first is None:
            first = got
        assert torch.equal(got, first), (pad, begin)
    hide = torch.ones(rows, rows, dtype=torch.bool, device=dev).triu(1)
    for h in range(heads):
        g = h // (heads // kvh)
        s = q[:, h].double() @ k[:, g].double().t().contiguous() * 0.2
        w = s.masked_fill(hide, -math.inf).softmax(-1)
        vb = v[:, g].double()
        bound = (w @ vb).abs() * 2 ** -8 + (w @ vb.abs()) * 2 ** -7
        assert ((first[:, h].double() - w @ vb).abs() <= bound + 1e-5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [33, 48, 49, 64])
@pytest.mark.parametrize("n,k", [(64, 512), (4160, 1024), (10240, 2048),
                                 (16384, 1536)])
def test_swiglu_of_small_workgroups(rows, n, k):
    """silu within the decode GEMM of 33 to 64 rows, and gates as large as make
    its exponential infinite or 0; an f32 sum of k products, silu and one
    rounding."""
    from rbg_amd import ops
    assert ops._glu(rows, n, k)
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(rows + n)
    x = torch.randn(rows, k, device=dev, generator=gen).bfloat16()
    w = (torch.randn(n, k, device=dev, generator=gen) / k ** 0.5).bfloat16()
    w[:8] *= 64
    full = x.double() @ w.double().t().contiguous()
    size = (x.double().abs() @ w.double().abs().t().contiguous()) * 2 ** -18
    gate, up = full.chunk(2, 1)
    want = torch.nn.functional.silu(gate) * up
    # silu grows by at most 1.1 of what its argument does
    bound = want.abs() * 2 ** -8 + 1.1 * size[:, :n // 2] * up.abs() + \
        size[:, n // 2:] * gate.abs() + 1e-6
    got = ops.linear_swiglu(x, w)
    assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("group", [1, 2, 4, 8])
@pytest.mark.parametrize("lens,splits", [
    ([1, 256, 257, 0, 513, 5000], 32), ([16000], 32), ([300], 2),
    ([2080] * 100, 4), ([2049, 2560, 2561, 2048] * 100, 4)])
def test_decode_attention_tickets(group, lens, splits):
    """Parts added up by a sequence's last workgroup as by a launch of its own:
    one part, two, more than a round of loads, longer ones than the least, and a
    longer single one where there are many; again and again with the same tickets
    and sums' memory, eagerly and replayed, with other queries, rows and order of
    lengths each time, so that sums of a former time would show.  The same f32 sums in another order: a rounding of the result
    apart, 2^-8 of it, or of the values' size where they cancel."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(group + len(lens))
    kvh, width = 2, (max(lens) + 15) // 16
    n = len(lens)
    q = torch.randn(n, kvh * group, 128, device=dev,
                    generator=gen).bfloat16()
    k, v = torch.randn(2, 1200, kvh, 16, 128, device=dev,
                       generator=gen).bfloat16()
    tables = torch.randint(0, 1200, (n, width), device=dev, generator=gen,
                           dtype=torch.int32)
    lens = torch.tensor(lens, dtype=torch.int32, device=dev)
    tickets = torch.zeros(n * kvh, dtype=torch.int32, device=dev)

    def run(t):
        return ops.decode_attention(q, k, v, tables, lens, 0.2,
                                    num_splits=splits, variant=7, tickets=t)

    def others():
        for t in (q, k, v):
            t.copy_(torch.randn(t.shape, device=dev, generator=gen))
        lens.copy_(lens[torch.randperm(n, device=dev, generator=gen)])

    def check(got):
        want = run(None).float()
        bound = want.abs() * 2 ** -7 + 2 ** -9
        assert ((got.float() - want).abs() <= bound).all()
        assert not tickets.any()
    for _ in range(3):
        got = run(tickets)
        check(got)
        others()
    g = torch.cuda.CUDAGraph()
    with torch.inference_mode(), torch.cuda.graph(g):
        out = run(tickets)
    for _ in range(4):
        others()
        with torch.inference_mode():
            out.zero_()
        g.replay()
        torch.cuda.synchronize()
        check(out)
        assert torch.equal(out, run(tickets))


@pytest.mark.gpu
@pytest.mark.parametrize("rows,width,seqs,used", [
    (1, 512, 1, 1), (4, 7, 3, 7), (128, 1024, 97, 131), (2, 512, 1, 512)])
def test_place_inputs(rows, width, seqs, used):
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    fields = torch.randint(0, 1 << 40, (4 * rows,), device=dev)
    tables = torch.randint(1, 1 << 30, (seqs, used), device=dev,
                           dtype=torch.int32)
    to_fields = torch.full_like(fields, -1)
    to_tables = torch.full((rows, width), -1, device=dev, dtype=torch.int32)
    ops.place_inputs(to_fields, to_tables, fields, tables)
    assert torch.equal(to_fields, fields)
    assert torch.equal(to_tables[:seqs, :used], tables)
    to_tables[:seqs, :used] = 0
    assert not to_tables.any()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,width,seqs,used", [
    (1, 512, 1, 1), (4, 7, 3, 7), (128, 1024, 97, 131), (2, 512, 1, 512)])
def test_place_host_inputs(rows, width, seqs, used):
    """Of arrays of the host, one after another without a wait, so that pinned memory
    is used again for other numbers; beside a stream that keeps the GPU busy."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(rows)
    to_fields = torch.full((4 * rows,), -1, device=dev)
    to_tables = torch.full((rows, width), -1, device=dev, dtype=torch.int32)
    busy = torch.ones(1 << 22, device=dev)
    kept = []
    for i in range(200):
        fields = rng.integers(0, 1 << 40, 4 * rows)
        tables = rng.integers(1, 1 << 30, (seqs, used), dtype=np.int32)
        if i % 7 == 0:
            busy.cos_()
        ops.place_host_inputs(to_fields, to_tables, fields, tables)
        kept.append((fields, tables, to_fields.clone(), to_tables.clone()))
        if i % 20 > 9:          # the memory is free again at once
            torch.cuda.synchronize()
    for fields, tables, got_fields, got_tables in kept:
        assert np.array_equal(got_fields.cpu().numpy(), fields)
        got = got_tables.cpu().numpy()
        assert np.array_equal(got[:seqs, :used], tables)
        got[:seqs, :used] = 0
        assert not got.any()
    with pytest.raises(RuntimeError):
        ops._hip.place_host_inputs(to_fields, to_tables, to_fields, to_tables)


@pytest.mark.gpu
@pytest.mark.parametrize("width,dtype", [(8, torch.bfloat16), (4096, torch.bfloat16),
                                         (4100, torch.bfloat16),
                                         (64, torch.float32)])
def test_rows_at(width, dtype):
    """Rows by the kernel, or by indexing where it does not take them; again and again
    from the same pinned memory; none, all, and from the end."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    x = torch.randn(300, width, device=dev).to(dtype)
    rng = np.random.default_rng(width)
    got = [(rows, ops.rows_at(x, rows)) for rows in
           [[], [0], [-1, 299, -300], list(range(300))] +
           [rng.integers(0, 300, 5).tolist() for _ in range(40)]]
    for rows, y in got:
        assert torch.equal(y, x[torch.tensor(rows, dtype=torch.int64, device=dev)])
    if width % 8 == 0 and dtype == torch.bfloat16:
        for row in (300, -301):
            with pytest.raises(IndexError):
                ops.rows_at(x, [row])


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,k", [
    (1, 32, 4096), (4, 2048, 4096), (3, 1024, 14336), (2, 2048, 5632),
    (1, 5120, 8192), (1, 6144, 8704), (1, 4128, 14336), (5, 2048, 2048),
    (64, 32768, 2048), (128, 1024, 4096)])
def test_rows_of_pairs_and_f32(rows, n, k):
    """Forms whose tiles take two chunks of k at a time, at the ends of the rule
    for them, and results in f32, which are the rounded ones: 2^-8 of each, and
    f32 sums of k products."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(rows + n + k)
    x = torch.randn(rows, k, device=dev, generator=gen).bfloat16()
    w = torch.randn(n, k, device=dev, generator=gen).bfloat16()
    want = x.double() @ w.double().t().contiguous()
    size = x.double().abs() @ w.double().abs().t().contiguous()
    got = ops._hip.skinny_gemm(x, w)
    assert ((got.double() - want).abs() <=
            want.abs() * 2 ** -8 + size * 2 ** -18).all()
    wide = ops._hip.skinny_gemm(x, w, wide=True)
    assert wide.dtype == torch.float32 and torch.equal(wide, got.float())
    assert torch.equal(ops.linear_f32(x, w), ops.linear(x, w).float())


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kvh", [(4, 1), (6, 2), (32, 8)])
@pytest.mark.parametrize("news,pasts", [
    ([1], [2500]), ([70, 1, 300], [2500, 0, 0]), ([129], [1900])])
def test_prefill_flash_cut(heads, kvh, news, pasts):
    """Blocks cut by keys, beside whole ones: parts that end anywhere in a
    sequence and on its diagonal, scores that move the maximum from part to
    part, sums that a capture replays.  Bounds as in test_prefill_flash."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(heads * 1000 + sum(news))
    cu = [0] + torch.tensor(news).cumsum(0).tolist()
    cu_k = [0] + (torch.tensor(news) + torch.tensor(pasts)).cumsum(0).tolist()
    q = torch.randn(cu[-1], heads, 128, device=dev, generator=gen).bfloat16()
    k, v = torch.randn(2, cu_k[-1], kvh, 128, device=dev,
                       generator=gen).bfloat16()
    k[::333] *= 4
    n = cu_k[-1] // 16 + 1
    slots = torch.randperm(n * 16, device=dev, generator=gen)[:cu_k[-1]]
    pages = torch.zeros(2, n, kvh, 16, 128, dtype=torch.bfloat16, device=dev)
    pages[0, slots // 16, :, slots % 16] = k
    pages[1, slots // 16, :, slots % 16] = v
    plan = ops.prefill_plan(cu, cu_k, heads, kvh, dev)
    assert plan.items is not None
    for scale in (0.3, -0.09):
        got = ops.prefill_attention(q, k, v, None, scale, plan=plan)
        for b, past in enumerate(pasts):
            kb, vb = (t[cu_k[b]:cu_k[b + 1]].double() for t in (k, v))
            at = past + torch.arange(news[b], device=dev)
            hide = torch.arange(len(kb), device=dev)[None] > at[:, None]
            for h in range(heads):
                g = h // (heads // kvh)
                s = q[cu[b]:cu[b + 1], h].double() @ kb[:, g].t().contiguous()
                w = (s * scale).masked_fill(hide, -math.inf).softmax(-1)
                want = w @ vb[:, g]
                bound = want.abs() * 2 ** -8 + (w @ vb[:, g].abs()) * 2 ** -7
                err = (got[cu[b]:cu[b + 1], h].double() - want).abs()
                assert (err <= bound + 1e-5).all(), (scale, b, h)
        paged = ops.prefill_attention(q, pages[0], pages[1], None, scale,
                                      plan=plan, slots=slots.int())
        assert torch.equal(paged, got)
    g = torch.cuda.CUDAGraph()
    with torch.inference_mode(), torch.cuda.graph(g):
        out = ops.prefill_attention(q, k, v, None, -0.09, plan=plan)
    for _ in range(3):
        with torch.inference_mode():
            out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, got)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 3, 4])
@pytest.mark.parametrize("k", [2048, 8192])
@pytest.mark.parametrize("first", [False, True])
def test_norm_rows(rows, k, first):
    """Norm, GEMM and each of its ends in one launch against float64.  The
    operand is rounded once, as the separate norm rounds it: 2^-8 of the sums'
    size, which for rows of a norm is the root of k times the weights'."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(rows * 10 + k)
    def rnd(*shape):
        return torch.randn(*shape, device=dev, generator=gen).bfloat16()
    heads, kvh = 4, 2
    src = None if first else rnd(rows, k)
    res, nw = rnd(rows, k) * 3, rnd(k)
    w = (torch.randn(1024, k, device=dev, generator=gen) / k ** 0.5).bfloat16()
    total = res.double() + (0 if first else src.double())
    h = total * torch.rsqrt(total.square().mean(-1, keepdim=True) + 1e-5) * \
        nw.double()
    full = h @ w.double().t().contiguous()
    for end, want in ((0, full), (1, torch.nn.functional.silu(full[:, :512]) *
                                  full[:, 512:])):
        old = res.clone()
        out, new = ops._hip.norm_rows(src, res, nw, 1e-5, w, end)
        assert torch.equal(res, old)
        assert ((new.double() - total).abs() <= total.abs() * 2 ** -8).all()
        assert (out.double() - want).norm() <= 2 ** -7 * want.norm(), end
    table = ref.build_cos_sin_table(128, 512, device=dev)
    pos = torch.randint(0, 512, (rows,), device=dev, generator=gen).int()
    slots = torch.randperm(32, device=dev, generator=gen)[:rows].int()
    slots[-1] = -1
    caches = [torch.zeros(2, kvh, 16, 128, dtype=torch.bfloat16, device=dev)
              for _ in range(4)]
    for norms in ((None, None), (rnd(128), rnd(128))):
        got, _ = ops.norm_heads(src, res.clone(), nw, 1e-5, w, heads, *norms,
                                *caches[:2], table, pos, slots)
        want = ops.rope_heads(full.float()[None], heads, *norms, 1e-5,
                              *caches[2:], table, pos, slots)
        assert (got.double() - want.double()).norm() <= \
            2 ** -6.5 * want.double().norm()
        for a, b in zip(caches[:2], caches[2:]):
            assert ((a != 0) == (b != 0)).all()
            held = got.view(rows, -1, 128)
        for t, s in enumerate(slots.tolist()):
            if s >= 0:
                assert torch.equal(caches[0][s // 16, :, s % 16],
                                   held[t, heads:heads + kvh])
                assert torch.equal(caches[1][s // 16, :, s % 16],
                                   held[t, heads + kvh:])


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 2, 3, 4])
@pytest.mark.parametrize("n", [1024, 1056, 3104, 16416])
@pytest.mark.parametrize("k", [1024, 1280, 2304, 3072, 4096, 5120, 5376, 8192,
                               16640])
def test_stream_rows(rows, n, k):
    """Products of up to four rows against float64: waves with and without a last
    segment, workgroups with and without a last group, long rows, 512 k at a time and
    256; plain, in f32, after a norm and with silu.  Bounds as in test_norm_rows; plain
    ones half a unit of bf16's last place, 2^-8 of a value, and of f32 sums 1e-4, the
    root of k units of 2^-24 of values of 1 and what is rounded on the way.  After a norm
    every value too: a row is rounded twice, by up to 2^-9 of a value each, evenly, which
    makes sqrt(2/3) 2^-9 of a term and of the root of the terms' squares; eight times
    that, and the result's own rounding.  silu changes a gate's error by 1.1 at most."""
    from rbg_amd import ops
    if n * k > 3e7 and rows != 3:
        pytest.skip("large once")
    assert ops._stream(rows, n, k)
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(rows * 100000 + n + k)
    def rnd(*shape):
        return torch.randn(*shape, device=dev, generator=gen).bfloat16()
    x, w = rnd(rows, k), (rnd(n, k).float() / k ** 0.5).bfloat16()
    w[n - 1, k - 1] = math.inf              # in the last piece, that others repeat
    x[0, k - 1] = 1.0
    want = x.double() @ w.double().t().contiguous()
    got = ops.linear(x, w)
    assert got[0, n - 1] == math.inf
    err = (got.double() - want)[:, :n - 1].abs()
    assert (err <= want[:, :n - 1].abs() * 2 ** -8 + 1e-4).all()
    sums = ops._hip.stream_linear(x, w, 2)
    assert sums.shape == (1, rows, n) and sums.dtype == torch.float32
    parts = ops.linear_parts(x, w)
    assert torch.equal(parts, got if parts.dim() == 2 else sums)
    assert ((sums[0].double() - want)[:, :n - 1].abs() <= 1e-4).all()
    assert torch.equal(sums[0].bfloat16(), got)
    assert torch.equal(ops.linear_f32(x, w), got.float())
    if k > 8192:
        return
    w[n - 1, k - 1] = 1.0
    res, nw = rnd(rows, k) * 3, rnd(k)
    for src in (x, torch.randn(1, rows, k, device=dev, generator=gen), None):
        total = res.double() + (0 if src is None else src.double().view(rows, k))
        h = total * torch.rsqrt(total.square().mean(-1, keepdim=True) + 1e-5) * \
            nw.double()
        full = h @ w.double().t().contiguous()
        old = res.clone()
        assert ops._takes_rows(src, res, nw, w)
        out, new = ops._norm_project(src, res, nw, 1e-5, w)
        assert out.shape == (1, rows, n) and torch.equal(res, old)
        assert torch.equal(out[0].bfloat16(),
                           ops._hip.norm_rows(src, res, nw, 1e-5, w, 0)[0])
        assert ((new.double() - total).abs() <= total.abs() * 2 ** -8).all()
        assert (out.double() - full).norm() <= 2 ** -7 * full.norm()
        off = 8 * 2 ** -9 * (2 / 3) ** 0.5 * (
            h.square() @ w.double().square().t().contiguous()).sqrt()
        assert ((out.double() - full).abs() <= off + 1e-4).all()
        gate, up = full[:, :n // 2], full[:, n // 2:]
        want = torch.nn.functional.silu(gate) * up
        out, new2 = ops.norm_swiglu(src, res, nw, 1e-5, w)
        assert torch.equal(new2, new)
        assert (out.double() - want).norm() <= 2 ** -7 * want.norm()
        at_gate, at_up = off[:, :n // 2], off[:, n // 2:]
        bound = 1.1 * at_gate * (up.abs() + at_up) + gate.abs() * at_up
        assert ((out.double() - want).abs()
                <= bound + want.abs() * 2 ** -8 + 1e-4).all()


@pytest.mark.gpu
def test_linear_takes_what_the_library_takes():
    """Transposed and misaligned operands and gradients, at a shape that the
    decode GEMM would take otherwise."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    x = torch.randn(8, 1024, device=dev).bfloat16()
    w = torch.randn(1024, 256, device=dev).bfloat16()
    want = x.float() @ w.float()
    def near(got):
        return ((got.float() - want).abs() <=
                want.abs() * 2 ** -7 + 0.05).all()
    assert near(ops.linear(x, w.t()))
    odd = torch.empty(8 * 1024 + 1, device=dev, dtype=torch.bfloat16)[1:]
    odd.copy_(x.flatten())
    wt = w.t().contiguous()
    assert near(ops.linear(odd.view(8, 1024), wt))
    x.requires_grad_(True)
    got = ops.linear(x, wt)
    got.float().sum().backward()
    assert near(got) and x.grad is not None


def _paged(dev, lens, kvh, capacity, page=16, seed=0):
    """Keys, values, tables of that many keys, lengths; pages in no order."""
    gen = torch.Generator(device=dev).manual_seed(seed + len(lens))
    pages = [(n + page - 1) // page for n in lens]
    total = sum(pages) + 1
    kv = torch.randn(2, total, kvh, page, 128, device=dev,
                     generator=gen).bfloat16()
    perm = (torch.randperm(total - 1, device=dev, generator=gen) + 1).int()
    tables = torch.zeros(len(lens), capacity // page, dtype=torch.int32,
                         device=dev)
    at = 0
    for i, n in enumerate(pages):
        tables[i, :n] = perm[at:at + n]
        at += n
    return kv[0], kv[1], tables, torch.tensor(lens, dtype=torch.int32,
                                              device=dev)


def _near_decode(got, q, kc, vc, tables, lens, scale):
    """Weights are rounded to bf16 (2^-9 of a weighted mean of |v|) and so is
    the result."""
    qpg, kvh, page = q.shape[1] // kc.shape[1], kc.shape[1], kc.shape[2]
    for i, n in enumerate(lens.tolist()):
        at = tables[i, :(n + page - 1) // page].long()
        k, v = (t[at].transpose(0, 1).reshape(kvh, -1, 128)[:, :n].double()
                for t in (kc, vc))
        qi = q[i].view(kvh, qpg, 128).double()
        w = torch.stack([qi[h] @ k[h].t().contiguous() * scale
                         for h in range(kvh)]).softmax(-1)
        want = torch.stack([w[h] @ v[h] for h in range(kvh)]).view(-1, 128)
        most = torch.stack([w[h] @ v[h].abs()
                            for h in range(kvh)]).view(-1, 128)
        err = (got[i].double() - want).abs()
        assert (err <= want.abs() * 2 ** -8 + most * 2 ** -7 + 1e-5).all(), i


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [
    [2048], [2900 - 390 * i for i in range(7)],
    [2500 - 40 * i for i in range(45)]])
def test_decode_parts_follow_the_lengths(lens):
    """The same parts, and so the same bits, whatever a table could hold."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    q = torch.randn(len(lens), 32, 128, device=dev).bfloat16()
    outs = []
    for capacity in (8192, 40960, 131072):
        kv = _paged(dev, lens, 8, capacity)
        outs.append(ops.decode_attention(
            q, *kv, 0.1, ops.pick_decode_splits(len(lens), 8, capacity)))
    _near_decode(outs[0], q, *kv, 0.1)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.gpu
@pytest.mark.parametrize("splits,span", [(1, 256), (4, 256), (4, 100),
                                         (12, 128)])
def test_decode_part_lengths(splits, span):
    """Lengths about the end of a part, and beyond what the grid holds of the
    least parts, whose parts grow."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    lens = [1, 255, 256, 257, 512, 1023, 1024, 1025, 1536, 1537, 2100]
    q = torch.randn(len(lens), 8, 128, device=dev).bfloat16()
    kv = _paged(dev, lens, 2, 4096)
    got = ops._hip.decode_attention(q, *kv, 0.3, splits, 7, span)
    _near_decode(got, q, *kv, 0.3)


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [4, 7])
@pytest.mark.parametrize("page", [8, 16, 32, 64])
@pytest.mark.parametrize("splits", [1, 2, 8, 9, 31])
def test_decode_parts_of_any_page(variant, page, splits):
    """Forms whose every part leaves sums, empty ones too: one share and four,
    more than a round of eight each."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    lens = [1, 17, 300, 497, 1000]
    q = torch.randn(len(lens), 8, 128, device=dev).bfloat16()
    kv = _paged(dev, lens, 2, 2048, page)
    got = ops.decode_attention(q, *kv, 0.2, splits, variant)
    _near_decode(got, q, *kv, 0.2)
    _near_decode(ops.decode_attention(q, *kv, 0.2), q, *kv, 0.2)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kvh,parts,norms", [
    (8, 8, 0, False), (4, 2, 1, True), (32, 8, 5, False), (32, 8, 9, True),
    (64, 8, 8, True), (16, 2, 13, False)])
@pytest.mark.parametrize("splits,span,many", [(1, 256, 1), (5, 256, 1),
                                              (17, 128, 1), (4, 512, 10)])
def test_decode_takes_raw_heads(heads, kvh, parts, norms, splits, span, many):
    """The rotation, the store and the attention in one launch as in two: new keys
    in the first step of a wave and behind it, first, last and only ones of a part,
    in a row that held no numbers; rows that are not stored, or elsewhere; no keys."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    lens = [1, 2, 17, 32, 33, 128, 129, 160, 255, 256, 257, 513, 2048, 2100, 700,
            701, 5] * many
    kc, vc, tables, ctx = _paged(dev, lens, kvh, 4096)
    n, width = len(lens), (heads + 2 * kvh) * 128
    at = (ctx - 1).long()
    slots = (tables.gather(1, at[:, None] // 16)[:, 0] * 16 + at % 16).int()
    for c in (kc, vc):
        c[slots.long() // 16, :, slots.long() % 16] = math.nan
    kc[slots[14] // 16, :, slots[14] % 16] = 0.5    # not stored: the old row counts
    vc[slots[14] // 16, :, slots[14] % 16] = 0.25
    slots[14] = -1
    ctx[16] = 0                                     # stored, not read
    gen = torch.Generator(device=dev).manual_seed(7)
    proj = torch.randn(max(1, parts), n, width, device=dev, generator=gen)
    if parts == 0:
        proj = proj[0].bfloat16()
    pos = torch.randint(0, 4096, (n,), device=dev, generator=gen).int()
    table = ops.build_cos_sin_table(128, 4096, 10000.0, device=dev)
    nw = [torch.randn(128, device=dev, generator=gen).bfloat16()
          if norms else None for _ in range(2)]
    other = [kc.clone(), vc.clone()]
    qkv = ops.rope_heads(proj.clone(), heads, *nw, 1e-6, *other, table, pos, slots)
    q = qkv[:, :heads * 128].view(n, heads, 128)
    want = ops._hip.decode_attention(q, *other, tables, ctx, 0.09, splits, 7, span)
    tickets = torch.zeros(n * kvh, dtype=torch.int32, device=dev)
    for t in (None, tickets):
        mine = [kc.clone(), vc.clone()]
        # with tickets: lengths and tables of a batch that has more rows
        more = [] if t is None else [tables[:1], ctx[:1]]
        got = ops._hip.decode_heads(proj, heads, *nw, 1e-6, *mine, table, pos,
                                    slots, torch.cat([tables, *more[:1]]),
                                    torch.cat([ctx, *more[1:]]), 0.09, splits, span,
                                    t)
        assert not tickets.any()
        for a, b in zip(mine, other):
            # the last bit of a value, for another order of a norm's sum
            err = (a.float() - b.float()).abs()
            assert (err.nan_to_num() <= b.float().abs().nan_to_num() * 2 ** -7
                    ).all() and torch.equal(a.isnan(), b.isnan())
        assert got.isfinite().all()
        err = (got.float() - want.float()).norm() / want.float().norm()
        assert err <= 2 ** -8       # of queries' and keys' last bits


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [1, 4, 12])
@pytest.mark.parametrize("bad", [math.nan, math.inf])
def test_decode_shows_broken_rows(splits, bad):
    """A query or key that is no number leaves no plausible zeros, and stays
    in its row; a sequence without keys is zeros."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    q = torch.randn(4, 8, 128, device=dev).bfloat16()
    kc, vc, tables, lens = _paged(dev, [900, 900, 900, 1], 2, 1024)
    q[1, 5, 7] = bad
    kc[tables[2, 3], 0, 5, 0] = math.nan
    lens[3] = 0
    got = ops._hip.decode_attention(q, kc, vc, tables, lens, 0.1, splits, 7)
    assert got[1, 5].isnan().all() and got[2, :4].isnan().all()
    assert (got[3] == 0).all()
    rest = got.clone()
    rest[1, 5] = rest[2, :4] = 0
    assert rest.isfinite().all()


@pytest.mark.gpu
@pytest.mark.parametrize("k", [32768, 34816])
def test_norm_swiglu_widest_row(k):
    """The widest row that the one launch holds, and one that it does not."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(k)
    def rnd(*shape):
        return torch.randn(*shape, device=dev, generator=gen)
    x, res, nw = rnd(1, k).bfloat16(), rnd(1, k).bfloat16(), rnd(k).bfloat16()
    w = (rnd(64, k) / k ** 0.5).bfloat16()
    total = x.double() + res.double()
    h = total * torch.rsqrt(total.square().mean() + 1e-5) * nw.double()
    full = h @ w.double().t().contiguous()
    want = torch.nn.functional.silu(full[:, :32]) * full[:, 32:]
    for src in (x, None):
        got, new = ops.norm_swiglu(src, res.clone(), nw, 1e-5, w)
        if src is not None:
            assert (got.double() - want).norm() <= 2 ** -7 * want.norm()
            assert (new.double() - total).norm() <= 2 ** -8 * total.norm()
        else:
            assert torch.equal(new, res) and got.isfinite().all()


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kvh", [(4, 1), (32, 8), (6, 2)])
def test_prefill_fewer_keys_than_queries(heads, kvh):
    """Queries before the first key are zeros; no keys at all, first, between
    and last; rows beside pages."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    news, lens = [70, 200, 33, 130, 40], [0, 100, 40, 1, 0]
    cu = [0] + torch.tensor(news).cumsum(0).tolist()
    cu_k = [0] + torch.tensor(lens).cumsum(0).tolist()
    q = torch.randn(cu[-1], heads, 128, device=dev).bfloat16()
    k, v = torch.randn(2, cu_k[-1], kvh, 128, device=dev).bfloat16()
    slots = torch.randperm(160, device=dev)[:cu_k[-1]]
    pages = torch.zeros(2, 10, kvh, 16, 128, dtype=torch.bfloat16, device=dev)
    pages[0, slots // 16, :, slots % 16] = k
    pages[1, slots // 16, :, slots % 16] = v
    cut = torch.tensor(cu, dtype=torch.int32, device=dev)
    cut_k = torch.tensor(cu_k, dtype=torch.int32, device=dev)
    got = ops.prefill_attention(q, k, v, cut, 0.2, cut_k)
    assert torch.equal(got, ops.prefill_attention(
        q, pages[0], pages[1], cut, 0.2, cut_k, slots=slots.int()))
    for b, (new, n) in enumerate(zip(news, lens)):
        rows = got[cu[b]:cu[b + 1]]
        behind = max(0, new - n)
        assert (rows[:behind] == 0).all()
        if behind == new:
            continue
        at = torch.tensor([0, new - behind], dtype=torch.int32, device=dev)
        at_k = torch.tensor([0, n], dtype=torch.int32, device=dev)
        kb, vb = (t[cu_k[b]:cu_k[b + 1]] for t in (k, v))
        want = ref.prefill_attention(q[cu[b] + behind:cu[b + 1]].float(),
                                     kb.float(), vb.float(), at, 0.2, at_k)
        # bf16 weights and result, values of unit variance
        assert (rows[behind:].float() - want).abs().max() < 3e-2


@pytest.mark.gpu
@pytest.mark.parametrize("dim,shift", [(64, 0), (128, 1), (128, 4), (256, 0)])
@pytest.mark.parametrize("tokens", [1, 37])
def test_rope_store_kv_any_rows(dim, shift, tokens):
    """Head sizes and rows that the kernel of heads of 128 does not take: others
    than 128, and queries and keys that begin between multiples of 16 bytes."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    heads, kvh = 6, 2
    gen = torch.Generator(device=dev).manual_seed(dim + tokens)
    q, k = (torch.randn(tokens, h * dim + 8, device=dev, generator=gen)
            .bfloat16()[:, shift:shift + h * dim] for h in (heads, kvh))
    v = torch.randn(tokens, kvh * dim + 8, device=dev,
                    generator=gen).bfloat16()[:, :kvh * dim]
    table = ref.build_cos_sin_table(dim, 512, device=dev)
    pos = torch.randint(0, 512, (tokens,), device=dev, generator=gen).int()
    slots = torch.randperm(48, device=dev, generator=gen)[:tokens].int()
    if tokens > 1:
        slots[1] = -1
    kc, vc = torch.zeros(2, 3, kvh, 16, dim, device=dev).bfloat16()
    cs = table[pos.long()].double()[:, None]
    half = dim // 2

    def rotated(t):
        t = t.double().view(tokens, -1, dim)
        a, b = t[..., :half], t[..., half:]
        return torch.cat([a * cs[..., :half] - b * cs[..., half:],
                          b * cs[..., :half] + a * cs[..., half:]], -1)
    wants = [rotated(q), rotated(k)]
    old = v.clone()
    ops.rope_store_kv(q, k, v, kc, vc, table, pos, slots)
    for got, want in zip((q, k), wants):
        err = (got.double().view_as(want) - want).abs()
        assert (err <= want.abs() * 2 ** -8 + 2e-5).all()
    assert torch.equal(v, old)
    for cache, rows in ((kc, k), (vc, v)):
        want = torch.zeros_like(cache)
        for t, s in enumerate(slots.tolist()):
            if s >= 0:
                want[s // 16, :, s % 16] = rows[t].view(kvh, dim)
        assert torch.equal(cache, want)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 4, 5, 16, 32, 33, 65, 200])
@pytest.mark.parametrize("n,k", [(64, 512), (96, 8192), (1024, 14336),
                                 (4128, 1536), (9216, 2560), (14336, 1024)])
def test_skinny_gemm_forms(m, n, k):
    """The forms of summed products: a few rows, one part, up to 16 parts of
    unequal length, workgroups of 4 and 8 waves.  Bounds as above: half an ulp
    of the result and k roundings of 2^-24 of the sums of magnitudes."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(m * 1000003 + n + k)
    x = torch.randn(m, k, device=dev, generator=gen).bfloat16()
    w = torch.randn(n, k, device=dev, generator=gen).bfloat16()
    want = x.double() @ w.double().t().contiguous()
    bound = want.abs() * 2 ** -8 + \
        (x.double().abs() @ w.double().abs().t().contiguous()) * k * 2 ** -24
    for got in (ops._hip.skinny_gemm(x, w), ops.linear(x, w)):
        assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kvh", [(4, 4), (8, 2), (32, 8), (16, 16)])
@pytest.mark.parametrize("lens", [
    [0, 700], [1, 128, 129, 256, 257], [9000, 40, 3000], [2049] * 16,
    [100 + 37 * i for i in range(31)], [0] * 15 + [5000], list(range(64)),
    [1500, 30] * 32, [0], [384], [385], [2049], [16000],
    [500] * 31 + [16000], [5874 - 199 * i for i in range(28)] + [1] * 4,
    [8000] * 17 + [1] * 7, [15000] * 9 + [1] * 7, [300] * 64 + [3000]])
@pytest.mark.parametrize("splits", [2, 7, 32])
def test_decode_shares_out_lengths(heads, kvh, lens, splits):
    """Workgroups dealt out by the lengths, which a call with tickets takes for up to
    256 / kvh sequences and 64, two for each of these where sequences or rows without
    any leave none over, against parts of a fixed length and their own join: weights
    round to bf16 after other maxima (2^-9 of them each), results to bf16.  Twice, as
    the tickets are zeros again."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(sum(lens) + kvh)
    pages = sum((n + 15) // 16 for n in lens) + 1
    kc, vc = (torch.randn(pages, kvh, 16, 128, device=dev, generator=gen).bfloat16()
              for _ in "kv")
    most = max((n + 15) // 16 for n in lens) + 3
    table = torch.zeros(len(lens), most, dtype=torch.int32)
    order, at = torch.randperm(pages - 1) + 1, 0
    for i, n in enumerate(lens):
        table[i, :(n + 15) // 16] = order[at:at + (n + 15) // 16]
        at += (n + 15) // 16
    q = torch.randn(len(lens), heads, 128, device=dev, generator=gen).bfloat16()
    ctx = torch.tensor(lens, dtype=torch.int32, device=dev)
    tickets = torch.zeros(len(lens) * kvh, dtype=torch.int32, device=dev)
    args = q, kc, vc, table.to(dev), ctx, 0.09, splits
    want = ops.decode_attention(*args).double()
    bound = want.abs() * 2 ** -8 + vc.double().abs().max() * 2 ** -8
    for _ in range(2):
        got = ops.decode_attention(*args, tickets=tickets).double()
        assert ((got - want).abs() <= bound).all()
        assert not tickets.any()


@pytest.mark.gpu
def test_decode_cuts_one_long_among_many():
    """As many sequences as a key head has CUs: the long one is cut all the same.  The
    call with tickets takes about half of the time of fixed parts and their join; 2.2
    times of it with the long one whole."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    kc, vc, tables, ctx = _paged(dev, [500] * 31 + [16000], 8, 16384)
    q = torch.randn(32, 32, 128, device=dev).bfloat16()
    tickets = torch.zeros(32 * 8, dtype=torch.int32, device=dev)

    def least(**kw):
        times = []
        for _ in range(20):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in "be")
            begin.record()
            for _ in range(10):
                ops.decode_attention(q, kc, vc, tables, ctx, 0.09, 8, **kw)
            end.record()
            torch.cuda.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)
    assert least(tickets=tickets) < 1.2 * least()


@pytest.mark.gpu
@pytest.mark.parametrize("m", [5, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(4096, 768), (8192, 1280), (11264, 2816),
                                 (16448, 2304), (66048, 768), (16448, 2112)])
def test_swiglu_of_odd_lengths(m, n, k):
    """Gate/up of k that are no multiple of 512, or of 256, on whichever way; the bound
    of test_linear_swiglu."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(m * 7 + n + k)
    x = torch.randn(m, k, device=dev, generator=gen).bfloat16()
    w = (torch.randn(n, k, device=dev, generator=gen) / k ** 0.5).bfloat16()
    full = x.double() @ w.double().t().contiguous()
    gate, up = full[:, :n // 2], full[:, n // 2:]
    want = torch.nn.functional.silu(gate) * up
    bound = 2 ** -7 * (gate.abs() + 1) * (up.abs() + 1)
    assert ((ops.linear_swiglu(x, w).double() - want).abs() <= bound).all()
    assert ops._glu(m, n, k) or ops._tile_few(m, n, k) or k == 2816 and m > 32


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 7, 256, 257, 512, 513])
@pytest.mark.parametrize("hidden", [4, 256, 4096, 4100, 8192, 8196, 12288, 12292,
                                    16384])
def test_norm_of_rows(rows, hidden):
    """Every number of pieces that a thread holds, rows that end within one, and
    numbers of parts around what is in flight.  The sum is rounded to bf16 (2^-8 of
    it); the norm reads what was rounded and is rounded itself, from squares whose
    sum is off by 2^-8 at most where each is."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(rows + hidden)
    res = torch.randn(rows, hidden, device=dev, generator=gen).bfloat16()
    w = torch.randn(hidden, device=dev, generator=gen).bfloat16()

    def normed(t):
        return t * (t.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * w.double()
    if hidden % 8 == 0:
        want = normed(res.double())
        assert ((ops.rmsnorm(res, w, 1e-5).double() - want).abs()
                <= want.abs() * 2 ** -8 + 1e-6).all()
    for parts in (0, 1, 2, 3, 5, 7, 8, 9, 16):
        src = torch.randn(parts or 1, rows, hidden, device=dev, generator=gen)
        src = src if parts else src[0].bfloat16()
        total = (src.double().sum(0) if parts else src.double()) + res.double()
        got = res.clone()
        out = ops._hip.add_rmsnorm(src, got, w, 1e-5)
        assert ((got.double() - total).abs() <= total.abs() * 2 ** -8 + 1e-5).all()
        want = normed(total)
        # the residual's rounding is not in the norm's sum of squares
        assert ((out.double() - want).abs()
                <= want.abs() * 2 ** -7 + 1e-4 * w.double().abs() + 1e-5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m", [5, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(32832, 768), (32864, 1280), (57344, 512),
                                 (57376, 512)])
def test_skinny_gemm_wide(m, n, k):
    """32 rows of W a wave: from 32769 to 57344 columns, a last workgroup of a
    few of them, halves of gate/up that are no multiple of 32, a result in f32.
    The bounds of test_skinny_gemm_forms and test_linear_swiglu."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(m * 1000003 + n + k)
    x = torch.randn(m, k, device=dev, generator=gen).bfloat16()
    w = torch.randn(n, k, device=dev, generator=gen).bfloat16()
    want = x.double() @ w.double().t().contiguous()
    bound = want.abs() * 2 ** -8 + \
        (x.double().abs() @ w.double().abs().t().contiguous()) * k * 2 ** -24
    got = ops._hip.skinny_gemm(x, w)
    assert ((got.double() - want).abs() <= bound).all()
    assert torch.equal(ops._hip.skinny_gemm(x, w, wide=True), got.float())
    w = (w.float() / k ** 0.5).bfloat16()
    full = x.double() @ w.double().t().contiguous()
    gate, up = full[:, :n // 2], full[:, n // 2:]
    want = torch.nn.functional.silu(gate) * up
    bound = 2 ** -7 * (gate.abs() + 1) * (up.abs() + 1)
    got = ops._hip.skinny_swiglu(x, w)
    assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 2, 4, 5, 17, 32, 33, 64])
@pytest.mark.parametrize("f,k", [(3584, 4096), (7168, 2048), (6176, 2560),
                                 (8160, 2048), (9216, 2560), (19456, 2048)])
def test_swiglu_routes(m, f, k):
    """Both sides of the rule for silu within the GEMM, workgroups of 4 waves
    up to 16384 columns and of 8 beyond; the bound of test_linear_swiglu."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(m * 7 + f)
    x = torch.randn(m, k, device=dev, generator=gen).bfloat16()
    w = (torch.randn(2 * f, k, device=dev, generator=gen) / k ** 0.5
         ).bfloat16()
    full = x.double() @ w.double().t().contiguous()
    want = torch.nn.functional.silu(full[:, :f]) * full[:, f:]
    bound = 2 ** -7 * (full[:, :f].abs() + 1) * (full[:, f:].abs() + 1)
    for got in (ops._hip.skinny_swiglu(x, w), ops.linear_swiglu(x, w)):
        assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,width", [(7, 8), (300, 256), (512, 4096),
                                        (64, 8200), (50, 20)])
@pytest.mark.parametrize("count", [0, 1, 131])
def test_embed_rows(rows, width, count):
    """The indexed rows, from the end below 0; ids without a row touch no
    memory and give NaN; a width that only indexing takes."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    table = torch.randn(rows, width, device=dev).bfloat16()
    ids = torch.randint(-rows, rows, (count,), device=dev)
    if count > 1:
        ids[0], ids[1] = -rows, rows - 1
    want = table.cpu()[ids.cpu()]
    assert torch.equal(ops.embed_rows(ids, table).cpu(), want)
    assert torch.equal(ops.embed_rows(ids.int(), table).cpu(), want)
    if count > 1 and width % 8 == 0:
        ids[2], ids[3], ids[4] = rows, -rows - 1, 1 << 40
        got = ops.embed_rows(ids, table)
        assert got[2:5].isnan().all()
        assert torch.equal(got[5:].cpu(), want[5:])


@pytest.mark.gpu
def test_host_memory_that_kernels_read():
    """Pinned memory is fine-grained, and kept by torch's allocator until the stream has
    read it; of other memory neither is taken for granted, and no error is left."""
    from rbg_amd import ops
    for _ in range(3):
        pinned = torch.empty(4096, dtype=torch.uint8, pin_memory=True)
        assert ops._hip.host_memory(pinned) == (True, True)
        assert ops._hip.host_memory(torch.empty(4096, dtype=torch.uint8)) == \
            (False, False)
    torch.ones(8, device="cuda:0").add_(1)
    torch.cuda.synchronize()
