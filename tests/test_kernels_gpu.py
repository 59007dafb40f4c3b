"""HIP/CDNA4 kernels vs the plain-PyTorch fp32 reference (ops/reference.py).

Every test runs the HIP op on cuda:0 and the reference on the same inputs
(asymmetric random data), then compares with bf16-level tolerances.
"""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

from llm_map_reduce_summarizer_amd.ops import hip, reference  # noqa: E402

DEV = "cuda:0"


def _rand(*shape, scale=1.0, seed=0):
    g = torch.Generator(device="cpu").manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16).to(DEV)


def _close(a, b, atol, rtol=2e-2):
    a, b = a.float().cpu(), b.float().cpu()
    err = (a - b).abs()
    tol = atol + rtol * b.abs()
    bad = (err > tol).sum().item()
    assert bad == 0, "max err %.4g (%d bad of %d)" % (err.max().item(), bad, a.numel())


def test_debug_sync_mode(monkeypatch):
    """--debug-sync: every launch is followed by a device sync + error check (and stays capturable)."""
    monkeypatch.setattr(hip, "DEBUG_SYNC", True)
    x, w = _rand(3, 512, seed=1), _rand(512, seed=2)
    _close(hip.rmsnorm(x, w, 1e-5), reference.rmsnorm(x, w, 1e-5), 2e-2)
    g = torch.cuda.CUDAGraph()
    out = torch.empty_like(x)
    with torch.cuda.graph(g):
        hip.rmsnorm(x, w, 1e-5, out=out)
    g.replay()
    torch.cuda.synchronize()
    _close(out, reference.rmsnorm(x, w, 1e-5), 2e-2)


@pytest.mark.parametrize("T,D", [(1, 4096), (5, 4096), (3, 8192), (2, 256)])
def test_rmsnorm(T, D):
    x = _rand(T, D, seed=1)
    w = _rand(D, seed=2) + 1
    _close(hip.rmsnorm(x, w, 1e-5), reference.rmsnorm(x, w, 1e-5), 2e-2)


@pytest.mark.parametrize("T,D", [(1, 4096), (7, 4096), (3, 8192)])
def test_add_rmsnorm(T, D):
    x = _rand(T, D, seed=3)
    r = _rand(T, D, seed=4)
    w = _rand(D, seed=5) + 1
    r1, r2 = r.clone(), r.clone()
    o1 = hip.add_rmsnorm(x, r1, w, 1e-5)
    o2 = reference.add_rmsnorm(x, r2, w, 1e-5)
    _close(r1, r2, 1e-2)
    _close(o1, o2, 3e-2)


def _cache_setup(hq, hkv, d, page, n_pages, seed=0):
    k = torch.zeros(n_pages, hkv, page, d, dtype=torch.bfloat16, device=DEV)
    v = torch.zeros_like(k)
    return k, v


def test_rope_kv():
    hq, hkv, d, page = 4, 2, 128, 64
    T = 9
    qkv = _rand(T, (hq + 2 * hkv) * d, seed=7)
    positions = torch.tensor([0, 1, 2, 63, 64, 65, 200, 5, 6], dtype=torch.int32, device=DEV)
    seq_idx = torch.tensor([0, 0, 0, 0, 0, 0, 0, 1, 1], dtype=torch.int32, device=DEV)
    bt = torch.tensor([[3, 5, 1, 7], [2, 0, 0, 0]], dtype=torch.int32, device=DEV)
    cs = reference.rope_cos_sin(1024, d, 500000.0, DEV)
    k1, v1 = _cache_setup(hq, hkv, d, page, 8)
    k2, v2 = _cache_setup(hq, hkv, d, page, 8)
    q1, q2 = qkv.clone(), qkv.clone()
    hip.rope_kv(q1, positions, seq_idx, bt, k1, v1, cs, hq, hkv, d, page, check_bounds=True)
    reference.rope_kv(q2, positions, seq_idx, bt, k2, v2, cs, hq, hkv, d, page)
    _close(q1, q2, 2e-2)
    _close(k1, k2, 2e-2)
    assert torch.equal(v1, v2)


def test_swiglu_embed():
    gu = _rand(5, 2 * 1024, seed=8)
    _close(hip.swiglu(gu), reference.swiglu(gu), 2e-2)
    table = _rand(1000, 256, seed=9)
    ids = torch.tensor([0, 999, 5, 5, 123], dtype=torch.int32, device=DEV)
    assert torch.equal(hip.embed(ids, table), reference.embed(ids, table))


# (6, 2) / (24, 8) / (10, 2): GQA ratios 3 and 5 (Llama-3.2-3B is 24 / 8) take the per-query-head fallback
@pytest.mark.parametrize("hq,hkv", [(4, 2), (8, 2), (8, 1), (2, 2), (6, 2), (24, 8), (10, 2)])
@pytest.mark.parametrize("seqlens", [[1, 37, 130, 300], [64], [129, 256], [1000, 33, 2100]])
def test_attn_prefill(hq, hkv, seqlens):
    """Causal varlen prefill attention vs fp32."""
    d = 128
    T = sum(seqlens)
    qkv = _rand(T, (hq + 2 * hkv) * d, seed=11)
    cu = torch.tensor([0] + list(torch.tensor(seqlens).cumsum(0)), dtype=torch.int32, device=DEV)
    sc = 1.0 / math.sqrt(d)
    o1 = hip.attn_prefill(qkv, cu, hq, hkv, d, sc)
    o2 = reference.attn_prefill(qkv, cu, hq, hkv, d, sc)
    _close(o1, o2, 2e-2)


@pytest.mark.parametrize("parts", [False, True])
@pytest.mark.parametrize("fmt", ["fp8", "fp8v"])
def test_rope_kv_fp8_cache(parts, fmt):
    """rope_kv / rope_kv_parts writing the fp8 slab cache (kv8.h: e4m3 rows + power-of-two row scales) ==
    the reference quantiser on the same rotated rows; rows of padding tokens (seq_idx < 0) are not written."""
    hq, hkv, d, page, T = 8, 2, 128, 64, 150
    g = torch.Generator().manual_seed(31)
    cs = reference.rope_cos_sin(4096, d, 500000.0, DEV)
    bt = (torch.randperm(40, generator=g)[:24] + 1).view(2, 12).to(torch.int32).to(DEV)
    pos = torch.cat([torch.arange(100), torch.arange(700, 750)]).to(torch.int32).to(DEV)
    sidx = torch.tensor([0] * 100 + [1] * 49 + [-1], dtype=torch.int32, device=DEV)
    c0 = torch.zeros(48, hkv, reference.kv8_slab(page, d), dtype=torch.uint8, device=DEV)
    k1, v1, k2, v2 = c0.clone(), c0.clone(), c0.clone(), c0.clone()
    if fmt == "fp8v":  # bf16 K cache beside the fp8 V slabs
        k1 = torch.zeros(48, hkv, page, d, dtype=torch.bfloat16, device=DEV)
        k2 = k1.clone()
    if parts:
        pr = (torch.randn(3, T, (hq + 2 * hkv) * d, generator=g) * 0.7).to(DEV)
        q1 = hip.rope_kv_parts(pr, pos, sidx, bt, k1, v1, cs, hq, hkv, d, page)
        q2 = reference.rope_kv_parts(pr, pos, sidx, bt, k2, v2, cs, hq, hkv, d, page)
    else:
        q1 = _rand(T, (hq + 2 * hkv) * d, seed=32)
        q2 = q1.clone()
        hip.rope_kv(q1, pos, sidx, bt, k1, v1, cs, hq, hkv, d, page)
        reference.rope_kv(q2, pos, sidx, bt, k2, v2, cs, hq, hkv, d, page)
    _close(q1, q2, 2e-2)
    if fmt == "fp8":
        _kv8_close(k1, k2, page, d)
    else:
        _close(k1, k2, 2e-2)
    _kv8_close(v1, v2, page, d)
    assert float(k1[0].float().abs().sum()) == 0 and int(v1[0].sum()) == 0  # page 0 (scratch) untouched


def test_rope_kv_fp8_cache_tiny_rows():
    """Rows whose max|x| is far below e4m3's range (a subnormal row scale made 1 / scale inf and
    0 * inf = NaN): the kernel clamps the scale to 2^-126 as the reference does -- every stored scale finite
    and normal, every byte a finite e4m3 value, the dequantised rows equal to the reference's."""
    hq, hkv, d, page, T = 2, 1, 128, 64, 4
    cs = reference.rope_cos_sin(256, d, 500000.0, DEV)
    bt = torch.tensor([[1, 2]], dtype=torch.int32, device=DEV)
    pos = torch.arange(T, dtype=torch.int32, device=DEV)
    sidx = torch.zeros(T, dtype=torch.int32, device=DEV)
    qkv = torch.zeros(T, (hq + 2 * hkv) * d, dtype=torch.bfloat16, device=DEV)
    kv0 = hq * d
    # normal fp32 / bf16 values with max|x| / 448 subnormal (< 2^-126)
    qkv[0, kv0 + 3] = 1e-36              # k row 0: one tiny element, the rest zero
    qkv[1, kv0 + d:kv0 + 2 * d] = 3e-37  # v row 1: all tiny
    qkv[2, kv0 + 1] = -2e-37
    c0 = torch.zeros(4, hkv, reference.kv8_slab(page, d), dtype=torch.uint8, device=DEV)
    k1, v1, k2, v2 = c0.clone(), c0.clone(), c0.clone(), c0.clone()
    hip.rope_kv(qkv.clone(), pos, sidx, bt, k1, v1, cs, hq, hkv, d, page)
    reference.rope_kv(qkv.clone(), pos, sidx, bt, k2, v2, cs, hq, hkv, d, page)
    torch.cuda.synchronize()
    for c1, c2 in ((k1, k2), (v1, v2)):
        a = reference.cache_pages(c1.cpu(), torch.tensor([1]), page, d)
        b = reference.cache_pages(c2.cpu(), torch.tensor([1]), page, d)
        assert torch.all(torch.isfinite(a)) and torch.allclose(a, b, rtol=0.07, atol=0.0)
        sc = c1.cpu()[1, 0, page * d:].contiguous().view(torch.float32)[:T]  # the T written rows
        assert torch.all(torch.isfinite(sc)) and torch.all(sc >= 2.0 ** -126), sc


@pytest.mark.parametrize("hq,hkv", [(4, 1), (8, 2), (8, 1), (2, 2), (6, 2)])
@pytest.mark.parametrize("spans", [[(0, 200)], [(130, 300), (0, 77), (1000, 1129)], [(64, 128), (2047, 2048)]])
@pytest.mark.parametrize("kv8", ["bf16", "fp8", "fp8v"])
def test_attn_prefill_paged(hq, hkv, spans, kv8):
    """Chunked-prefill attention: slice rows attend to [0, prefix + slice) of their sequence read from the
    paged cache (random non-contiguous pages, stale rows past the slice end), vs the fp32 reference."""
    from llm_map_reduce_summarizer_amd.ops import PagedPrefill
    d, page = 128, 64
    g = torch.Generator().manual_seed(21)
    n_pages, maxp = 160, 40
    kc = (torch.randn(n_pages, hkv, page, d, generator=g) * 0.5).to(torch.bfloat16).to(DEV)
    vc = torch.randn(n_pages, hkv, page, d, generator=g).to(torch.bfloat16).to(DEV)
    kc, vc = _kv_format(kc, vc, kv8)
    nseq = len(spans)
    perm = torch.randperm(n_pages - 1, generator=g)[: nseq * maxp] + 1
    bt = perm.view(nseq, maxp).to(torch.int32).to(DEV)
    lens = [e - b for b, e in spans]
    T = sum(lens)
    qkv = _rand(T, (hq + 2 * hkv) * d, seed=22)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    slots = list(range(nseq))[::-1]  # sequence i uses block-table row nseq-1-i
    bt = bt.flip(0).contiguous()
    pre = [b for b, _ in spans]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    pp = PagedPrefill(bt, i32(slots), i32(pre), slots, pre, kc, vc)
    sc = 1.0 / math.sqrt(d)
    o1 = hip.attn_prefill(qkv, cu, hq, hkv, d, sc, paged=pp)
    o2 = reference.attn_prefill_paged(qkv, cu, hq, hkv, d, sc, pp)
    _close(o1, o2, 2e-2)


@pytest.mark.parametrize("hq,hkv", [(8, 8), (4, 2), (8, 2), (16, 2), (6, 2)])
@pytest.mark.parametrize("edge", [-1, 0, 1])
def test_attn_prefill_halves_of_an_item(hq, hkv, edge):
    """Two workgroups run the query block of a work item: sequences that end before, at and behind the first one's last
    position (the second has no row, or one), in the first block and in a later one, over packed rows and over pages."""
    from llm_map_reduce_summarizer_amd.ops import PagedPrefill
    d, block = 128, hip.prefill_block_m(hq // hkv)
    lens = [block // 2 + edge, block + edge, 3 * block // 2 + edge, 65]
    qkv, sc = _rand(sum(lens), (hq + 2 * hkv) * d, seed=13), 1.0 / math.sqrt(d)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    want = reference.attn_prefill(qkv, cu, hq, hkv, d, sc)
    _close(hip.attn_prefill(qkv, cu, hq, hkv, d, sc), want, 2e-2)
    pages = [-(-n // 64) for n in lens]
    kc, vc = (torch.full((sum(pages) + 1, hkv, 64, d), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    bt, page = torch.zeros(len(lens), max(pages), dtype=torch.int32), sum(pages)
    for i, n in enumerate(lens):
        rows = qkv[int(cu[i]):int(cu[i]) + n].view(n, hq + 2 * hkv, d).transpose(0, 1)
        for p in range(pages[i]):
            m = min(64, n - 64 * p)
            kc[page, :, :m], vc[page, :, :m] = rows[hq:hq + hkv, 64 * p:64 * p + m], rows[hq + hkv:, 64 * p:64 * p + m]
            bt[i, p], page = page, page - 1
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    slots, pre = list(range(len(lens))), [0] * len(lens)
    pp = PagedPrefill(bt.to(DEV), i32(slots), i32(pre), slots, pre, kc, vc)
    _close(hip.attn_prefill(qkv, cu, hq, hkv, d, sc, paged=pp), want, 2e-2)


@pytest.mark.parametrize("hq", [4, 8])
def test_attn_prefill_spike(hq):
    """A key far larger than the rest forces the online-softmax rescale path mid-sequence."""
    hkv, d = 1, 128
    seqlens = [300]
    T = 300
    qkv = _rand(T, (hq + 2 * hkv) * d, scale=0.5, seed=12)
    q0 = qkv[:, :d].float()
    kcol = hq * d
    qkv[200, kcol:kcol + d] = (q0[250] * 8).to(torch.bfloat16)  # key 200 spikes for query 250 (tile 3)
    cu = torch.tensor([0, T], dtype=torch.int32, device=DEV)
    sc = 1.0 / math.sqrt(d)
    _close(hip.attn_prefill(qkv, cu, hq, hkv, d, sc), reference.attn_prefill(qkv, cu, hq, hkv, d, sc), 2e-2)


@pytest.mark.parametrize("hq,hkv", [(4, 2), (8, 2), (8, 1), (4, 4), (16, 1), (6, 2), (24, 8), (10, 2)])
@pytest.mark.parametrize("splits", [1, 3, 16, 48, 100])  # 100 > 64: the merge's lanes hold several splits
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("kv8", ["bf16", "fp8", "fp8v"])
def test_attn_decode(hq, hkv, splits, fused, kv8):
    d, page = 128, 64
    ctxs = [1, 65, 700, 129, 64, 1000]
    B = len(ctxs)
    n_pages = 64
    g = torch.Generator().manual_seed(13)
    kc = (torch.randn(n_pages, hkv, page, d, generator=g)).to(torch.bfloat16).to(DEV)
    vc = (torch.randn(n_pages, hkv, page, d, generator=g)).to(torch.bfloat16).to(DEV)
    kc, vc = _kv_format(kc, vc, kv8)  # fp8 slab caches (kv8.h); the reference dequantises the same bytes
    perm = torch.randperm(n_pages - 1, generator=g) + 1
    bt = torch.zeros(B, 20, dtype=torch.int32)
    used = 0
    for b, c in enumerate(ctxs):
        npg = -(-c // page)
        bt[b, :npg] = perm[used:used + npg]
        used += npg
    bt = bt.to(DEV)
    pos = torch.tensor([c - 1 for c in ctxs], dtype=torch.int32, device=DEV)
    q = _rand(B, (hq + 2 * hkv) * d, seed=14)
    sc = 1.0 / math.sqrt(d)
    ws = hip.DecodeWorkspace(B, hq, d, splits, DEV, hip.decode_groups(hq, hkv), fused_combine=fused)
    # poisoned workspace (a reused allocation may hold NaN / inf): splits past a short context must not
    # leave stale slabs for the merge to multiply by a zero weight (0 x NaN = NaN)
    ws.part_o.fill_(float("nan"))
    ws.part_ml.fill_(float("nan"))
    o2 = reference.attn_decode(q, kc, vc, bt, pos, hq, hkv, d, page, sc)
    for _ in range(3):  # replays re-use (and must re-arm) the arrival counters
        o1 = hip.attn_decode(q, kc, vc, bt, pos, hq, hkv, d, page, sc, workspace=ws)
        _close(o1, o2, 2e-2)
    if fused:
        assert int(ws.counters.abs().sum()) == 0


@pytest.mark.parametrize("kv8", ["bf16", "fp8"])
@pytest.mark.parametrize("gate", [False, True])
def test_attn_decode_pages_of_a_split(kv8, gate):
    """One to six pages in a split, the last of one key or all, in the form that keeps one page in flight; with a gate the softmax
    weights in two terms (bf16)."""
    hq, hkv, d, page = 8, 2, 128, 64
    ctxs = [1, 63, 64, 65, 128, 129, 192, 193, 256, 257, 320, 321, 384]
    B, g = len(ctxs), torch.Generator().manual_seed(17)
    kc = torch.randn(60, hkv, page, d, generator=g).to(torch.bfloat16).to(DEV)
    vc = torch.randn(60, hkv, page, d, generator=g).to(torch.bfloat16).to(DEV)
    kc, vc = _kv_format(kc, vc, kv8)
    bt = torch.zeros(B, 6, dtype=torch.int32)
    perm, used = torch.randperm(59, generator=g) + 1, 0
    for b, c in enumerate(ctxs):
        n = -(-c // page)
        bt[b, :n] = perm[used:used + n]
        used += n
    bt, pos = bt.to(DEV), torch.tensor([c - 1 for c in ctxs], dtype=torch.int32, device=DEV)
    q, sc = _rand(B, (hq + 2 * hkv) * d, seed=18), 1.0 / math.sqrt(d)
    want = reference.attn_decode(q, kc, vc, bt, pos, hq, hkv, d, page, sc)
    factors = torch.rand(B, hq, generator=g).to(DEV) if gate else None
    if gate:
        want = (want.view(B, hq, d).float() * factors[:, :, None]).view(B, -1)
    for splits in (1, 2, 6):
        ws = hip.DecodeWorkspace(B, hq, d, splits, DEV, hkv)
        ws.part_o.fill_(float("nan"))
        _close(hip.attn_decode(q, kc, vc, bt, pos, hq, hkv, d, page, sc, workspace=ws, gate=factors), want, 2e-2)


@pytest.mark.parametrize("kv8", ["bf16", "fp8"])
@pytest.mark.parametrize("ctx", [64 * 33, 64 * 40 - 1])
def test_attn_decode_of_one_row(kv8, ctx):
    """One row on either side of the 256 workgroups from which its pages are read past the caches: the same bits as the same
    row beside another."""
    hq, hkv, d, page = 32, 8, 128, 64
    n, g = -(-ctx // page), torch.Generator().manual_seed(23)
    kc = torch.randn(n + 1, hkv, page, d, generator=g).to(torch.bfloat16).to(DEV)
    vc = torch.randn(n + 1, hkv, page, d, generator=g).to(torch.bfloat16).to(DEV)
    kc, vc = _kv_format(kc, vc, kv8)
    bt = (torch.randperm(n, generator=g) + 1).to(torch.int32).view(1, n).to(DEV)
    pos = torch.tensor([ctx - 1], dtype=torch.int32, device=DEV)
    q, sc = _rand(1, (hq + 2 * hkv) * d, seed=24), 1.0 / math.sqrt(d)
    want = reference.attn_decode(q, kc, vc, bt, pos, hq, hkv, d, page, sc)
    for splits in (31, 32):
        two = hip.attn_decode(q.repeat(2, 1), kc, vc, bt.repeat(2, 1), pos.repeat(2), hq, hkv, d, page, sc,
                              workspace=hip.DecodeWorkspace(2, hq, d, splits, DEV, hkv))
        got = hip.attn_decode(q, kc, vc, bt, pos, hq, hkv, d, page, sc, workspace=hip.DecodeWorkspace(1, hq, d, splits, DEV, hkv))
        _close(got, want, 2e-2)
        assert torch.equal(got[0], two[0]) and torch.equal(got[0], two[1])


@pytest.mark.parametrize("splits,fused", [(64, False), (160, False), (256, False), (256, True)])
def test_attn_decode_many_splits_one_kv_head(splits, fused):
    """A TP shard's single kv head at a long context split up to the merge's 256 ways (decode_attn_plan's
    TP-shard rule; the merge's lanes hold four splits each) -- vs the fp32 reference, replayed."""
    hq, hkv, d, page, ctx = 8, 1, 128, 64, 20000
    npg = -(-ctx // page)
    g = torch.Generator().manual_seed(91)
    kc = torch.randn(npg + 1, hkv, page, d, generator=g).to(torch.bfloat16).to(DEV)
    vc = torch.randn(npg + 1, hkv, page, d, generator=g).to(torch.bfloat16).to(DEV)
    bt = (torch.randperm(npg, generator=g).to(torch.int32) + 1).view(1, npg).to(DEV)
    pos = torch.tensor([ctx - 1], dtype=torch.int32, device=DEV)
    q = _rand(1, (hq + 2 * hkv) * d, seed=92)
    sc = 1.0 / math.sqrt(d)
    ws = hip.DecodeWorkspace(1, hq, d, splits, DEV, hip.decode_groups(hq, hkv), fused_combine=fused)
    ws.part_o.fill_(float("nan"))
    o2 = reference.attn_decode(q, kc, vc, bt, pos, hq, hkv, d, page, sc)
    for _ in range(2):
        o1 = hip.attn_decode(q, kc, vc, bt, pos, hq, hkv, d, page, sc, workspace=ws)
        _close(o1, o2, 2e-2)


class _St:
    def __init__(self, B, V, temps, seeds, positions, max_new=100):
        i32 = dict(dtype=torch.int32, device=DEV)
        self.next_ids = torch.zeros(B, **i32)
        self.positions = torch.tensor(positions, **i32)
        self.gen_count = torch.zeros(B, **i32)
        self.max_new = torch.full((B,), max_new, **i32)
        self.out_tokens = torch.zeros(B, 8, **i32)
        self.done = torch.zeros(B, **i32)
        self.result = torch.zeros(B, dtype=torch.int64, device=DEV)
        self.temps = torch.tensor(temps, dtype=torch.float32, device=DEV)
        self.seeds = torch.tensor(seeds, dtype=torch.int64, device=DEV)
        self.eos = torch.tensor([7, -1, -1, -1], **i32)


def test_sampler_greedy_and_gumbel():
    B, V = 4, 128256
    logits = _rand(B, V, scale=2.0, seed=15)
    temps, seeds, pos = [0.0, 0.3, 1.0, 0.3], [1, 2, 3, 4], [5, 0, 17, 4000]
    st = _St(B, V, temps, seeds, pos)
    hip.sample(logits, st)
    got = st.out_tokens[:, 0].cpu()
    ref = reference.sample_tokens(logits.cpu(), torch.tensor(temps), torch.tensor(seeds), torch.tensor(pos))
    for b in range(B):
        row = logits[b].float().cpu()
        if temps[b] > 0:
            row = row / temps[b] + reference.gumbel_noise(seeds[b], pos[b], V)
        # same winner, or a near-tie within fp rounding of the fast log
        assert int(got[b]) == int(ref[b]) or row[int(got[b])] >= row.max() - 1e-3
    assert st.positions.cpu().tolist() == [p + 1 for p in pos]
    assert st.gen_count.cpu().tolist() == [1] * B
    assert torch.equal(st.next_ids.cpu(), got)
    assert st.result.abs().sum().item() == 0


def test_sampler_eos_and_max_new():
    B, V = 2, 1000
    logits = torch.full((B, V), -5.0, dtype=torch.bfloat16, device=DEV)
    logits[0, 7] = 5.0  # eos
    logits[1, 3] = 5.0
    st = _St(B, V, [0.0, 0.0], [0, 0], [10, 10], max_new=1)
    st.max_new[0] = 50
    hip.sample(logits, st)
    assert st.done.cpu().tolist() == [1, 1]
    assert st.positions.cpu().tolist() == [10, 10]  # retired rows keep their position
    hip.sample(logits, st)  # retired rows are untouched
    assert st.gen_count.cpu().tolist() == [1, 1]


@pytest.mark.parametrize("M", [1, 5, 16, 24, 48, 64])
@pytest.mark.parametrize("N,K", [(6144, 4096), (256, 1024), (4096, 14336)])
def test_skinny_linear(M, N, K):
    x = _rand(M, K, seed=21)
    w = _rand(N, K, scale=0.05, seed=22)
    ref = (x.float() @ w.float().t())
    _close(hip.linear(x, w), ref, 2e-2)


@pytest.mark.parametrize("M", [1, 7, 33])
@pytest.mark.parametrize("splits", [1, 2, 4, 7])
def test_skinny_linear_parts(M, splits):
    N, K = 512, 3584
    x = _rand(M, K, seed=23)
    w = _rand(N, K, scale=0.05, seed=24)
    parts = hip.linear_parts(x, w, splits)
    assert parts.shape == (splits, M, N)
    ref = reference.linear_parts(x, w, splits)
    _close(parts, ref, 1e-3, 1e-3)


@pytest.mark.parametrize("M", [1, 17, 64])
def test_skinny_swiglu(M):
    F, K = 1024, 2048
    x = _rand(M, K, seed=25)
    wg = _rand(F, K, scale=0.05, seed=26)
    wu = _rand(F, K, scale=0.05, seed=27)
    wgu = reference.interleave_gate_up(wg, wu).contiguous()
    g, u = x.float() @ wg.float().t(), x.float() @ wu.float().t()
    ref = g * torch.sigmoid(g) * u
    _close(hip.linear_swiglu(x, wgu), ref, 2e-2)
    # prefill path: hipBLASLt GEMM + blocked-layout swiglu kernel
    _close(hip.swiglu(torch.nn.functional.linear(x, wgu)), ref, 3e-2)


@pytest.mark.parametrize("S,T,D", [(1, 3, 4096), (4, 9, 4096), (2, 1, 8192)])
def test_add_rmsnorm_parts(S, T, D):
    g = torch.Generator().manual_seed(28)
    parts = torch.randn(S, T, D, generator=g).to(DEV)
    r = _rand(T, D, seed=29)
    w = _rand(D, seed=30) + 1
    r1, r2 = r.clone(), r.clone()
    o1 = hip.add_rmsnorm_parts(parts, r1, w, 1e-5)
    o2 = reference.add_rmsnorm_parts(parts, r2, w, 1e-5)
    _close(r1, r2, 2e-2)
    _close(o1, o2, 3e-2)


@pytest.mark.parametrize("S", [1, 3])
def test_rope_kv_parts(S):
    hq, hkv, d, page = 4, 2, 128, 64
    T = 5
    W = (hq + 2 * hkv) * d
    g = torch.Generator().manual_seed(31)
    parts = torch.randn(S, T, W, generator=g).to(DEV)
    positions = torch.tensor([0, 63, 64, 7, 300], dtype=torch.int32, device=DEV)
    seq_idx = torch.tensor([0, 0, 0, 1, 1], dtype=torch.int32, device=DEV)
    bt = torch.tensor([[3, 5, 1, 7, 2, 6], [4, 0, 0, 0, 6, 2]], dtype=torch.int32, device=DEV)
    cs = reference.rope_cos_sin(1024, d, 500000.0, DEV)
    k1, v1 = _cache_setup(hq, hkv, d, page, 8)
    k2, v2 = _cache_setup(hq, hkv, d, page, 8)
    o1 = hip.rope_kv_parts(parts, positions, seq_idx, bt, k1, v1, cs, hq, hkv, d, page)
    o2 = reference.rope_kv_parts(parts, positions, seq_idx, bt, k2, v2, cs, hq, hkv, d, page)
    _close(o1, o2, 3e-2)
    _close(k1, k2, 3e-2)
    _close(v1, v2, 3e-2)



@pytest.mark.parametrize("M", [1, 17, 33, 48, 64])
@pytest.mark.parametrize("K", [1024, 640])
def test_skinny_lds_all_epilogues(M, K):
    x = _rand(M, K, seed=40)
    w = _rand(512, K, scale=0.05, seed=41)
    ref = x.float() @ w.float().t()
    o = torch.empty(M, 512, dtype=torch.bfloat16, device=DEV)
    _close(hip._skinny_lds(x, w, o, hip.EPI_BF16, 1, 512), ref, 2e-2)
    for S in ((1, 2, 8) if K == 1024 else (1, 5)):  # K=640: 5 k blocks
        parts = hip.linear_parts(x, w, S, kernel="lds")
        _close(parts.sum(0), ref, 1e-3, 1e-3)
    for wpb in (5, 6, 7, 8):  # 16 * wpb-row tiles
        n = 16 * wpb * 3
        ww = _rand(n, K, scale=0.05, seed=44)
        S = 2 if (K // 128) % 2 == 0 else 1
        oo = torch.empty(S, M, n, dtype=torch.float32, device=DEV)
        _close(hip._skinny_lds(x, ww, oo, hip.EPI_F32_PARTIAL, S, n, wpb).sum(0),
               x.float() @ ww.float().t(), 1e-3, 1e-3)


@pytest.mark.parametrize("M", [1, 9, 16, 39, 64])
@pytest.mark.parametrize("wpb", [4, 5, 6, 7, 8])
@pytest.mark.parametrize("K", [128, 384, 1024, 2304])  # 1 .. 18 k blocks: ring prologue / tail paths
def test_stream_gemm(M, wpb, K):
    x = _rand(M, K, seed=60)
    n = 16 * wpb * 3
    w = _rand(n, K, scale=0.05, seed=61)
    ref = x.float() @ w.float().t()
    o = torch.empty(M, n, dtype=torch.bfloat16, device=DEV)
    _close(hip._stream_gemm(x, w, o, hip.EPI_BF16, 1, n, wpb), ref, 2e-2)
    nkb = K // 128
    for S in sorted({1, 2 if nkb % 2 == 0 else 1, nkb}):
        parts = torch.empty(S, M, n, dtype=torch.float32, device=DEV)
        _close(hip._stream_gemm(x, w, parts, hip.EPI_F32_PARTIAL, S, n, wpb).sum(0), ref, 1e-3, 1e-3)
    f = 8 * wpb * 3
    wg = _rand(f, K, scale=0.05, seed=62)
    wu = _rand(f, K, scale=0.05, seed=63)
    g, u = x.float() @ wg.float().t(), x.float() @ wu.float().t()
    act = torch.empty(M, f, dtype=torch.bfloat16, device=DEV)
    _close(hip._stream_gemm(x, reference.interleave_gate_up(wg, wu).contiguous(), act, hip.EPI_SWIGLU, 1, f, wpb),
           g * torch.sigmoid(g) * u, 2e-2)
    wg = _rand(256, K, scale=0.05, seed=42)
    wu = _rand(256, K, scale=0.05, seed=43)
    g, u = x.float() @ wg.float().t(), x.float() @ wu.float().t()
    _close(hip.linear_swiglu(x, reference.interleave_gate_up(wg, wu).contiguous(), kernel="lds"),
           g * torch.sigmoid(g) * u, 2e-2)


@pytest.mark.parametrize("M,K", [(1, 128), (16, 256), (17, 1152), (32, 2048), (33, 256), (64, 1024)])
@pytest.mark.parametrize("norm", [False, True])
def test_stream_gemm_many_rounds(M, K, norm):
    """Grids of more than two rounds share CUs in pairs with shallow rings (K blocks fewer than the ring's slots, as many and
    more): the bits of the same columns from grids of one round, whose rings are deep."""
    n = 64 * 514
    x, w = _rand(M, K, seed=64), _rand(n, K, scale=0.05, seed=65)
    half, kw = n // 2, {}
    if norm:
        kw["norm"] = ((x.float() ** 2).view(M, 32, -1).sum(-1).contiguous(), 1e-5)

    def run(w, epi):
        n = w.shape[0]
        shape = {hip.EPI_BF16: (M, n), hip.EPI_F32_PARTIAL: (1, M, n), hip.EPI_SWIGLU: (M, n // 2)}[epi]
        o = torch.empty(shape, dtype=torch.float32 if epi == hip.EPI_F32_PARTIAL else torch.bfloat16, device=DEV)
        return hip._stream_gemm(x, w, o, epi, 1, shape[-1], 4, **kw)
    for epi in (hip.EPI_BF16, hip.EPI_F32_PARTIAL, hip.EPI_SWIGLU):
        assert torch.equal(run(w, epi), torch.cat([run(w[:half], epi), run(w[half:], epi)], -1))
    if not norm:
        _close(run(w, hip.EPI_F32_PARTIAL)[0], x.float() @ w.float().t(), 1e-3, 1e-3)


@pytest.mark.parametrize("M", [1, 10, 39, 64])
@pytest.mark.parametrize("N,K,wpb,S", [(3584, 4096, 7, 8), (7168, 4096, 7, 4), (448, 1024, 4, 2), (896, 512, 8, 4)])
def test_stream_swiglu_split(M, N, K, wpb, S):
    """split-K SwiGLU (last arriving split of a column tile applies silu(gate) * up): vs fp32, and the
    arrival tickets re-arm (repeated launches and a replayed hipGraph give the same answer)."""
    x = _rand(M, K, seed=64)
    wg = _rand(N // 2, K, scale=0.05, seed=65)
    wu = _rand(N // 2, K, scale=0.05, seed=66)
    g, u = x.float() @ wg.float().t(), x.float() @ wu.float().t()
    ref = g * torch.sigmoid(g) * u
    w = reference.interleave_gate_up(wg, wu).contiguous()
    out = torch.empty(M, N // 2, dtype=torch.bfloat16, device=DEV)
    for _ in range(3):
        out.zero_()
        _close(hip.stream_swiglu_split(x, w, out, wpb, S), ref, 2e-2)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        hip.stream_swiglu_split(x, w, out, wpb, S)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        _close(out, ref, 2e-2)
    assert int(hip._tile_counters(x.device, N // (16 * wpb))[: N // (16 * wpb)].abs().sum()) == 0


@pytest.mark.parametrize("M", [1, 5, 17, 48, 64, 200])
@pytest.mark.parametrize("N,K", [(1280, 8192), (512, 3584)])
def test_fp8_linear(M, N, K):
    from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight
    x = _rand(M, K, seed=50)
    w = Fp8Weight.quantize(_rand(N, K, scale=0.05, seed=51))
    ref = x.float() @ w.dequant().t()
    out = hip.fp8_linear(x, w)
    if M <= hip.SKINNY_MAX_M:
        _close(out, ref, 2e-2)  # W8A16: exact weights, bf16 activations
    else:  # hipBLASLt fp8 with dynamic per-token activation scales: e4m3 activation rounding (~3.6% per
        # element, independent over K) -> check the relative RMS error, not every element
        rel = ((out.float().cpu() - ref.cpu()).norm() / ref.cpu().norm()).item()
        assert rel < 0.05, rel
    for S in (1, 2):
        parts = hip.fp8_linear_parts(x[:min(M, 64)], w, S)
        _close(parts.sum(0), ref[:min(M, 64)], 2e-3, 2e-3)


@pytest.mark.parametrize("N,K,S", [(256, 8192, 1), (128, 28672, 1), (128, 28672, 4), (96, 32768, 1), (64, 1024, 2)])
def test_skinny_fp8_m1_x_in_lds(N, K, S):
    """Register-streaming fp8 kernel at M = 1 (x slice staged in LDS when it fits 56 KiB: K / S <= 28672,
    else x from global): bf16 out, split-K fp32 slabs and SwiGLU vs fp32 of the dequantised weights."""
    from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight, interleave_gate_up
    x = _rand(1, K, seed=60)
    w = Fp8Weight.quantize(_rand(N, K, scale=0.05, seed=61))
    ref = x.float() @ w.dequant().t()
    if S == 1:
        out = torch.empty(1, N, dtype=torch.bfloat16, device=DEV)
        _close(hip._skinny_fp8(x, w, out, hip.EPI_BF16, 1, 1, N), ref, 2e-2)
    parts = torch.empty(S, 1, N, dtype=torch.float32, device=DEV)
    _close(hip._skinny_fp8(x, w, parts, hip.EPI_F32_PARTIAL, 2 if N % 32 == 0 else 1, S, N).sum(0), ref, 2e-3, 2e-3)
    if S == 1:
        wg = Fp8Weight.quantize(_rand(N, K, scale=0.05, seed=62))
        wu = Fp8Weight.quantize(_rand(N, K, scale=0.05, seed=63))
        g, u = x.float() @ wg.dequant().t(), x.float() @ wu.dequant().t()
        wgu = Fp8Weight(interleave_gate_up(wg.q.view(torch.uint8), wu.q.view(torch.uint8)).view(torch.float8_e4m3fn)
                        .contiguous(), interleave_gate_up(wg.scale[:, None], wu.scale[:, None])[:, 0].contiguous())
        act = torch.empty(1, N, dtype=torch.bfloat16, device=DEV)
        _close(hip._skinny_fp8(x, wgu, act, hip.EPI_SWIGLU, 1, 1, N), g * torch.sigmoid(g) * u, 3e-2)


@pytest.mark.parametrize("M", [1, 9, 17, 40, 64])
@pytest.mark.parametrize("N,K,wpb,S", [(640, 1024, 5, 1), (512, 2048, 4, 2), (896, 768, 7, 3), (1024, 512, 8, 2)])
def test_stream_fp8(M, N, K, wpb, S):
    """fp8 LDS-DMA stream GEMM (256-wide k slots): bf16 out, split-K fp32 slabs and SwiGLU vs fp32 of the
    dequantised weights."""
    from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight
    x = _rand(M, K, seed=80)
    w = Fp8Weight.quantize(_rand(N, K, scale=0.05, seed=81))
    ref = x.float() @ w.dequant().t()
    out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    _close(hip._stream_fp8(x, w, out, hip.EPI_BF16, 1, N, wpb), ref, 2e-2)
    parts = torch.empty(S, M, N, dtype=torch.float32, device=DEV)
    _close(hip._stream_fp8(x, w, parts, hip.EPI_F32_PARTIAL, S, N, wpb).sum(0), ref, 2e-3, 2e-3)
    wg, wu = _rand(N // 2, K, scale=0.05, seed=82), _rand(N // 2, K, scale=0.05, seed=83)
    wgu = Fp8Weight.quantize(reference.interleave_gate_up(wg, wu).contiguous())
    g, u = reference.split_gate_up(x.float() @ wgu.dequant().t())
    act = torch.empty(M, N // 2, dtype=torch.bfloat16, device=DEV)
    _close(hip._stream_fp8(x, wgu, act, hip.EPI_SWIGLU, 1, N // 2, wpb), g * torch.sigmoid(g) * u, 3e-2)


@pytest.mark.parametrize("M", [1, 10, 16, 40])
@pytest.mark.parametrize("N,K,wpb,S", [(7168, 8192, 7, 4), (7168, 8192, 4, 2), (896, 1024, 7, 2), (1024, 512, 8, 1)])
def test_stream_fp8_swiglu_split(M, N, K, wpb, S, monkeypatch):
    """fp8 stream GEMM with the split-K SwiGLU epilogue (a narrow gate_up, e.g. a Llama-3-70B TP=8 shard's
    7168 rows: S workgroups per column tile, the last to arrive applies silu(gate) * up) vs fp32 of the
    dequantised weights; twice in a row (the tickets re-arm), and through fp8_linear_swiglu with the split
    configuration forced."""
    from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight
    x = _rand(M, K, seed=84)
    wg, wu = _rand(N // 2, K, scale=0.05, seed=85), _rand(N // 2, K, scale=0.05, seed=86)
    wgu = Fp8Weight.quantize(reference.interleave_gate_up(wg, wu).contiguous())
    g, u = reference.split_gate_up(x.float() @ wgu.dequant().t())
    ref = g * torch.sigmoid(g) * u
    parts = torch.empty(S, M, N, dtype=torch.float32, device=DEV)
    cnt = hip._tile_counters(x.device, N // (16 * wpb))
    first = None
    for _ in range(2):
        act = torch.empty(M, N // 2, dtype=torch.bfloat16, device=DEV)
        hip._stream_fp8(x, wgu, act, hip.EPI_SWIGLU_SPLIT, S, N // 2, wpb, parts=parts, counters=cnt)
        _close(act, ref, 3e-2)
        first = act.clone() if first is None else first
        assert torch.equal(act, first)
    assert int(cnt[:N // (16 * wpb)].abs().sum()) == 0
    if S > 1 and M <= hip.SKINNY_MAX_M:
        monkeypatch.setattr(hip, "stream_config_fp8", lambda N_, K_, swiglu=False, splits=None, M=1: (wpb, S))
        _close(hip.fp8_linear_swiglu(x, wgu), ref, 3e-2)
    # consuming a deferred RMSNorm (per-tile sums of squares of the un-normalised rows, the TP-push producer's
    # output): the row scale multiplies every split's partial tile before the last arriver sums them
    tiles = 64
    h = x * 3
    ssq = h.float().pow(2).view(M, tiles, K // tiles).sum(-1).contiguous()
    hf = h.float()
    gn, un = reference.split_gate_up((hf * torch.rsqrt(hf.pow(2).mean(-1, keepdim=True) + 1e-5)) @ wgu.dequant().t())
    act = torch.empty(M, N // 2, dtype=torch.bfloat16, device=DEV)
    hip._stream_fp8(h, wgu, act, hip.EPI_SWIGLU_SPLIT, S, N // 2, wpb, parts=parts, counters=cnt, norm=(ssq, 1e-5))
    _close(act, gn * torch.sigmoid(gn) * un, 3e-2, 3e-2)


def test_fp8_swiglu_and_quant():
    from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight
    M, F, K = 9, 512, 1024
    x = _rand(M, K, seed=52)
    wg, wu = _rand(F, K, scale=0.05, seed=53), _rand(F, K, scale=0.05, seed=54)
    w = Fp8Weight.quantize(reference.interleave_gate_up(wg, wu).contiguous())
    full = x.float() @ w.dequant().t()
    g, u = reference.split_gate_up(full)
    _close(hip.fp8_linear_swiglu(x, w), g * torch.sigmoid(g) * u, 3e-2)
    q, s = hip.quant_fp8_rows(x)
    ref_q = (x.float() / s[:, None]).to(torch.float8_e4m3fn)
    assert torch.allclose(s.cpu(), x.float().abs().amax(1).cpu() / 448, rtol=1e-5)
    assert (q.float() - ref_q.float()).abs().max().item() <= 16.0  # at most one e4m3 ulp at the top binade
    assert (q.float() == ref_q.float()).float().mean().item() > 0.98


@pytest.mark.parametrize("hq,hkv,S", [(32, 8, 4), (4, 1, 1), (16, 1, 3), (8, 2, 2), (4, 1, 16), (6, 2, 2), (24, 8, 4)])
@pytest.mark.parametrize("fused_combine", [False, True])
@pytest.mark.parametrize("kv8", ["bf16", "fp8", "fp8v"])
def test_attn_decode_rope_fused(hq, hkv, S, fused_combine, kv8):
    """attn_decode_rope (q/k RoPE + new K/V written into the cache + attention, from the QKV GEMM's
    fp32 split-K slabs) == reference rope_kv_parts followed by reference attention."""
    d, page = 128, 64
    ctxs = [1, 64, 65, 700, 129, 1000]
    B = len(ctxs)
    n_pages = 64
    g = torch.Generator().manual_seed(77)
    kc0 = torch.randn(n_pages, hkv, page, d, generator=g).to(torch.bfloat16)
    vc0 = torch.randn(n_pages, hkv, page, d, generator=g).to(torch.bfloat16)
    perm = torch.randperm(n_pages - 1, generator=g) + 1
    bt = torch.zeros(B, 20, dtype=torch.int32)
    used = 0
    for b, c in enumerate(ctxs):
        npg = -(-c // page)
        bt[b, :npg] = perm[used:used + npg]
        used += npg
    bt = bt.to(DEV)
    pos = torch.tensor([c - 1 for c in ctxs], dtype=torch.int32, device=DEV)
    W = (hq + 2 * hkv) * d
    parts = (torch.randn(S, B, W, generator=g) * 0.5).to(DEV)
    cs = reference.rope_cos_sin(2048, d, 500000.0, DEV)
    sc = 1.0 / math.sqrt(d)
    sidx = torch.arange(B, dtype=torch.int32, device=DEV)
    kc0, vc0 = _kv_format(kc0, vc0, kv8)
    k2, v2 = kc0.clone().to(DEV), vc0.clone().to(DEV)
    qkv = reference.rope_kv_parts(parts, pos, sidx, bt, k2, v2, cs, hq, hkv, d, page)
    o2 = reference.attn_decode(qkv, k2, v2, bt, pos, hq, hkv, d, page, sc)
    k1, v1 = kc0.clone().to(DEV), vc0.clone().to(DEV)
    ng = hip.decode_groups(hq, hkv)
    ws = hip.DecodeWorkspace(B, hq, d, hip.decode_splits(B, ng, 20 * page), DEV, ng, fused_combine=fused_combine)
    ws.part_o.fill_(float("nan"))  # poisoned workspace: empty splits must publish zero slabs
    for _ in range(3):  # idempotent: later calls rewrite the same K/V row (and re-armed merge tickets)
        o1 = hip.attn_decode_rope(parts, cs, k1, v1, bt, pos, hq, hkv, d, page, sc, workspace=ws)
        if kv8 != "bf16":  # the kernel rotates the fp32 slab sums, the reference their bf16 rounding: an element
            # of the new row on an e4m3 rounding boundary may land one step apart, so compare in relative L2
            a, b = o1.float().cpu(), o2.float().cpu()
            assert float((a - b).norm() / b.norm()) < 2e-2
        else:
            _close(o1, o2, 2e-2)
    if fused_combine:
        assert int(ws.counters.abs().sum()) == 0
    for c1, c2 in ((k1, k2), (v1, v2)):
        if c1.dtype == torch.uint8:
            _kv8_close(c1, c2, page, d)
        else:
            _close(c1, c2, 3e-2)


def _kv_format(kc, vc, fmt):
    """bf16 caches [pages, hkv, P, d] in the engine's format ``fmt``: bf16, fp8 (K and V slabs) or fp8v (V
    slabs, K bf16); same device as the inputs."""
    dev = kc.device
    if fmt == "fp8":
        kc = reference.kv8_from_bf16(kc.cpu()).to(dev)
    if fmt in ("fp8", "fp8v"):
        vc = reference.kv8_from_bf16(vc.cpu()).to(dev)
    return kc, vc


def _kv8_close(c1, c2, page, d):
    """Two fp8 slab caches hold the same rows: dequantised within 2 % relative L2 (the kernels rotate / sum
    in fp32 where the reference rounds to bf16 first, so an element on an e4m3 rounding boundary may land
    one step -- 6-12 % -- apart) and >= 95 % of the row bytes identical."""
    allp = torch.arange(c1.shape[0])
    a = reference.cache_pages(c1.cpu(), allp, page, d)
    b = reference.cache_pages(c2.cpu(), allp, page, d)
    assert float((a - b).norm() / b.norm().clamp_min(1e-12)) <= 2e-2
    written = (c2.cpu()[..., :page * d] != 0) | (c1.cpu()[..., :page * d] != 0)
    same = (c1.cpu()[..., :page * d] == c2.cpu()[..., :page * d])[written].float().mean()
    assert float(same) >= 0.95, float(same)


@pytest.mark.parametrize("tp", [2, 4, 8])
@pytest.mark.parametrize("M", [1, 10, 39, 48, 64])
def test_tp_shard_decode_blocks(tp, M):
    """The fused decode blocks (ops.qkv_rope + attn_decode, proj_add_rmsnorm, gate_up_swiglu) at the
    per-rank shard shapes of Llama-3-8B under TP=tp (e.g. TP=8: 1 KV head, QKV N=768, o K=512, gate_up
    N=3584, down K=1792) -- whatever GEMM plan they pick -- against the fp32 reference."""
    from llm_map_reduce_summarizer_amd import ops
    hid, hd, page = 4096, 128, 64
    hq, hkv, ffn = 32 // tp, 8 // tp, 14336 // tp
    sc = 1.0 / math.sqrt(hd)
    x = _rand(M, hid, seed=70)
    wqkv = _rand((hq + 2 * hkv) * hd, hid, scale=0.02, seed=71)
    wo = _rand(hid, hq * hd, scale=0.02, seed=72)
    wgu = _rand(2 * ffn, hid, scale=0.02, seed=73)
    wd = _rand(hid, ffn, scale=0.02, seed=74)
    ln = (torch.rand(hid) + 0.5).to(torch.bfloat16).to(DEV)
    cs = reference.rope_cos_sin(4096, hd, 500000.0, DEV)
    n_pages = M * 3 + 1
    g = torch.Generator().manual_seed(75)
    k0 = torch.randn(n_pages, hkv, page, hd, generator=g).to(torch.bfloat16)
    v0 = torch.randn(n_pages, hkv, page, hd, generator=g).to(torch.bfloat16)
    bt = (1 + torch.arange(M * 3, dtype=torch.int32).view(M, 3)).to(DEV)
    pos = torch.tensor([(37 * i) % 190 for i in range(M)], dtype=torch.int32, device=DEV)
    sidx = torch.arange(M, dtype=torch.int32, device=DEV)
    # attention block: fused GPU path vs reference rope_kv + attention
    k1, v1 = k0.clone().to(DEV), v0.clone().to(DEV)
    k2, v2 = k0.clone().to(DEV), v0.clone().to(DEV)
    q1 = ops.qkv_rope(x, wqkv, pos, sidx, bt, k1, v1, cs, hq, hkv, hd, page, defer=True)
    a1 = ops.attn_decode(q1, k1, v1, bt, pos, hq, hkv, hd, page, sc)
    qkv2 = reference.linear(x, wqkv)
    reference.rope_kv(qkv2, pos, sidx, bt, k2, v2, cs, hq, hkv, hd, page)
    a2 = reference.attn_decode(qkv2, k2, v2, bt, pos, hq, hkv, hd, page, sc)
    _close(a1, a2, 3e-2, 5e-2)
    # o projection + residual + norm, gate_up + SwiGLU, down + residual + norm
    r1, r2 = x.clone(), x.clone()
    h1 = ops.proj_add_rmsnorm(a2, wo, r1, ln, 1e-5, "o")
    h2 = reference.add_rmsnorm(reference.linear(a2, wo), r2, ln, 1e-5)
    _close(r1, r2, 3e-2)
    _close(h1, h2, 5e-2, 5e-2)
    act1 = ops.gate_up_swiglu(h2, wgu)
    act2 = reference.swiglu(reference.linear(h2, wgu))
    _close(act1, act2, 3e-2, 5e-2)
    d1 = ops.proj_add_rmsnorm(act2, wd, r1.copy_(x), ln, 1e-5, "down")
    d2 = reference.add_rmsnorm(reference.linear(act2, wd), r2.copy_(x), ln, 1e-5)
    _close(d1, d2, 5e-2, 5e-2)


@pytest.mark.parametrize("M", [1, 39, 64])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("N,K,wpb,S", [(4096, 4096, 4, 4), (4096, 14336, 4, 4), (2048, 1024, 8, 2), (4096, 2048, 4, 1),
                                       (8192, 8192, 8, 4), (8192, 28672, 8, 4)])
def test_stream_resid_and_norm_consumer(M, fp8, N, K, wpb, S):
    """The deferred-RMSNorm kernels at every decode M (ops uses them up to DEFER_NORM_MAX_M rows): the
    split-K residual-update producer (bf16 / fp8 weights) vs fp32, its per-tile sums of squares, and a
    stream consumer (fp32 slabs) scaling its rows by the deferred norm."""
    from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight
    if fp8 and K % 256:
        pytest.skip("fp8 stream slots are 256 wide")
    x = _rand(M, K, seed=100)
    w = _rand(N, K, scale=0.02, seed=101)
    wq = Fp8Weight.quantize(w) if fp8 else w
    w32 = wq.dequant() if fp8 else w.float()
    res0 = _rand(M, N, seed=102)
    res = res0.clone()
    ssp = hip.stream_resid(x, wq, res, wpb, S)
    ref = (res0.float() + x.float() @ w32.t()).to(torch.bfloat16)
    _close(res, ref, 2e-2, 2e-2)
    tiles = N // (16 * wpb)
    _close(ssp, res.float().pow(2).view(M, tiles, 16 * wpb).sum(-1), 1e-3, 1e-3)
    if tiles % 32 == 0:  # consumer: rows of ``res`` normalised through the deferred norm
        w2 = _rand(1024, N, scale=0.02, seed=103)
        parts = torch.empty(2, M, 1024, dtype=torch.float32, device=DEV)
        hip._stream_gemm(res, w2, parts, hip.EPI_F32_PARTIAL, 2, 1024, 4, norm=(ssp, 1e-5))
        hf = res.float()
        xn = hf * torch.rsqrt(hf.pow(2).mean(-1, keepdim=True) + 1e-5)
        _close(parts.sum(0), xn @ w2.float().t(), 2e-3, 2e-3)
    assert all(int(t.abs().sum()) == 0 for t in hip._TILE_COUNTERS.values())


@pytest.mark.parametrize("M", [1, 10, 16])
@pytest.mark.parametrize("fp8", [False, True])
def test_deferred_norm_decode_layer(M, fp8):
    """Deferred RMSNorm through a Llama-3-8B decode layer (TP=1, unit gains as after folding): the o / down
    projections update the residual in their split-K last-arriver epilogue and return an ops.NormRows
    (per-tile sums of squares); qkv (+ fused RoPE attention), gate_up + SwiGLU and the LM head scale their
    product rows by the deferred norm -- each against the fp32 reference of the plain composition
    (add + RMSNorm, then the GEMM); a captured hipGraph replays it with re-armed tickets."""
    from llm_map_reduce_summarizer_amd import ops
    from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight
    hid, hd, page, hq, hkv, ffn, eps = 4096, 128, 64, 32, 8, 14336, 1e-5
    sc = 1.0 / math.sqrt(hd)
    q8 = (lambda t: Fp8Weight.quantize(t)) if fp8 else (lambda t: t)
    w32 = (lambda w: w.dequant()) if fp8 else (lambda w: w.float())  # exact fp8 x scale weights
    x0 = _rand(M, hid, seed=90)
    a = _rand(M, hq * hd, seed=91)
    wo, wd = q8(_rand(hid, hq * hd, scale=0.02, seed=92)), q8(_rand(hid, ffn, scale=0.02, seed=93))
    wgu, wqkv = q8(_rand(2 * ffn, hid, scale=0.02, seed=94)), q8(_rand((hq + 2 * hkv) * hd, hid, scale=0.02, seed=95))
    head = _rand(16384, hid, scale=0.02, seed=96)
    one = torch.ones(hid, dtype=torch.bfloat16, device=DEV)

    def rms32(h):  # the consumer sees the un-rounded normalised rows: the fp32 oracle of the deferred norm
        hf = h.float()
        return hf * torch.rsqrt(hf.pow(2).mean(-1, keepdim=True) + eps)

    def swiglu32(gu):
        gg, uu = reference.split_gate_up(gu)
        return gg * torch.sigmoid(gg) * uu
    # o projection -> NormRows; residual and the per-tile sums of squares
    r1, r2 = x0.clone(), x0.clone()
    nr = ops.proj_add_rmsnorm(a, wo, r1, None, eps, "o")
    assert isinstance(nr, ops.NormRows) and nr.h is r1
    h2 = reference.add_rmsnorm(reference.linear(a, wo), r2, one, eps)
    _close(r1, r2, 2e-2, 2e-2)
    tiles = nr.ssq.shape[1]
    _close(nr.ssq, r1.float().pow(2).view(M, tiles, hid // tiles).sum(-1), 1e-3, 1e-3)
    _close(nr.materialize(), h2, 3e-2, 3e-2)
    # gate_up + SwiGLU consumes the deferred norm
    # a consumer on the stream kernel takes the deferred norm (fp32 oracle); others get materialised bf16 rows
    takes = hip.fp8_swiglu_takes_norm(M, 2 * ffn, hid) if fp8 else \
        hip.plan("gate_up", M, 2 * ffn, hid)[0] in ("stream", "stream_split")
    _close(ops.gate_up_swiglu(nr, wgu), swiglu32((rms32(r2) if takes else h2.float()) @ w32(wgu).t()),
           3e-2, 5e-2)
    act2 = reference.swiglu(reference.linear(h2, wgu))
    # down -> NormRows -> next layer's qkv + fused RoPE attention, and the LM head
    r1.copy_(x0)
    r2.copy_(x0)
    nr2 = ops.proj_add_rmsnorm(act2, wd, r1, None, eps, "down")
    h3 = reference.add_rmsnorm(reference.linear(act2, wd), r2, one, eps)
    _close(r1, r2, 2e-2, 2e-2)
    g = torch.Generator().manual_seed(97)
    k0 = torch.randn(M * 3 + 1, hkv, page, hd, generator=g).to(torch.bfloat16)
    v0 = torch.randn(M * 3 + 1, hkv, page, hd, generator=g).to(torch.bfloat16)
    bt = (1 + torch.arange(M * 3, dtype=torch.int32).view(M, 3)).to(DEV)
    pos = torch.tensor([(41 * i) % 190 for i in range(M)], dtype=torch.int32, device=DEV)
    sidx = torch.arange(M, dtype=torch.int32, device=DEV)
    cs = reference.rope_cos_sin(4096, hd, 500000.0, DEV)
    k1, v1, k2, v2 = k0.clone().to(DEV), v0.clone().to(DEV), k0.clone().to(DEV), v0.clone().to(DEV)
    q1 = ops.qkv_rope(nr2, wqkv, pos, sidx, bt, k1, v1, cs, hq, hkv, hd, page, defer=True)
    at1 = ops.attn_decode(q1, k1, v1, bt, pos, hq, hkv, hd, page, sc)
    qkv2 = (rms32(r2) @ w32(wqkv).t()).to(torch.bfloat16)
    reference.rope_kv(qkv2, pos, sidx, bt, k2, v2, cs, hq, hkv, hd, page)
    _close(at1, reference.attn_decode(qkv2, k2, v2, bt, pos, hq, hkv, hd, page, sc), 3e-2, 5e-2)
    _close(ops.linear(nr2, head), rms32(r2) @ head.float().t(), 3e-2, 5e-2)
    _close(nr2.materialize(), h3, 3e-2, 3e-2)
    # hipGraph: capture producer + consumer once, replay from the same residual -> same output
    r1.copy_(x0)
    out = {}
    graph = torch.cuda.CUDAGraph()
    ops.gate_up_swiglu(ops.proj_add_rmsnorm(a, wo, r1, None, eps, "o"), wgu)  # tickets / buffers before capture
    with torch.cuda.graph(graph):
        out["act"] = ops.gate_up_swiglu(ops.proj_add_rmsnorm(a, wo, r1, None, eps, "o"), wgu)
    r2.copy_(x0)
    reference.add_rmsnorm(reference.linear(a, wo), r2, one, eps)
    ref = swiglu32((rms32(r2) if takes else rms32(r2).to(torch.bfloat16).float()) @ w32(wgu).t())
    for _ in range(3):
        r1.copy_(x0)
        graph.replay()
        torch.cuda.synchronize()
        _close(out["act"], ref, 3e-2, 5e-2)
    assert all(int(t.abs().sum()) == 0 for t in hip._TILE_COUNTERS.values())


@pytest.mark.parametrize("N,K,S", [(10240, 8192, 4), (1024, 8192, 1), (512, 28672, 8), (256, 4096, 2)])
def test_skinny_fp8_deferred_norm(N, K, S):
    """One decode row through the register-streaming fp8 kernel with the x slice in LDS, consuming a deferred
    RMSNorm (per-tile sums of squares of the un-normalised row): split-K slabs, bf16 and SwiGLU epilogues
    against the fp32 oracle rmsnorm(h) @ W^T -- the Llama-3-70B M = 1 qkv / gate_up consumers."""
    from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight
    h = _rand(1, K, seed=110) * 3
    tiles = 64
    ssq = h.float().pow(2).view(1, tiles, K // tiles).sum(-1).contiguous()
    hf = h.float()
    xn = hf * torch.rsqrt(hf.pow(2).mean(-1, keepdim=True) + 1e-5)
    w = Fp8Weight.quantize(_rand(N, K, scale=0.02, seed=111))
    ref = xn @ w.dequant().t()
    assert hip.skinny_fp8_takes_norm(1, K, S)
    parts = hip.fp8_linear_parts(h, w, S, 1, norm=(ssq, 1e-5))
    _close(parts.sum(0), ref, 2e-3, 2e-3)
    out = torch.empty(1, N, dtype=torch.bfloat16, device=DEV)
    _close(hip._skinny_fp8(h, w, out, hip.EPI_BF16, 1, 1, N, norm=(ssq, 1e-5)), ref, 2e-2, 2e-2)
    g, u = reference.split_gate_up(ref)
    act = torch.empty(1, N // 2, dtype=torch.bfloat16, device=DEV)
    _close(hip._skinny_fp8(h, w, act, hip.EPI_SWIGLU, 1, 1, N // 2, norm=(ssq, 1e-5)), g * torch.sigmoid(g) * u,
           3e-2, 3e-2)


@pytest.mark.parametrize("M", [65, 96, 128, 200, 256])
@pytest.mark.parametrize("wpb,S", [(4, 4), (7, 1)])
def test_stream_gemm_row_chunks(M, wpb, S):
    """Decode batches above 64 rows (the 24 h map's bucket 96) run the stream GEMM over 64-row chunks: bf16
    rows, fp32 split-K slabs written at their row offset of every [S, M, N] slab (slab row stride M) and
    SwiGLU -- each against fp32; the ops-level plan takes the stream kernel up to 256 rows (gate_up 128)."""
    K = 1024
    x = _rand(M, K, seed=70)
    n = 16 * wpb * 4
    w = _rand(n, K, scale=0.05, seed=71)
    ref = x.float() @ w.float().t()
    o = torch.empty(M, n, dtype=torch.bfloat16, device=DEV)
    _close(hip._stream_gemm(x, w, o, hip.EPI_BF16, 1, n, wpb), ref, 2e-2)
    parts = torch.full((S, M, n), float("nan"), dtype=torch.float32, device=DEV)
    _close(hip._stream_gemm(x, w, parts, hip.EPI_F32_PARTIAL, S, n, wpb).sum(0), ref, 1e-3, 1e-3)
    f = 8 * wpb * 4
    wg, wu = _rand(f, K, scale=0.05, seed=72), _rand(f, K, scale=0.05, seed=73)
    g, u = x.float() @ wg.float().t(), x.float() @ wu.float().t()
    act = torch.empty(M, f, dtype=torch.bfloat16, device=DEV)
    _close(hip._stream_gemm(x, reference.interleave_gate_up(wg, wu).contiguous(), act, hip.EPI_SWIGLU, 1, f, wpb),
           g * torch.sigmoid(g) * u, 2e-2)
    assert hip.plan("o", M, 4096, 4096)[0] == "stream"
    assert hip.plan("gate_up", M, 28672, 4096)[0] == ("stream" if M <= 128 else "gemm")


@pytest.mark.parametrize("M", [65, 96, 200])
def test_fp8_linear_row_chunks(M):
    """fp8 decode batches of 65-256 rows: the W8A16 streaming kernels over 64-row chunks (bf16 rows, SwiGLU
    up to 128 rows) against the fp32 product of the dequantised weights."""
    from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight
    K, N = 1024, 768
    x = _rand(M, K, seed=80)
    w = Fp8Weight.quantize(_rand(N, K, scale=0.05, seed=81))
    ref = x.float() @ w.dequant().t()
    _close(hip.fp8_linear(x, w), ref, 3e-2, 3e-2)
    if M <= hip.STREAM_MAX_M_SWIGLU:  # above: the W8A8 fp8 GEMM (activation quantisation, own tests)
        g, u = reference.split_gate_up(ref)
        _close(hip.fp8_linear_swiglu(x, w), g * torch.sigmoid(g) * u, 3e-2, 3e-2)


def test_kv_scatter_matches_reference():
    """Context-parallel prefill: all-gathered K/V rows [n, 2, hkv, d] land in the paged cache at (page, slot);
    page -1 rows (own rows, all-gather padding) are skipped."""
    g = torch.Generator().manual_seed(31)
    pages, hkv, P, d, n = 12, 2, 64, 128, 300
    rows = torch.randn(n, 2, hkv, d, generator=g).to(torch.bfloat16)
    perm = torch.randperm(pages * P, generator=g)[:n]
    page = (perm // P).to(torch.int32)
    slot = (perm % P).to(torch.int32)
    page[::7] = -1
    kc0 = torch.randn(pages, hkv, P, d, generator=g).to(torch.bfloat16)
    vc0 = torch.randn(pages, hkv, P, d, generator=g).to(torch.bfloat16)
    kr, vr = kc0.clone(), vc0.clone()
    reference.kv_scatter(rows, page, slot, kr, vr)
    kg, vg = kc0.to(DEV), vc0.to(DEV)
    hip.kv_scatter(rows.to(DEV), page.to(DEV), slot.to(DEV), kg, vg)
    assert torch.equal(kg.cpu(), kr) and torch.equal(vg.cpu(), vr)
    assert not torch.equal(kr, kc0)  # something was written


@pytest.mark.parametrize("M", [7, 39])
@pytest.mark.parametrize("fp8", [False, True])
def test_stream_resid_tp_push_group_of_one(fp8, M):
    """TP-push residual producer over a group of ONE rank (parallel/custom_ar.py LocalPush: the TP-shard
    measurement path): push to its own slot, flag, wait, rank-ordered sum -- against the fp32 reference
    residual update, eager and graph-replayed with changing inputs (the self-test), and against the local
    (non-TP) producer on the same operands."""
    from llm_map_reduce_summarizer_amd.parallel.custom_ar import LocalPush, _test_push
    h = LocalPush(max_bytes=1 << 20)
    try:
        if not fp8 and M == 7:
            assert _test_push(h, torch.device(DEV), 3)
        N, K = 4096, 1024
        x = _rand(M, K, scale=0.5, seed=3)
        wb = _rand(N, K, scale=0.05, seed=4)
        w = reference.Fp8Weight.quantize(wb) if fp8 else wb
        res0 = _rand(M, N, seed=5)
        wpb, S = (8, 2) if fp8 else (4, 4)
        r_tp, r_loc = res0.clone(), res0.clone()
        ss_tp = hip.stream_resid(x, w, r_tp, wpb, S, tp=h.push_handle())
        ss_loc = hip.stream_resid(x, w, r_loc, wpb, S)
        ref = (res0.float() + reference.linear(x, w).float()).to(torch.bfloat16)
        _close(r_tp, ref, 3e-2, 2e-2)
        _close(r_tp, r_loc, 3e-2, 2e-2)
        _close(ss_tp, ss_loc, 1.0, 1e-2)
        assert h.error() == 0
    finally:
        h.close()


@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("tp", [False, True])
@pytest.mark.parametrize("K", [1024, 3584])
def test_skinny_fp8_resid_producer(M, tp, K):
    """fp8-weight register-streaming residual producer (skinny_fp8_kernel EPI_RESID; 70B TP=8 shard o / down
    shapes): residual += x @ dequant(w)^T through the TP push over a group of one when ``tp``, per-tile row
    sums of squares -- against fp32, repeated calls (push epochs advance)."""
    from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight
    from llm_map_reduce_summarizer_amd.parallel.custom_ar import LocalPush
    h = LocalPush(max_bytes=1 << 20) if tp else None
    try:
        N = 8192
        x = _rand(M, K, scale=0.5, seed=31)
        w = Fp8Weight.quantize(_rand(N, K, scale=0.05, seed=32))
        res0 = _rand(M, N, seed=33)
        res = res0.clone()
        for _ in range(3):
            res.copy_(res0)
            ssp = hip.skinny_resid(x, w, res, tp=h.push_handle() if tp else None)
        ref = (res0.float() + x.float() @ w.dequant().t()).to(torch.bfloat16)
        _close(res, ref, 3e-2, 2e-2)
        _close(ssp, res.float().pow(2).reshape(M, N // 16, 16).sum(-1), 1e-2, 1e-3)
        if tp:
            assert h.error() == 0
    finally:
        if h is not None:
            h.close()


@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("tp", [False, True])
def test_skinny_resid_producer(M, tp):
    """Register-streaming deferred-norm producer (skinny_gemm.hip EPI_RESID): residual += x @ w^T (through
    the TP push over a group of one when ``tp``) and per-16-column-tile row sums of squares -- against the
    fp32 reference; the SwiGLU consumer with that deferred norm against the materialised RMSNorm rows."""
    from llm_map_reduce_summarizer_amd.parallel.custom_ar import LocalPush
    h = LocalPush(max_bytes=1 << 20) if tp else None
    try:
        N, K, F = 4096, 1024, 3584
        x = _rand(M, K, scale=0.5, seed=11)
        w = _rand(N, K, scale=0.05, seed=12)
        res0 = _rand(M, N, seed=13)
        res = res0.clone()
        for it in range(3):  # repeated calls: the TP push epochs / slot parities advance
            res.copy_(res0)
            ssp = hip.skinny_resid(x, w, res, tp=h.push_handle() if tp else None)
        ref = (res0.float() + reference.linear(x, w).float()).to(torch.bfloat16)
        _close(res, ref, 3e-2, 2e-2)
        ss = res.float().pow(2).reshape(M, N // 16, 16).sum(-1)
        _close(ssp, ss, 1e-2, 1e-3)
        wgu = _rand(F, N, scale=0.02, seed=14)
        eps = 1e-5
        y = hip.linear_swiglu(res, wgu, kernel="skinny", norm=(ssp, eps))
        xn = reference.rmsnorm(res, torch.ones(N, dtype=torch.bfloat16, device=DEV), eps)
        _close(y, hip.linear_swiglu(xn, wgu, kernel="skinny"), 2e-2, 3e-2)
        if tp:
            assert h.error() == 0
    finally:
        if h is not None:
            h.close()


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("M", [1, 7, 16, 40])
def test_skinny_waves_every_epilogue(waves, M):
    """Register-streaming kernels (bf16 and fp8 weights) with 4- and 8-wave workgroups (hip.skinny_waves):
    bf16 out, split-K fp32 slabs (k blocks not a multiple of the wave count), SwiGLU with and without the
    deferred norm, the residual producer -- against fp32 references."""
    from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight, interleave_gate_up
    old = hip.SKINNY_WAVES_FORCE
    hip.SKINNY_WAVES_FORCE = waves
    try:
        N, K = 512, 1792  # 14 k blocks: 8 waves -> waves 6, 7 take one block fewer
        x = _rand(M, K, seed=90)
        w = _rand(N, K, scale=0.05, seed=91)
        ref = x.float() @ w.float().t()
        for nt in (1, 2):
            out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
            _close(hip._skinny(x, w, out, hip.EPI_BF16, nt, 1, N), ref, 2e-2)
        parts = torch.empty(7, M, N, dtype=torch.float32, device=DEV)
        _close(hip._skinny(x, w, parts, hip.EPI_F32_PARTIAL, 1, 7, N).sum(0), ref, 2e-3, 2e-3)
        wgu = interleave_gate_up(_rand(N, K, scale=0.05, seed=92), _rand(N, K, scale=0.05, seed=93)).contiguous()
        g, u = (x.float() @ wgu.float().t()).reshape(M, -1, 2, 8).unbind(2)
        act = hip.linear_swiglu(x, wgu, kernel="skinny")
        _close(act, (g * torch.sigmoid(g) * u).reshape(M, N), 2e-2, 3e-2)
        if M <= 16:
            res0 = _rand(M, N, seed=94)
            res = res0.clone()
            ssp = hip.skinny_resid(x, w, res)
            _close(res, (res0.float() + ref).to(torch.bfloat16), 3e-2, 2e-2)
            _close(ssp, res.float().pow(2).reshape(M, N // 16, 16).sum(-1), 1e-2, 1e-3)
            y = hip.linear_swiglu(res, wgu[:, :N].contiguous(), kernel="skinny", norm=(ssp, 1e-5))
            xn = reference.rmsnorm(res, torch.ones(N, dtype=torch.bfloat16, device=DEV), 1e-5)
            _close(y, hip.linear_swiglu(xn, wgu[:, :N].contiguous(), kernel="skinny"), 2e-2, 3e-2)
        w8 = Fp8Weight.quantize(w)
        ref8 = x.float() @ w8.dequant().t()
        out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        _close(hip._skinny_fp8(x, w8, out, hip.EPI_BF16, 1, 1, N), ref8, 2e-2)
        parts = torch.empty(7, M, N, dtype=torch.float32, device=DEV)
        _close(hip._skinny_fp8(x, w8, parts, hip.EPI_F32_PARTIAL, 2, 7, N).sum(0), ref8, 2e-3, 2e-3)
    finally:
        hip.SKINNY_WAVES_FORCE = old


@pytest.mark.parametrize("add", [False, True])
@pytest.mark.parametrize("D", [4096, 8192])
def test_rmsnorm_fp8_matches_norm_then_quant(add, D):
    """Fused norm + row-wise e4m3fn quantisation (norm.hip Q8) against rmsnorm / add_rmsnorm followed by
    quant_fp8_rows: the same residual update, dequantised rows within one e4m3 step of the two-pass result
    (the fused pass quantises the fp32 values, not their bf16 rounding)."""
    T = 300
    x = _rand(T, D, seed=21)
    res0 = _rand(T, D, seed=22)
    w = (torch.rand(D, generator=torch.Generator().manual_seed(23)) + 0.5).to(torch.bfloat16).to(DEV)
    r1, r2 = res0.clone(), res0.clone()
    q, sc = hip.rmsnorm_fp8(x, w, 1e-5, residual=r1 if add else None)
    y = hip.add_rmsnorm(x, r2, w, 1e-5) if add else hip.rmsnorm(x, w, 1e-5)
    q2, sc2 = hip.quant_fp8_rows(y)
    if add:
        assert torch.equal(r1, r2)
    torch.testing.assert_close(sc, sc2, rtol=1e-2, atol=0)
    deq = q.float() * sc[:, None]
    ref = y.float()
    # half an e4m3 step of the top binade (32 quantised units) plus the bf16 rounding of the two-pass rows
    # (<= 2^-8 of 448 units)
    step = sc[:, None] * 32
    assert ((deq - ref).abs() <= step * 0.5 + sc[:, None] * 448 * 2 ** -8 + 1e-6).all()
    assert (q.float() == q2.float()).float().mean() > 0.9


@pytest.mark.parametrize("add", [False, True])
def test_rmsnorm_fp8_two_term(add):
    """Two-term fp8 rows (norm.hip Q8 == 2): [hi | lo] on one row scale, hi + lo / 16 reproduces the
    normalised row to ~2^-8 of its magnitude (16x finer than the single-term rows), and the two-term GEMM
    (gemm.hip: the lo K-tiles re-read W with E8M0 block scale 2^-4) equals (hi + lo / 16) s @ W^T."""
    T, D, N = 300, 4096, 1280
    x = _rand(T, D, seed=41)
    res0 = _rand(T, D, seed=42)
    w = (torch.rand(D, generator=torch.Generator().manual_seed(43)) + 0.5).to(torch.bfloat16).to(DEV)
    r1, r2 = res0.clone(), res0.clone()
    q, sc = hip.rmsnorm_fp8(x, w, 1e-5, residual=r1 if add else None, split=True)
    q1, sc1 = hip.rmsnorm_fp8(x, w, 1e-5, residual=r2 if add else None)
    assert q.shape == (T, 2 * D) and torch.equal(sc, sc1) and torch.equal(q[:, :D].float(), q1.float())
    y = hip.add_rmsnorm(x, res0.clone(), w, 1e-5) if add else hip.rmsnorm(x, w, 1e-5)
    two = (q[:, :D].float() + q[:, D:].float() / 16) * sc[:, None]
    one = q1.float() * sc[:, None]
    e2 = float((two - y.float()).norm() / y.float().norm())
    e1 = float((one - y.float()).norm() / y.float().norm())
    assert e2 < e1 / 6, (e1, e2)  # bf16 rounding of the reference row bounds e2 from below
    from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight
    wq = Fp8Weight.quantize(_rand(N, D, seed=44, scale=0.02))
    out = hip.gemm_fp8(q, sc, wq)
    ref = two @ wq.dequant().t()
    _close(out, ref, 2e-2)


@pytest.mark.parametrize("M", [65, 92, 128, 200])
def test_stream_gemm_tall_tiles_match_row_chunks(M, monkeypatch):
    """65-128 decode rows run in ONE pass over the weights on 96- / 128-row x tiles (hip.STREAM_TALL_M); every
    output element accumulates over k in the same order as the 64-row chunks, so the two are bit-identical --
    bf16 rows, fp32 split-K slabs and SwiGLU, at Llama-3-8B widths."""
    K = 4096
    x = _rand(M, K, seed=80)
    for n, S, epi in ((6144, 4, hip.EPI_F32_PARTIAL), (4096, 1, hip.EPI_BF16), (2048, 1, hip.EPI_SWIGLU)):
        w = _rand(n, K, scale=0.02, seed=81)
        wpb = 4 if epi != hip.EPI_F32_PARTIAL else 6
        shape = (S, M, n) if epi == hip.EPI_F32_PARTIAL else (M, n // 2 if epi == hip.EPI_SWIGLU else n)
        dt = torch.float32 if epi == hip.EPI_F32_PARTIAL else torch.bfloat16
        outs = []
        for tall in (128, 64):
            monkeypatch.setattr(hip, "STREAM_TALL_M", tall)
            o = torch.full(shape, float("nan"), dtype=dt, device=DEV)
            outs.append(hip._stream_gemm(x, w, o, epi, S, n // 2 if epi == hip.EPI_SWIGLU else n, wpb))
        torch.cuda.synchronize()
        assert torch.equal(outs[0], outs[1]), (n, S, epi)
        if epi == hip.EPI_F32_PARTIAL:
            _close(outs[0].sum(0), x.float() @ w.float().t(), 1e-3, 1e-3)


@pytest.mark.parametrize("M,wpb", [(65, 8), (80, 7), (81, 7), (96, 4), (96, 8), (97, 6), (112, 7), (113, 5),
                                   (113, 6), (128, 7), (128, 8)])
def test_stream_gemm_tall_widths(M, wpb):
    """Every tile height and the widths it newly takes, slots of 64 and 128 of k: equal to the 64-row chunks, bit for bit."""
    K, n = 1024, 16 * wpb * 3
    x, w = _rand(M, K, seed=82), _rand(n, K, scale=0.05, seed=83)
    for epi, S in ((hip.EPI_F32_PARTIAL, 2), (hip.EPI_BF16, 1), (hip.EPI_SWIGLU, 1)):
        cols = n // 2 if epi == hip.EPI_SWIGLU else n
        shape, dt = ((S, M, n), torch.float32) if epi == hip.EPI_F32_PARTIAL else ((M, cols), torch.bfloat16)
        one, two = (torch.full(shape, float("nan"), dtype=dt, device=DEV) for _ in range(2))
        hip._stream_launch(x, w, one, epi, S, cols, wpb, None, None, None, None, None, M if S > 1 else 0)
        for a, b in ((0, 64), (64, M)):
            o = two[:, a:b] if S > 1 else two[a:b]
            hip._stream_launch(x[a:b], w, o, epi, S, cols, wpb, None, None, None, None, None, M if S > 1 else 0)
        assert torch.equal(one, two), epi


@pytest.mark.parametrize("M", [65, 96, 128])
def test_linear_tall_lm_head(M):
    """linear() of 65-128 rows of a stream shape (the decode LM head of the 24 h map's bucket 96) runs the
    tall-tile stream GEMM: against fp32, and equal to the 256 x 256-tile GEMM within bf16 rounding."""
    K, N = 4096, 16 * 4 * 1002  # a vocabulary-like width that the stream kernel tiles (wpb 4)
    x, w = _rand(M, K, seed=90), _rand(N, K, scale=0.02, seed=91)
    out = hip.linear(x, w)
    torch.cuda.synchronize()
    _close(out, x.float() @ w.float().t(), 2e-2)
