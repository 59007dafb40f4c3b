"""Large-M MFMA GEMMs (csrc/kernels/gemm_bf16.hip, gemm.hip) vs a plain PyTorch fp32 reference.

Covers ragged M (tiles past M), N tails (a vocab shard that is not a multiple of 256),
strided activations, both epilogues (LDS-staged 16-B row stores for aligned outputs, register
stores for outputs that are not 16-B aligned), the fused SwiGLU epilogue, and the fp8
(OCP e4m3fn, block-scaled MFMA with unit scales) path against the dequantised fp32 product.
Data is asymmetric random (an output transpose or a row/column swap would not pass).
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

from llm_map_reduce_summarizer_amd.ops import hip, reference  # noqa: E402
from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight  # noqa: E402

DEV = "cuda:0"


def _rand(*shape, scale=1.0, seed=0, offset=0.0):
    g = torch.Generator(device="cpu").manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale + offset).to(torch.bfloat16).to(DEV)


def _check(out, ref, tol=2e-2):
    out, ref = out.float(), ref.float()
    err = (out - ref).abs()
    bound = tol * (ref.abs() + ref.abs().mean())
    bad = int((err > bound).sum())
    assert bad == 0, "max err %.4g (%d bad of %d), ref mean |x| %.4g" % (err.max(), bad, out.numel(),
                                                                         ref.abs().mean())


@pytest.mark.parametrize("M,N,K", [(65, 256, 128), (1000, 1280, 4096), (4097, 6144, 4096),
                                   (300, 16032, 1024), (16384 + 13, 4096, 1024), (257, 4096, 14336)])
@pytest.mark.parametrize("aligned", [True, False])
def test_gemm_bf16(M, N, K, aligned):
    x = _rand(M, K, seed=1, scale=0.5, offset=0.05)
    w = _rand(N, K, seed=2, scale=0.02, offset=0.001)
    ref = x.float() @ w.float().t()
    if aligned:
        out = hip.gemm(x, w)
    else:  # an 8-byte (not 16-byte) aligned output view: the register-store epilogue
        big = torch.zeros(M, N + 8, dtype=torch.bfloat16, device=DEV)
        out = hip.gemm(x, w, out=big[:, 4:4 + N])
    torch.cuda.synchronize()
    _check(out, ref)


def test_gemm_bf16_identity_asymmetric():
    """A = I exposes a transposed store; W asymmetric so a row/col swap shows."""
    K = 256
    x = torch.eye(K, dtype=torch.bfloat16, device=DEV)
    w = (torch.arange(512 * K, device=DEV, dtype=torch.float32).reshape(512, K) % 97 - 48).to(torch.bfloat16)
    out = hip.gemm(x, w)
    torch.cuda.synchronize()
    assert torch.equal(out.float(), w.float().t()), "C = I . W^T must equal W^T exactly"


def test_gemm_strided_input_and_out():
    M, K, N = 700, 1024, 512
    big = _rand(M, K + 64, seed=3, scale=0.3)
    x = big[:, 32:32 + K]
    w = _rand(N, K, seed=4, scale=0.05)
    for off in (0, 4):  # 16-B aligned view (LDS epilogue) and 8-B aligned view (register epilogue)
        out_big = torch.zeros(M, N + 16, dtype=torch.bfloat16, device=DEV)
        hip.gemm(x, w, out=out_big[:, off:off + N])
        torch.cuda.synchronize()
        _check(out_big[:, off:off + N], x.float() @ w.float().t())
        assert float(out_big[:, N + off:].abs().max()) == 0.0 and float(out_big[:, :off].abs().max() if off else 0) == 0.0, \
            "wrote outside the output view"


@pytest.mark.parametrize("M", [100, 3000])
def test_gemm_swiglu(M):
    K, F = 4096, 1792
    x = _rand(M, K, seed=5, scale=0.5)
    wg, wu = _rand(F, K, seed=6, scale=0.03), _rand(F, K, seed=7, scale=0.03)
    wgu = reference.interleave_gate_up(wg, wu).contiguous()
    out = hip.gemm(x, wgu, swiglu=True)
    torch.cuda.synchronize()
    g, u = x.float() @ wg.float().t(), x.float() @ wu.float().t()
    _check(out, torch.nn.functional.silu(g) * u, tol=3e-2)


@pytest.mark.parametrize("M,N,K", [(77, 1280, 8192), (2049, 7168, 8192), (513, 16032, 1024)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_gemm_fp8(M, N, K, swiglu):
    x = _rand(M, K, seed=8, scale=0.5, offset=0.02)
    w = Fp8Weight.quantize(_rand(N, K, seed=9, scale=0.02))
    xq, xs = hip.quant_fp8_rows(x)
    out = hip.gemm_fp8(xq, xs, w, swiglu=swiglu)
    torch.cuda.synchronize()
    xd = xq.float() * xs[:, None]
    ref = xd @ w.dequant().t()
    if swiglu:
        g = (xd @ w.dequant().t()).reshape(M, -1, 2, 8)
        ref = (torch.nn.functional.silu(g[:, :, 0]) * g[:, :, 1]).reshape(M, -1)
    _check(out, ref, tol=3e-2)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("aligned", [True, False])
def test_gemm_mfma32_variant(fp8, swiglu, aligned):
    """The 32x32-MFMA tile variant (group_m bit 8) of the 8-bit GEMM against fp32, ragged M and an N % 32 == 16 tail; bf16 has one
    form of tile and gives the bits of a call without it."""
    M, N, K = 777, 1040 if not swiglu else 1056, 1024
    x = _rand(M, K, seed=10, scale=0.5, offset=0.02)
    wb = _rand(N, K, seed=11, scale=0.03, offset=0.001)
    n_out = N // 2 if swiglu else N
    big = torch.zeros(M, n_out + 8, dtype=torch.bfloat16, device=DEV)
    out = big[:, :n_out] if aligned else big[:, 4:4 + n_out]
    if fp8:
        w = Fp8Weight.quantize(wb)
        xq, xs = hip.quant_fp8_rows(x)
        hip.gemm_fp8(xq, xs, w, out=out, swiglu=swiglu, group_m=4 | 256)
        y = (xq.float() * xs[:, None]) @ w.dequant().t()
    else:
        hip.gemm(x, wb, out=out, swiglu=swiglu, group_m=4 | 256)
        assert torch.equal(out, hip.gemm(x, wb, swiglu=swiglu, group_m=4))
        y = x.float() @ wb.float().t()
    torch.cuda.synchronize()
    if swiglu:
        g = y.reshape(M, -1, 2, 8)
        y = (torch.nn.functional.silu(g[:, :, 0]) * g[:, :, 1]).reshape(M, -1)
    _check(out, y, tol=3e-2)


def test_gemm_graph_capture():
    x, w = _rand(512, 1024, seed=10), _rand(768, 1024, seed=11, scale=0.05)
    out = torch.empty(512, 768, dtype=torch.bfloat16, device=DEV)
    hip.gemm(x, w, out=out)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        hip.gemm(x, w, out=out)
    out.zero_()
    g.replay()
    torch.cuda.synchronize()
    _check(out, x.float() @ w.float().t())


@pytest.mark.parametrize("M,N,K", [(1, 32, 2048), (130, 544, 2112), (257, 4096, 2112), (4097, 4096, 2048),
                                   (3300, 2560, 12288)])
@pytest.mark.parametrize("epi", ["bf16", "swiglu", "gelu", "f32"])
def test_gemm_split_tail(M, N, K, epi):
    """Tiles behind the last whole round run in slices of K that a second launch adds: one tile of one row, a ragged
    last slice, few tiles, 16 sliced tiles behind a whole round, and two rounds of thirds; repeated calls are the same bits."""
    assert hip.gemm_splits(M, N, K // 64)[1] > 1
    x, w = _rand(M, K, seed=12, scale=0.5, offset=0.02), _rand(N, K, seed=13, scale=0.03, offset=0.001)
    if epi == "swiglu":
        w[-16:] *= 2
    kw = {} if epi == "bf16" else {epi: True}
    out = hip.gemm(x, w, **kw)
    assert torch.equal(out, hip.gemm(x, w, **kw))
    y = x.double() @ w.double().t()
    if epi == "f32":
        # each of the K products and sums rounds by at most 2^-24 of the sum of magnitudes
        bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
        assert out.dtype == torch.float32 and bool(((out.double() - y).abs() <= bound).all())
        return
    if epi == "swiglu":
        g = y.reshape(M, -1, 2, 8)
        y = (torch.nn.functional.silu(g[:, :, 0]) * g[:, :, 1]).reshape(M, -1)
    elif epi == "gelu":
        y = torch.nn.functional.gelu(y, approximate="tanh")
    # one bf16 rounding (2^-9 relative) behind fp32 sums; the activations' fp32 exponentials add far less
    assert bool(((out.double() - y).abs() <= 2.0 ** -8 * y.abs() + 1e-4).all())


@pytest.mark.parametrize("K", [64, 128, 192, 384, 704])
@pytest.mark.parametrize("epi", ["bf16", "swiglu", "gelu", "f32"])
@pytest.mark.parametrize("off", [0, 4])
def test_gemm_tile_after_tile(K, epi, off):
    """More tiles than CUs, so that requests run on into the next tile: K-tiles from one (a tile per workgroup) over two
    (every request past the tile's own) to more than the ring's images, ragged last rows and columns, into columns of
    wider rows, 16-byte aligned (counted stores) and not."""
    M, N = 4100, 4128
    x, w = _rand(M, K, seed=22, scale=0.5, offset=0.02), _rand(N, K, seed=23, scale=0.05, offset=0.001)
    n, dtype = N // 2 if epi == "swiglu" else N, torch.float32 if epi == "f32" else torch.bfloat16
    rows = torch.full((M, n + 16), 7.0, dtype=dtype, device=DEV)
    out = rows[:, off:off + n]
    for _ in range(2):
        hip.gemm(x, w, out=out, **({} if epi == "bf16" else {epi: True}))
    y = x.double() @ w.double().t()
    slack = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    if epi == "swiglu":
        h, e = y.reshape(M, -1, 2, 8), slack.reshape(M, -1, 2, 8)
        y = (torch.nn.functional.silu(h[:, :, 0]) * h[:, :, 1]).reshape(M, -1)
        slack = (1.1 * e[:, :, 0] * h[:, :, 1].abs() + h[:, :, 0].abs() * e[:, :, 1]).reshape(M, -1)  # |silu'| <= 1.1
    elif epi == "gelu":
        y, slack = torch.nn.functional.gelu(y, approximate="tanh"), 1.2 * slack + 1e-5  # |gelu'| < 1.2; its fp32 exponential
    # sums of K exact products in fp32, then one bf16 rounding
    assert bool(((out.double() - y).abs() <= (0 if epi == "f32" else 2.0 ** -8) * y.abs() + slack).all())
    assert bool((rows[:, :off] == 7).all() and (rows[:, off + n:] == 7).all())


@pytest.mark.parametrize("M,N,K,two", [(1, 48, 4096, False), (300, 1040, 4224, False), (257, 528, 2176, True), (4097, 4096, 4096, False),
                                       (2100, 4096, 12288, True)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_gemm_fp8_split_tail(M, N, K, two, swiglu):
    """The 8-bit product in slices of K, row and column scales behind the added slices; a slice border inside the low term of
    two-term rows and between the terms."""
    g = torch.Generator().manual_seed(18)
    f8 = lambda *s: (torch.randn(*s, generator=g) * 8).to(torch.float8_e4m3fn)  # noqa: E731
    xq, w = f8(M, (2 if two else 1) * K), Fp8Weight(f8(N, K).to(DEV), (torch.rand(N, generator=g) / 64 + 1 / 64).to(DEV))
    xs = (torch.rand(M, generator=g) + 0.5) / K ** 0.5 / 8
    n0 = N // 32 * 32 if swiglu else N
    kb = (2 if two else 1) * K // 128
    splits = hip.gemm_splits_fp8(M, n0, kb)[1]
    assert splits > 1 and (not two or any(kb // 2 < kb * i // splits for i in range(splits)))
    w = Fp8Weight(w.q[:n0].contiguous(), w.scale[:n0].contiguous())
    out = hip.gemm_fp8(xq.to(DEV), xs.to(DEV), w, swiglu=swiglu, group_m=hip.GEMM_GROUP_M)
    assert torch.equal(out, hip.gemm_fp8(xq.to(DEV), xs.to(DEV), w, swiglu=swiglu, group_m=hip.GEMM_GROUP_M))
    x = xq.to(DEV).double()
    x = (x[:, :K] + x[:, K:] / 16 if two else x) * xs.to(DEV).double()[:, None]
    wd = w.q.double() * w.scale.double()[:, None]
    y = x @ wd.t()
    # sums of K exact products in fp32 (a few roundings of 2^-24 of the largest partial sum each), one bf16 rounding
    slack = K * 2.0 ** -24 * (x.abs() @ wd.abs().t())
    if swiglu:
        h, e = y.reshape(M, -1, 2, 8), slack.reshape(M, -1, 2, 8)
        gate, up = h[:, :, 0], h[:, :, 1]
        y = (torch.nn.functional.silu(gate) * up).reshape(M, -1)
        slack = (1.1 * e[:, :, 0] * up.abs() + gate.abs() * e[:, :, 1]).reshape(M, -1)  # |silu'| <= 1.1, |silu| <= |gate|
    assert bool(((out.double() - y).abs() <= 2.0 ** -8 * y.abs() + slack).all())


@pytest.mark.parametrize("epi", ["bf16", "swiglu", "gelu", "f32"])
def test_gemm_split_tail_strided(epi):
    """Slices of K into columns of wider rows, as whole tiles write them."""
    M, N, K = 300, 544, 2048
    assert hip.gemm_splits(M, N, K // 64)[1] > 1
    big, w = _rand(M, K + 64, seed=20, scale=0.5), _rand(N, K, seed=21, scale=0.03)
    x, n = big[:, 32:32 + K], N // 2 if epi == "swiglu" else N
    kw = {} if epi == "bf16" else {epi: True}
    want = hip.gemm(x.contiguous(), w, **kw)
    for off in (0, 4):
        rows = torch.full((M, n + 16), 7.0, dtype=want.dtype, device=DEV)
        hip.gemm(x, w, out=rows[:, off:off + n], **kw)
        assert torch.equal(rows[:, off:off + n], want)
        assert bool((rows[:, :off] == 7).all() and (rows[:, off + n:] == 7).all())


@pytest.mark.parametrize("K", [64, 2048])
def test_gemm_swiglu_small_gates(K):
    """sigmoid(gate) below the smallest normal number (gates under -87.3) times a large up value, one launch (K 64) and
    slices of K (2048): the quotient gate / (1 + e^-gate) is a normal number and must not become 0."""
    gate = torch.tensor([-86.0, -87.0, -88.0, -88.5], dtype=torch.float64)
    x, w = torch.zeros(4, K, dtype=torch.bfloat16), torch.zeros(32, K, dtype=torch.bfloat16)
    x[range(4), range(4)] = 1
    w[:, :4] = torch.where(torch.arange(32)[:, None] % 16 < 8, gate, torch.tensor(2.0 ** 100, dtype=torch.float64))
    out = hip.gemm(x.to(DEV), w.to(DEV), swiglu=True).cpu().double()
    want = (gate / (1 + torch.exp(-gate)) * 2.0 ** 100)[:, None].expand(4, 16)
    # one bf16 rounding (2^-9); the fp32 exponential of 88 is good to 88 * 2^-23
    assert bool(((out - want).abs() <= 2.0 ** -8 * want.abs()).all())


@pytest.mark.parametrize("K", [64, 2048])
@pytest.mark.parametrize("up", [2.0 ** 100, 1.0])
def test_gemm_swiglu_tiny_gates(K, up):
    """Gates of 2^-90 to 2^-126, whose half is the product with sigmoid(gate) = 1/2, in one launch (K 64) and in slices of K
    (2048): exact in fp32 down to the smallest normal number, and no scaling on the way may lose bits of it."""
    assert (hip.gemm_splits(8, 32, K // 64)[1] > 1) == (K == 2048)
    gate = torch.tensor([s * f * 2.0 ** -e for e in (90, 100, 110, 125) for s, f in ((1, 1.0), (-1, 1.9921875))], dtype=torch.float64)
    x, w = torch.zeros(8, K, dtype=torch.bfloat16), torch.zeros(32, K, dtype=torch.bfloat16)
    x[range(8), range(8)] = 1
    w[:, :8] = torch.where(torch.arange(32)[:, None] % 16 < 8, gate, torch.tensor(up, dtype=torch.float64))
    out = hip.gemm(x.to(DEV), w.to(DEV), swiglu=True).cpu().double()
    # gate, up and half their product have 8 bits: nothing rounds
    assert torch.equal(out, (gate / 2 * up)[:, None].expand(8, 16))


@pytest.mark.parametrize("M", [128, 129, 256, 257])
def test_stream_parts_beyond_tall_tiles(M):
    """linear_parts gives the slabs it is asked for at any row count; consumers that add however many there are get one
    fp32 slab of the tile GEMM above the stream kernel's tallest x tile."""
    x, w = _rand(M, 1024, seed=14, scale=0.5), _rand(4096, 1024, seed=15, scale=0.03)
    bound = 1024 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    for parts, n in ((hip.linear_parts(x, w, 2, nt=4, kernel="stream"), 2), (hip.stream_slabs(x, w, 2, 4), 2 if M <= 128 else 1)):
        assert parts.dtype == torch.float32 and parts.shape == (n, M, 4096)
        assert bool(((parts.sum(0).double() - x.double() @ w.double().t()).abs() <= bound).all())


@pytest.mark.parametrize("M,N,K", [(1, 32, 2048), (130, 544, 2112), (257, 4096, 2112), (3300, 2560, 12288)])
def test_gemm_slabs(M, N, K):
    """A grid whose tiles all run in slices of K leaves the slices apart; other grids give none."""
    x, w = _rand(M, K, seed=16, scale=0.5), _rand(N, K, seed=17, scale=0.03)
    parts = hip.gemm_slabs(x, w)
    assert parts.shape == (hip.gemm_splits(M, N, K // 64)[1], M, N) and parts.dtype == torch.float32
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert bool(((parts.double().sum(0) - x.double() @ w.double().t()).abs() <= bound).all())
    assert hip.gemm_slabs(x[:, :64], w[:, :64]) is None and hip.gemm_slabs(_rand(4097, K), _rand(4096, K)) is None


@pytest.mark.parametrize("M,N,K", [(1967, 4096, 4096), (2400, 4096, 14336), (1569, 4096, 4096), (2048, 4096, 4096)])
def test_gemm_slabs_of_whole_tiles(M, N, K):
    """Row counts whose lower tiles run whole: consumers of slabs still get the product in fp32, as one slab."""
    from llm_map_reduce_summarizer_amd import ops
    assert hip.gemm_splits(M, N, K // 64)[1] == 1 and hip.gemm_splits_fp8(M, N, K // 64)[1] > 1
    x, w = _rand(M, K, seed=28, scale=0.5), _rand(N, K, seed=29, scale=0.03)
    parts = ops.project(x, w, "o")
    assert parts.shape == (1, M, N) and parts.dtype == torch.float32
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())  # fp32 sums of K exact products
    assert bool(((parts[0].double() - x.double() @ w.double().t()).abs() <= bound).all())


@pytest.mark.parametrize("rows", [128, 160, 192, 224])
@pytest.mark.parametrize("epi", ["bf16", "swiglu", "gelu", "f32"])
@pytest.mark.parametrize("M,N,K,splits", [(1, 32, 64, 1), (129, 288, 128, 1), (449, 544, 704, 3), (4100, 4128, 192, 1), (4100, 4128, 320, 1)])
def test_gemm_tile_rows(monkeypatch, rows, epi, M, N, K, splits):
    """Tiles of fewer rows than 256: one K-tile and two (past the end of which the loop asks for nothing that is read), ragged
    rows and columns, slices of K, and tile after tile with few and more K-tiles.  Whole tiles add a row's products in the
    same order at every height, so they have the bits of 256 rows; slices are held to the bound of fp32 sums."""
    x, w = _rand(M, K, seed=24, scale=0.5, offset=0.02), _rand(N, K, seed=25, scale=0.05, offset=0.001)
    kw = {} if epi == "bf16" else {epi: True}

    def run(rows, splits):
        tiles = -(-M // rows) * -(-N // 256)
        whole = tiles if splits == 1 else 0
        monkeypatch.setattr(hip, "gemm_splits", lambda *_: (whole, splits, (tiles - whole) * splits * rows * 256, rows))
        return hip.gemm(x, w, **kw)
    want, got = run(256, 1), run(rows, splits)
    assert torch.equal(got, run(rows, splits))
    if splits == 1:
        assert torch.equal(got, want)
    else:
        # fp32 sums of K exact products, either way off by at most K 2^-24 of the sum of magnitudes; gate and up (|silu'| <=
        # 1.1) or gelu (< 1.2) pass that on; then one bf16 rounding each
        slack = 2.4 * K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
        if epi == "swiglu":
            h, e = (x.double() @ w.double().t()).reshape(M, -1, 2, 8).abs(), slack.reshape(M, -1, 2, 8)
            slack = (e[:, :, 0] * h[:, :, 1] + h[:, :, 0] * e[:, :, 1]).reshape(M, -1)
        rounding = 0 if epi == "f32" else 2.0 ** -7
        assert bool(((got.double() - want.double()).abs() <= rounding * want.double().abs() + slack + 1e-30).all())


@pytest.mark.parametrize("M", [1, 100, 129, 300, 522, 903, 2000, 7615])
@pytest.mark.parametrize("N,K", [(32, 64), (1536, 4096), (4096, 22528), (28672, 4096)])
def test_gemm_plan_is_one_the_kernel_takes(M, N, K):
    whole, splits, room, rows = hip.gemm_splits(M, N, K // 64)
    tiles = -(-M // rows) * -(-N // 256)
    assert rows in (128, 160, 192, 224, 256) and splits >= 1 and room == (tiles - whole) * splits * rows * 256
    assert whole == tiles if splits == 1 else 0 <= whole < tiles and whole % hip.N_CU == 0 and K // 64 // splits >= 4


@pytest.mark.parametrize("M", [64, 65, 128, 129])
@pytest.mark.parametrize("N", [48896, 49152, 65536, 65792])
def test_lm_heads_of_65_to_128_rows(M, N):
    """``linear`` and ``logits32`` on both sides of the row counts and widths at which the tile GEMM takes over."""
    x, w = _rand(M, 256, seed=26, scale=0.5), _rand(N, 256, seed=27, scale=0.05)
    y = x.double() @ w.double().t()
    slack = 256 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())  # fp32 sums; bf16 results round once
    assert bool(((hip.linear(x, w).double() - y).abs() <= 2.0 ** -8 * y.abs() + slack).all())
    got = hip.logits32(x, w)
    assert got.dtype == torch.float32 and bool(((got.double() - y).abs() <= slack).all())
