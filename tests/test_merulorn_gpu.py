"""The Merulorn design on the MI355X kernels against its float64 oracle (tests/merulorn_oracle.py): every mechanism
alone, then whole models in bf16 and fp32 through the engine's step function, scheduler and captured decode graphs."""
import pytest
import torch

import merulorn_cases as M
import merulorn_oracle as O

pytestmark = pytest.mark.gpu
BF, F32, DEV = torch.bfloat16, torch.float32, "cuda:0"
DTYPES = [BF, F32]


def rnd(*shape, seed=0, std=1.0, dtype=F32):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * std).to(dtype)


def dev(t, dtype=None):
    return t.to(device=DEV, dtype=dtype or t.dtype).contiguous()


def rel(got, want):
    want = want.double()
    return float((got.double().cpu() - want).pow(2).mean().sqrt() / want.pow(2).mean().sqrt())


def forms(u):
    """A projection result [T, N] in the forms its consumers take: (source, compute dtype, the values it holds)."""
    b = u.to(BF)
    k = rnd(3, *u.shape, seed=99, std=0.3)
    slabs = torch.stack([k[0], k[1], u - k[0] - k[1]])
    return [(dev(b), BF, b.double()), (dev(slabs), BF, slabs.double().sum(0)), (dev(u)[None].contiguous(), F32, u.double())]


def segments(lens, slots, pos0):
    from llm_map_reduce_summarizer_amd import ops
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    rows = [i for i, n in enumerate(lens) for _ in range(n)]
    return ops.Segments(i32(slots), i32(pos0), i32(cu), i32(rows), lens)


# ------------------------------------------------------------------ mechanisms
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [64, 51])
def test_embedding_and_positions(dtype, width):
    from llm_map_reduce_summarizer_amd import ops
    table = rnd(40, width, dtype=BF)
    freq = (10000.0 ** (-torch.arange(0, width + width % 2, 2, dtype=torch.float64) / width)).to(DEV)
    for start in (0, 1000, 120000):
        ids = [3, 39, 0, 17]
        pos = torch.arange(start, start + 4, dtype=torch.int32, device=DEV)
        got = ops.embed_pos(torch.tensor(ids, dtype=torch.int32, device=DEV), pos, dev(table, dtype), 5.0, freq)
        want = O.embed(ids, table.double(), 5.0, start)
        assert float((got.double().cpu() - want).abs().max()) < 2e-6


@pytest.mark.parametrize("D", [96, 50, 5120])
def test_residual_norm(D):
    from llm_map_reduce_summarizer_amd import ops
    r0, w = rnd(7, D), rnd(D, seed=1)
    for src, dt, vals in forms(rnd(7, D + (-D) % 16, seed=2)):
        r = dev(r0.clone())
        out = ops.add_norm32(r, src, dev(1 + w), 1e-4, dt, D + (-D) % 128)
        want_r = r0.double() + vals[:, :D]
        assert rel(r, want_r) < 1e-6
        assert rel(out[:, :D], O.one_plus_norm(want_r, w.double(), 1e-4)) < (4e-3 if dt == BF else 1e-6)
        assert not out[:, D:].any()


def test_clamped_glu_epilogues():
    """The clamped GLU in the epilogues of the GEMM kernels every row count takes, and the 32-bit kernel."""
    from llm_map_reduce_summarizer_amd import ops
    from llm_map_reduce_summarizer_amd.ops.reference import interleave_gate_up
    for F, K in ((128, 128), (3584, 512), (14336, 256)):
        g, u = rnd(F, K, std=3 * K ** -0.5, dtype=BF), rnd(F, K, seed=1, std=3 * K ** -0.5, dtype=BF)
        w = dev(interleave_gate_up(g, u))
        for T in (1, 5, 20, 40, 100, 300):
            x = rnd(T, K, seed=T, dtype=BF)
            want = O.clamped_glu(x.double() @ g.double().T, x.double() @ u.double().T, 1.25)
            assert rel(ops.project_glu(dev(x), w, 1.25, 1.702, 1.0), want) < 4e-3, (F, T)
        got = ops.project_glu(dev(x, F32), w.float(), 1.25, 1.702, 1.0)
        assert rel(got, want) < 1e-5


@pytest.mark.parametrize("taps", [1, 2, 4, 5])
def test_short_convolution(taps):
    from llm_map_reduce_summarizer_amd import ops
    C, at = 40, 16
    kern, bias = rnd(C, taps, std=0.5), rnd(C, seed=1)
    lens = [1, 1, 70, 2, 3]
    for k, (src, dt, vals) in enumerate(forms(rnd(sum(lens), 72, seed=3))):
        x = vals[:, at: at + C]
        x = x.to(BF).double() if dt == BF else x
        hist = rnd(len(lens), max(1, taps - 1), C, seed=5, dtype=BF)  # what slots hold before
        state = torch.full((9, max(1, taps - 1), C), 1e3, device=DEV)
        slots, pos0 = [4, 2, 7, 1, 3], [5, 0, 0, 900, 64]
        for i, s in enumerate(slots):
            if pos0[i]:
                state[s] = hist[i].to(DEV)
        got = ops.conv_silu(src, at, dev(kern.t().contiguous()), dev(bias), state, segments(lens, slots, pos0), dt)
        b = 0
        for i, n in enumerate(lens):
            h = hist[i, : taps - 1].double() if pos0[i] else torch.zeros(taps - 1, C, dtype=torch.float64)
            full = torch.cat([h, x[b: b + n]])
            want = O.silu(O.short_conv(full, kern.double(), bias.double()))[taps - 1:]
            assert rel(got[b: b + n], want) < (4e-3 if dt == BF else 1e-6), (k, i)
            if taps > 1:
                assert rel(state[slots[i]], full[-(taps - 1):]) < 1e-6
            b += n
        # one row per segment: the step form
        st = torch.full((9, max(1, taps - 1), C), 1e3, device=DEV)
        st[4] = hist[0].to(DEV)
        one = ops.Segments(torch.tensor([4, 2], dtype=torch.int32, device=DEV),
                           torch.tensor([5, 0], dtype=torch.int32, device=DEV))
        cut = src[:, :2].contiguous() if src.dim() == 3 else src[:2].contiguous()
        y = ops.conv_silu(cut, at, dev(kern.t().contiguous()), dev(bias), st, one, dt)
        assert torch.equal(y, got[:2])
        if taps > 1:
            assert torch.equal(st[[4, 2]], state[[4, 2]])


SCANS = [(3, 64, 128, 1), (4, 24, 40, 2), (2, 128, 64, 2), (2, 40, 200, 1), (5, 7, 5, 5), (2, 136, 260, 1), (6, 16, 16, 3)]


@pytest.mark.parametrize("heads,P,N,groups", SCANS)
@pytest.mark.parametrize("dtype", DTYPES)
def test_state_space_scan(heads, P, N, groups, dtype):
    """Decoded rows, short and long portions (long enough that few heads are cut into runs), fresh and continued
    slots holding garbage or carried state; then the same rows once more from the state the first half left."""
    from llm_map_reduce_summarizer_amd import ops
    C = heads * P + 2 * groups * N
    Cp = C + (-C) % 8
    lens = [1, 1, 2, 65, 700 if heads == 3 else 130]
    T = sum(lens)
    xbc = torch.zeros(T, Cp)
    xbc[:, :C] = rnd(T, C, std=0.7)
    xbc = xbc.to(dtype)
    u = rnd(T, 16, seed=1)
    dt_bias, A_log, D = rnd(heads, seed=2, std=1.5) - 2, rnd(heads, seed=3, std=1.5), rnd(heads, seed=4)
    slots, pos0 = [3, 1, 5, 2, 6], [9, 0, 7, 64, 0]
    init = rnd(len(lens), heads, P, N, seed=6, std=0.5)
    N4 = N + (-N) % 4
    for src, dt_, vals in forms(u):
        if dt_ != dtype:
            continue
        state = torch.full((8, heads, P, N4), 1e4, device=DEV)
        state[..., N:] = 0
        for i, s in enumerate(slots):
            if pos0[i]:
                state[s, ..., :N] = init[i].to(DEV)
        args = (dev(dt_bias), dev(-torch.exp(A_log)), dev(D), state)
        y = ops.ssm_scan(dev(xbc), src, 8, *args, segments(lens, slots, pos0), heads, P, N, groups)
        f = xbc.double()
        b = 0
        for i, n in enumerate(lens):
            x, Bm, Cm = f[b: b + n, :heads * P], f[b: b + n, heads * P: heads * P + groups * N], f[b: b + n, C - groups * N: C]
            dts = O.softplus(vals[b: b + n, 8: 8 + heads] + dt_bias.double())
            want, S = scan_with_state(x.view(n, heads, P), Bm.view(n, groups, N), Cm.view(n, groups, N), dts,
                                      A_log.double(), D.double(), groups, init[i].double() if pos0[i] else None)
            tol = 3e-5 if dtype == BF else 3e-6
            assert rel(y[b: b + n], want.reshape(n, -1)) < tol, ("y", i)
            assert rel(state[slots[i], ..., :N], S) < tol, ("state", i)
            b += n


@pytest.mark.parametrize("heads,P,N,lens", [(3, 40, 200, [65, 700]), (96, 8, 104, [512] * 4), (97, 8, 104, [512] * 4)])
def test_state_space_runs_without_a_scanning_wave(heads, P, N, lens):
    """Segments cut into runs where the state pass has four waves: states above 128, and 768 workgroups (which have five) and more."""
    from llm_map_reduce_summarizer_amd import ops
    from llm_map_reduce_summarizer_amd.ops import hip
    items, runs = hip.ssm_runs(lens, 0, heads)
    assert runs is not None and (heads == 3 or (len(items) * heads > 768) == (heads == 97))
    T, C = sum(lens), heads * P + 2 * N
    xbc, u = rnd(T, C, std=0.7).to(BF), rnd(T, heads + 8 - heads % 8, seed=1).to(BF)
    dt_bias, A_log, D = rnd(heads, seed=2, std=1.5) - 2, rnd(heads, seed=3, std=1.5), rnd(heads, seed=4)
    slots, pos0 = list(range(len(lens))), [7 * (i % 2) for i in range(len(lens))]
    init = rnd(len(lens), heads, P, N, seed=6, std=0.5)
    state = dev(init.clone())
    y = ops.ssm_scan(dev(xbc), dev(u), 0, dev(dt_bias), dev(-torch.exp(A_log)), dev(D), state, segments(lens, slots, pos0), heads, P,
                     N, 1).view(T, heads, P)
    f, some, b = xbc.double(), [0, heads // 2, heads - 1], 0
    for i, n in enumerate(lens):
        x, Bm, Cm = f[b: b + n, :heads * P].view(n, heads, P)[:, some], f[b: b + n, heads * P: heads * P + N], f[b: b + n, C - N:]
        dts = O.softplus(u[b: b + n, :heads].double() + dt_bias.double())[:, some]
        want, S = scan_with_state(x, Bm.view(n, 1, N), Cm.view(n, 1, N), dts, A_log[some].double(), D[some].double(), 1,
                                  init[i, some].double() if pos0[i] else None)
        # two terms of bf16 for everything that is not one, as above
        assert rel(y[b: b + n, some], want) < 3e-5 and rel(state[i, some], S) < 3e-5, i
        b += n


@pytest.mark.parametrize("copies,dtype,N,rows", [(1, F32, 24, 1), (2, F32, 24, 2), (4, F32, 7, 4), (2, F32, 128, 2), (4, F32, 128, 4),
                                                 (2, F32, 200, 2), (1, BF, 260 - 12, 4)])
def test_state_space_portions_token_by_token(copies, dtype, N, rows):
    """Portions around the 16 rows that the stepped kernel stages at a time, and the 16-bit head size that the chunked form
    does not take; ``rows`` state rows per lane group: one up to 512 workgroups at one row each, two up to 1024, then four."""
    from llm_map_reduce_summarizer_amd import ops
    from llm_map_reduce_summarizer_amd.ops import hip
    heads, P, groups = 64, 20 if dtype == F32 else 136, 2
    one = -(-P // 16) * heads * 4 * copies
    assert rows == (1 if one <= 512 else 2 if one <= 1024 else 4)
    lens = [1, 15, 16, 17, 33] * copies
    assert not (dtype == BF and hip.ssm_chunk_ok(P, N))
    T, Cp = sum(lens), heads * P + 2 * groups * N + (-(2 * groups * N)) % 8
    lens.sort(key=lambda n: n != 1)
    xbc, u = rnd(T, Cp, std=0.7).to(dtype), rnd(1, T, heads, seed=1)
    vec = [rnd(heads, seed=2, std=1.5) - 2, -torch.exp(rnd(heads, seed=3)), rnd(heads, seed=4)]
    slots, pos0 = list(range(1, len(lens) + 1)), [7 * (i % 2) for i in range(len(lens))]
    state = rnd(len(lens) + 1, heads, P, N + (-N) % 4, seed=5, std=0.5)
    state[..., N:] = 0
    got_s, want_s = dev(state), state.clone()
    segs = segments(lens, slots, pos0)
    got = ops.ssm_scan(dev(xbc), dev(u), 0, *map(dev, vec), got_s, segs, heads, P, N, groups)
    host = ops.Segments(segs.slots.cpu(), segs.pos0.cpu(), segs.cu.cpu(), segs.row_seg.cpu(), lens)
    want = ops.ssm_scan(xbc, u, 0, *vec, want_s, host, heads, P, N, groups)
    # both sides are fp32: a few roundings of 2^-24 a row, over up to 33 rows of a decaying state
    assert rel(got, want) < 3e-6 and rel(got_s, want_s) < 3e-6


@pytest.mark.parametrize("dtype,P,N", [(F32, 20, 24), (F32, 64, 128), (BF, 136, 248)])
def test_state_space_portions_total_decay(dtype, P, N):
    """A_log so large that -exp(A_log) is minus infinity: every row forgets the state before it, and the rows that pad a
    portion to the 16 that are staged at a time leave the last row's state alone."""
    from llm_map_reduce_summarizer_amd import ops
    heads, groups, lens = 3, 1, [1, 15, 16, 17]
    T, C = sum(lens), heads * P + 2 * groups * N
    xbc, u = rnd(T, C + (-C) % 8, std=0.7).to(dtype), rnd(1, T, 8, seed=1)
    A_log = torch.tensor([0.5, 89.0, 100.0])
    vec = [rnd(heads, seed=2), -torch.exp(A_log), rnd(heads, seed=4)]
    slots, pos0 = [2, 1, 4, 3], [5, 0, 9, 7]
    state = rnd(5, heads, P, N + (-N) % 4, seed=5, std=0.5)
    state[..., N:] = 0
    got_s, want_s = dev(state), state.clone()
    segs = segments(lens, slots, pos0)
    host = ops.Segments(segs.slots.cpu(), segs.pos0.cpu(), segs.cu.cpu(), segs.row_seg.cpu(), lens)
    got = ops.ssm_scan(dev(xbc), dev(u), 0, *map(dev, vec), got_s, segs, heads, P, N, groups)
    want = ops.ssm_scan(xbc, u, 0, *vec, want_s, host, heads, P, N, groups)
    assert bool(torch.isfinite(want).all() and torch.isfinite(want_s).all())
    # as above
    assert rel(got, want) < 3e-6 and rel(got_s, want_s) < 3e-6


@pytest.mark.parametrize("heads,P,N,groups", [(4, 64, 128, 2), (3, 20, 64, 1), (2, 40, 36, 2), (6, 32, 100, 3)])
@pytest.mark.parametrize("total", [False, True])
def test_state_space_chunks_of_fp32(heads, P, N, groups, total):
    """Portions around the 64 rows of a chunk, whole and partial blocks of value and state columns; ``total``: heads whose
    decay is total."""
    from llm_map_reduce_summarizer_amd import ops
    from llm_map_reduce_summarizer_amd.ops import hip
    lens = [1, 2, 63, 64, 65, 129]
    assert hip.ssm_chunk32_rows(lens[1:], heads, P)
    T, C = sum(lens), heads * P + 2 * groups * N
    xbc, u = rnd(T, C + (-C) % 8, std=0.7), rnd(1, T, 8, seed=1)
    A_log = rnd(heads, seed=3)
    if total:
        A_log[:2] = torch.tensor([89.0, 100.0])
    vec = [rnd(heads, seed=2, std=1.5) - 2, -torch.exp(A_log), rnd(heads, seed=4)]
    slots, pos0 = [2, 1, 4, 3, 6, 5], [5, 0, 9, 0, 7, 64]
    state = rnd(7, heads, P, N, seed=5, std=0.5)
    got_s, want_s = dev(state), state.clone()
    segs = segments(lens, slots, pos0)
    host = ops.Segments(segs.slots.cpu(), segs.pos0.cpu(), segs.cu.cpu(), segs.row_seg.cpu(), lens)
    got = ops.ssm_scan(dev(xbc), dev(u), 0, *map(dev, vec), got_s, segs, heads, P, N, groups)
    want = ops.ssm_scan(xbc, u, 0, *vec, want_s, host, heads, P, N, groups)
    # both sides are fp32: the reference rounds each of up to 129 rows of a decaying state, here sums of 64 rows and of N
    assert rel(got, want) < 3e-6 and rel(got_s, want_s) < 3e-6


@pytest.mark.parametrize("where", ["decay", "step"])
def test_state_space_chunks_of_fp32_keep_what_is_no_number(where):
    """A decay that is no number makes all of its head none, a step size that is none its row and those after it, as token by
    token."""
    from llm_map_reduce_summarizer_amd import ops
    from llm_map_reduce_summarizer_amd.ops import hip
    heads, P, N, groups, lens = 3, 32, 64, 1, [140, 70]
    assert hip.ssm_chunk32_rows(lens, heads, P)
    T, C = sum(lens), heads * P + 2 * groups * N
    xbc, u = rnd(T, C, std=0.7), rnd(1, T, 8, seed=1)
    vec = [rnd(heads, seed=2) - 2, -torch.exp(rnd(heads, seed=3)), rnd(heads, seed=4)]
    if where == "decay":
        vec[1][1] = float("nan")
    else:
        u[0, 77, 1] = float("nan")
    segs, state = segments(lens, [1, 0], [0, 0]), torch.zeros(2, heads, P, N, device=DEV)
    y = ops.ssm_scan(dev(xbc), dev(u), 0, *map(dev, vec), state, segs, heads, P, N, groups).view(T, heads, P).cpu()
    none, gone = torch.zeros(T, heads, P, dtype=torch.bool), torch.zeros(2, heads, P, N, dtype=torch.bool)
    if where == "decay":
        none[:, 1], gone[:, 1] = True, True
    else:
        none[77:140, 1], gone[1, 1] = True, True
    assert torch.equal(y.isnan(), none) and torch.equal(state.cpu().isnan(), gone)


@pytest.mark.parametrize("row,value", [(100, float("inf")), (64, float("nan")), (127, -float("inf"))])
def test_state_space_chunks_of_fp32_do_not_reach_back(row, value):
    """An input that is not finite leaves the rows before it, the other value columns and the other portions alone."""
    from llm_map_reduce_summarizer_amd import ops
    heads, P, N, groups, lens = 2, 64, 128, 1, [140, 140]
    T, C = sum(lens), heads * P + 2 * groups * N
    xbc, u = rnd(T, C, std=0.7), rnd(1, T, 8, seed=1)
    vec = [rnd(heads, seed=2) - 2, -torch.exp(rnd(heads, seed=3)), rnd(heads, seed=4)]
    segs = segments(lens, [1, 0], [0, 0])
    out = []
    for bad in (False, True):
        if bad:
            xbc[row, P + 9] = value
        state = torch.zeros(2, heads, P, N, device=DEV)
        out.append(ops.ssm_scan(dev(xbc), dev(u), 0, *map(dev, vec), state, segs, heads, P, N, groups).cpu())
        out.append(state.cpu())
    y, s, yb, sb = out
    after = torch.zeros(T, heads * P, dtype=torch.bool)
    after[row: lens[0], P + 9] = True
    assert not torch.isfinite(yb[after]).any() and torch.isfinite(yb[~after]).all()
    # the diagonal blocks of that chunk are summed in another order
    assert rel(yb[~after], y[~after]) < 1e-6
    hit = torch.zeros_like(s, dtype=torch.bool)
    hit[1, 1, 9] = True
    assert not torch.isfinite(sb[hit]).any() and torch.equal(sb[~hit], s[~hit])


def scan_with_state(x, B, C, dt, A_log, D, groups, S0):
    """The oracle's scan continued from S0 [heads, P, N]: the carried state as one more leading token is not possible,
    so its contribution decays beside the oracle's own output."""
    y = O.ssm_scan(x, B, C, dt, A_log, D, groups)
    heads = x.shape[1]
    S = torch.zeros(heads, x.shape[2], B.shape[2], dtype=torch.float64) if S0 is None else S0.clone()
    carried = S.clone()
    for t in range(x.shape[0]):
        for a in range(heads):
            g = a // (heads // groups)
            dec = torch.exp(-torch.exp(A_log[a]) * dt[t, a])
            carried[a] *= dec
            S[a] = dec * S[a] + dt[t, a] * torch.outer(x[t, a], B[t, g])
            y[t, a] += carried[a] @ C[t, g]
    return y, S


@pytest.mark.parametrize("n,groups", [(120, 5), (96, 2), (30, 3), (2048, 1), (2048, 8)])
def test_gated_group_norm(n, groups):
    from llm_map_reduce_summarizer_amd import ops
    T, zat, col, ld = 9, 8, 16, (n + 16 + 127) // 128 * 128
    y, w = rnd(T, n), rnd(n, seed=1) + 1
    for src, dt, vals in forms(rnd(T, zat + n + (-n) % 8, seed=2, std=2.0)):
        out = torch.full((T, ld), 3.0, dtype=dt, device=DEV)
        ops.gated_norm(dev(y), src, zat, dev(w), groups, 1e-3, 0.7, out, col)
        want = 0.7 * O.gated_group_norm(y.double(), vals[:, zat: zat + n], w.double(), groups, 1e-3)
        assert rel(out[:, col: col + n], want) < (4e-3 if dt == BF else 1e-6)
        assert (out[:, :col] == 3).all() and not out[:, col + n:].any()


@pytest.mark.parametrize("T,H,dim,C,taps", [(1, 8, 128, 24, 4), (5, 6, 40, 4 * 448, 4), (33, 8, 128, 4 * 1024 + 8, 4), (3, 64, 128, 64, 4),
                                            (2, 8, 128, 64, 3), (513, 2, 32, 40, 4)])
def test_convolution_beside_qkv(T, H, dim, C, taps, monkeypatch):
    """Decoded rows' convolution in the blocks behind those of q, k and v: less than one, whole and partial blocks a row; in a
    launch of its own beyond 8192 columns, 512 rows or at other than four taps.  The same bits either way."""
    from types import SimpleNamespace
    from llm_map_reduce_summarizer_amd import ops
    from llm_map_reduce_summarizer_amd.ops import hip
    G, page, i32 = 2, 64, dict(dtype=torch.int32, device=DEV)
    spec = SimpleNamespace(heads=H, kv_heads=G, dim=dim, vdim=dim, q_temp=None, head_gate=True)
    al = SimpleNamespace(spec=spec, q=0, k=H * dim, v=(H + G) * dim, g=(H + 2 * G) * dim, dk=dim, dv=dim)
    at = al.g + -(-H // 8) * 8
    u = rnd(T, at + C, std=0.5)
    bias, kernel, cb = rnd(at + C, seed=2), rnd(taps, C, seed=3), rnd(C, seed=4)
    one = (torch.arange(T, **i32), torch.arange(T, **i32), torch.arange(1, T + 1, **i32)[:, None].contiguous())
    pos = one[0] % page
    segs = ops.Segments(torch.arange(T, **i32).flip(0).contiguous(), pos)
    calls, plain = [], hip.conv_silu
    monkeypatch.setattr(hip, "conv_silu", lambda *a, **k: calls.append(1) or plain(*a, **k))
    for src, dt, _ in forms(u):
        got = []
        for beside in (False, True):
            state = dev(rnd(T, taps - 1, C, seed=5))
            kc, vc = (torch.zeros(T + 1, G, page, dim, dtype=dt, device=DEV) for _ in range(2))
            conv = (at, dev(kernel), dev(cb), state, segs)
            calls.clear()
            q, gate, *rows = ops.qkv_prep(src, al, dev(bias), None, None, 1e-5, 1.0, pos, one[1], one[2], kc, vc, page, dt,
                                          conv if beside else None)
            if not beside:
                rows = [ops.conv_silu(src, *conv, dt)]
            else:
                assert len(calls) == (0 if taps == 4 and T <= 512 and H * dim <= 4096 else 1)
            got.append((q, gate, kc, vc, rows[0], state))
        assert all(torch.equal(x, y) for x, y in zip(*got))


ATTN = [(8, 2, 128, 128), (6, 2, 40, 56), (4, 4, 64, 96), (16, 1, 96, 128), (10, 2, 24, 16), (2, 1, 136, 200)]


@pytest.mark.parametrize("H,G,dim,vdim", ATTN)
@pytest.mark.parametrize("dtype", DTYPES)
def test_attention_finds_the_key_that_stands_out(H, G, dim, vdim, dtype):
    """q / k / v preparation and attention (prompt portions and decoded tokens) over a paged cache whose unused rows
    hold large garbage: for chosen queries one far key, page-border key, the first key or the query's own key carries
    the score, the rest of the weight is spread over hundreds of keys."""
    from llm_map_reduce_summarizer_amd import ops
    from llm_map_reduce_summarizer_amd.engine.config import AttnSpec, HybridConfig, LayerSpec
    from llm_map_reduce_summarizer_amd.engine.hybrid import HybridModel
    scale, coef, every, eps = dim ** -0.5, 0.3, 17.0, 1e-5
    spec = AttnSpec(H, G, dim, vdim, scale, (coef, every))
    model = HybridModel(HybridConfig("t", 32, 64, (LayerSpec(spec),)), torch.device(DEV), dtype)
    la = model.layers[0]
    al = la.attn
    lens = [300, 97, 64, 65, 1]
    w = {n: rnd(r, 64, seed=i, std=0.125) for i, (n, r) in enumerate(
        (("q", H * dim), ("k", G * dim), ("v", G * vdim), ("g", H)))}
    w = {"a." + k: v.to(BF).double() for k, v in w.items()}
    for i, (n, r) in enumerate((("q", H * dim), ("k", G * dim), ("v", G * vdim))):
        w["a.%s.b" % n] = rnd(r, seed=20 + i, std=0.1).double()
    w["a.q.norm"], w["a.k.norm"] = rnd(H * dim, seed=30).double() * 0.1 + 1, rnd(G * dim, seed=31).double() * 0.1 + 1
    w["a.o"] = torch.eye(H * vdim, dtype=torch.float64)
    page, npg = 64, 40
    kc = torch.full((npg, G, page, al.dk), 30.0, dtype=dtype, device=DEV)
    vc = torch.full((npg, G, page, al.dv), -50.0, dtype=dtype, device=DEV)
    tables = torch.zeros(len(lens), 8, dtype=torch.int32)
    perm, at = (torch.randperm(npg - 1, generator=torch.Generator().manual_seed(1)) + 1).tolist(), 0
    us, wants, tok = [], [], []
    for s, n in enumerate(lens):
        need = -(-n // page)
        tables[s, :need] = torch.tensor(perm[at: at + need], dtype=torch.int32)
        at += need
        u = torch.zeros(n, la.n_in, dtype=torch.float64)
        h = rnd(n, 64, seed=40 + s, dtype=BF).double()
        for n_, c in (("q", al.q), ("k", al.k), ("v", al.v), ("g", al.g)):
            r = h @ w["a." + n_].T
            u[:, c: c + r.shape[1]] = r
        # the projection of query row t is steered onto the key row it should find
        pairs = [(t, j) for t, j in ((n - 1, 0), (n - 1 - n // 3, 63), (n // 2, n // 2), (n - 2, 64), (n // 3, 1))
                 if 0 <= j <= t < n]
        for t, j in pairs:
            k = u[j, al.k: al.k + G * dim].view(G, 1, dim).expand(G, H // G, dim).reshape(-1)
            u[t, al.q: al.q + H * dim] = 6.0 * k
        us.append(u)
        tok.append(pairs)
    uall = torch.cat(us).float()
    pos = torch.cat([torch.arange(n) for n in lens]).int().to(DEV)
    seq = torch.cat([torch.full((n,), s) for s, n in enumerate(lens)]).int().to(DEV)
    for src, dt, vals in forms(uall):
        if dt != dtype:
            continue
        b, wants = 0, []
        for n in lens:
            wants.append(attention_of(vals[b: b + n], w, al, H, G, dim, vdim, scale, coef, every, eps))
            b += n
        want = torch.cat(wants)
        bias = torch.zeros(la.n_in)
        for n_, c in (("q", al.q), ("k", al.k), ("v", al.v)):
            bias[c: c + w["a.%s.b" % n_].numel()] = w["a.%s.b" % n_].float()
        q, gate = ops.qkv_prep(src, al, dev(bias), dev(w["a.q.norm"].float()), dev(w["a.k.norm"].float()), eps, 0.6,
                               pos, seq, tables.to(DEV), kc, vc, page, dtype)
        out = torch.full((len(pos), H * al.vp + 8), 7.0, dtype=dtype, device=DEV)
        tol = 1e-2 if dtype == BF else 1e-5

        def same(o, rows, what):
            o = o[:, :H * al.vp].reshape(-1, H, al.vp)[:, :, :vdim].reshape(o.shape[0], -1)
            for i, t in enumerate(rows):
                assert rel(o[i], 0.6 * want[t]) < tol, (what, t)
        allrows = list(range(len(pos)))
        last = [sum(lens[:s + 1]) - 1 for s in range(len(lens))]
        if not al.mfma:
            ops.attn_rows(q, kc, vc, pos, seq, tables.to(DEV), H, G, al.vp, page, scale, gate, out)
            same(out, allrows, "rows")
            assert (out[:, H * al.vp:] == 7).all()
            continue
        # the last portions of the prompts: everything, then only rows from an odd place on
        for pre in ([0] * len(lens), [101, 64, 62, 1, 0]):
            part = [n - p for n, p in zip(lens, pre)]
            rows = [sum(lens[:s]) + p + i for s, (n, p) in enumerate(zip(lens, pre)) for i in range(n - p)]
            cu = torch.tensor([0] + torch.tensor(part).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
            ix = torch.tensor(rows, device=DEV)
            o = torch.full((len(rows), H * al.vp + 8), 7.0, dtype=dtype, device=DEV)
            i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
            pp = ops.PagedPrefill(tables.to(DEV), i32(range(len(lens))), i32(pre), list(range(len(lens))), pre, kc, vc)
            ops.attn_prefill(q[ix], cu, H, G, 128, scale, out=o, paged=pp, seqlens=part, gate=gate[ix].contiguous(),
                             pitch=al.vp)
            same(o, rows, "portion")
            assert (o[:, H * al.vp:] == 7).all()
        ix = torch.tensor(last, device=DEV)
        for fused in (True, False):
            for splits in (1, 3):
                from llm_map_reduce_summarizer_amd.ops.hip import DecodeWorkspace, decode_groups
                ws = DecodeWorkspace(len(last), H, 128, splits, DEV, decode_groups(H, G), fused_combine=fused)
                o = torch.full((len(last), H * al.vp + 8), 7.0, dtype=dtype, device=DEV)
                ops.attn_decode(q[ix].contiguous(), kc, vc, tables.to(DEV), pos[ix].contiguous(), H, G, 128, page, scale,
                                out=o, workspace=ws, gate=gate[ix].contiguous(), pitch=al.vp)
                same(o, last, "decode")
                assert (o[:, H * al.vp:] == 7).all()


def attention_of(u, w, al, H, G, dim, vdim, scale, coef, every, eps):
    """The oracle's attention fed with given projections: an identity stands where the weights would be."""
    n = u.shape[0]
    cols = torch.cat([u[:, c: c + k] for c, k in ((al.q, H * dim), (al.k, G * dim), (al.v, G * vdim), (al.g, H))], 1)
    eye = torch.eye(cols.shape[1], dtype=torch.float64)
    ww, at = dict(w), 0
    for name, k in (("q", H * dim), ("k", G * dim), ("v", G * vdim), ("g", H)):
        ww["a." + name] = eye[at: at + k]
        at += k
    c = {"heads": H, "kv_heads": G, "dim": dim, "vdim": vdim, "scale": scale, "q_temp": {"coef": coef, "every": every}}
    assert n == cols.shape[0]
    return O.attention(cols, ww, "a.", c, eps)


@pytest.mark.parametrize("n", [3, 86, 171, 342])  # 9, 258, 513 and 1026 pairs: 16, 8, 4 waves and one
@pytest.mark.parametrize("H,G,dk,dv", [(3, 1, 48, 20), (3, 3, 256, 256), (3, 1, 576, 512)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_row_attention_waves(H, G, dk, dv, dtype, n):
    """Decoded rows whose pages several waves share: fewer pages than waves, as many, and more; pages without a weight."""
    from llm_map_reduce_summarizer_amd import ops
    page, latent = 64, dk > 256
    have = [[1300, 64, 1, 65, 128, 2, 511, 1024][i % 8] for i in range(n)]
    kc = rnd(24, G, page, dk, seed=1, dtype=dtype)
    vc = kc if latent else rnd(24, G, page, dv, seed=2, dtype=dtype)
    g = torch.Generator().manual_seed(4)
    tables = torch.stack([torch.randperm(23, generator=g)[:21] for _ in range(n)]).int()
    tables[:, 1] = 23
    pos, seq = torch.tensor(have).int() - 1, torch.arange(n).int()
    q = rnd(n, H * dk, seed=3, std=2.0, dtype=dtype)
    if not latent:
        q[:, ::dk].abs_().add_(1)
        kc[23, :, :, 0] = float("-inf")  # the second page's scores
    i32, args = [pos, seq, tables], (page, dk ** -0.5)
    if latent:
        want = ops.latent_rows(q, kc, *i32, H, dv, *args)
        got = ops.latent_rows(dev(q), dev(kc), *map(dev, i32), H, dv, *args)
    else:
        gate = torch.sigmoid(rnd(n, H, seed=5))
        want, got = torch.zeros(n, H * dv, dtype=dtype), torch.zeros(n, H * dv, dtype=dtype, device=DEV)
        ops.attn_rows(q, kc, vc, *i32, H, G, dv, *args, gate, want)
        ops.attn_rows(dev(q), dev(kc), dev(vc), *map(dev, i32), H, G, dv, *args, dev(gate), got)
    # fp32 scores of dk products, exp, sums of up to 1300 keys: a few 2^-24 each; 16-bit results round by 2^-9
    assert rel(got.float(), want.float()) < (4e-3 if dtype == BF else 2e-6)


@pytest.mark.parametrize("copies", [1, 43, 86, 171])  # decoded rows: 6, 258, 516 and 1026 pairs; portions: tiles
@pytest.mark.parametrize("first", [20, 40, 100])
@pytest.mark.parametrize("H,G,dk,dv", [(6, 2, 64, 64), (6, 3, 200, 256), (6, 1, 576, 512)])
def test_row_attention_first_keys_without_weight(H, G, dk, dv, first, copies, monkeypatch):
    """Scores of minus infinity at the head of a sequence, over less than a tile, more than a tile and more than a page: rows
    that see a finite score give it the weight, rows that see none are no numbers, in every form of the kernels."""
    from llm_map_reduce_summarizer_amd import ops
    from llm_map_reduce_summarizer_amd.ops import hip
    latent, page, args = dk > 256, 64, (64, dk ** -0.5)
    kc = rnd(5, G, page, dk, seed=1)
    kc[1, :, :first, -1] = float("-inf")
    kc[2, :, :max(0, first - page), -1] = float("-inf")
    vc = kc if latent else rnd(5, G, page, dv, seed=2)
    pos = torch.cat([torch.tensor([first - 5, first, first + 60]).repeat(copies)[:copies],
                     torch.arange(first - 10, first + 50)]).int()
    n, singles = len(pos), copies
    seq = torch.cat([torch.arange(copies), torch.full((60,), copies)]).int()
    tables = torch.tensor([[1, 2, 3, 4]]).repeat(copies + 1, 1).int()
    q = rnd(n, H * dk, seed=3)
    q[:, dk - 1::dk].abs_().add_(1)
    monkeypatch.setattr(hip, "PORTION_PAIRS", 0)
    i32 = [pos, seq, tables]
    if latent:
        want = ops.latent_rows(q, kc, *i32, H, dv, *args)
        got = ops.latent_rows(dev(q), dev(kc), *map(dev, i32), H, dv, *args, singles=singles)
    else:
        gate = torch.sigmoid(rnd(n, H, seed=5))
        want, got = torch.zeros(n, H * dv), torch.zeros(n, H * dv, device=DEV)
        ops.attn_rows(q, kc, vc, *i32, H, G, dv, *args, gate, want)
        ops.attn_rows(dev(q), dev(kc), dev(vc), *map(dev, i32), H, G, dv, *args, dev(gate), got, singles=singles)
    got, some = got.cpu(), pos >= first
    assert bool(torch.isfinite(want[some]).all()) and bool(torch.isnan(want[~some]).all())
    assert bool(torch.isnan(got[~some]).all())
    # fp32 scores of dk products, exp, sums of up to 161 keys: a few 2^-24 each
    assert rel(got[some], want[some]) < 2e-6


@pytest.mark.parametrize("H,G,dk,dv", [(8, 2, 48, 32), (6, 2, 128, 100), (5, 5, 64, 64), (4, 1, 200, 256), (70, 1, 16, 8),
                                       (32, 1, 576, 512), (3, 1, 300, 20)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_row_attention_portions(H, G, dk, dv, dtype, monkeypatch):
    """Portions in tiles that rows and heads share: several sequences in a block, rows from the middle of a sequence, page
    and tile borders, a later key that is infinite, values that are the keys' first columns; decoded rows in front."""
    from llm_map_reduce_summarizer_amd import ops
    from llm_map_reduce_summarizer_amd.ops import hip
    monkeypatch.setattr(hip, "PORTION_PAIRS", 0)
    latent, page, lens, pre = dk > 256, 64, [1, 1, 2, 31, 130, 66, 20], [70, 0, 5, 0, 33, 63, 200]
    n, width = sum(lens), dk
    kc = rnd(40, G, page, width, seed=1, dtype=dtype)
    vc = kc if latent else rnd(40, G, page, dv, seed=2, dtype=dtype)
    tables = torch.zeros(len(lens), 8, dtype=torch.int32)
    at = 1
    for i, (a, b) in enumerate(zip(pre, lens)):
        need = -(-(a + b) // page)
        tables[i, :need] = torch.arange(at, at + need)
        at += need
        kc[at - 1, :, (a + b - 1) % page + 1:] = float("inf")  # rows past the sequence
        vc[at - 1, :, (a + b - 1) % page + 1:] = float("nan")
    pos = torch.cat([torch.arange(a, a + b) for a, b in zip(pre, lens)]).int()
    seq = torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens)).int()
    last = int(tables[4, (pre[4] + lens[4] - 1) // page]), (pre[4] + lens[4] - 1) % page
    q = rnd(n, H * dk, seed=3, std=2.0, dtype=dtype)
    if not latent:
        vc[last[0], :, last[1]] = float("inf")  # the last token of a sequence: its own row alone sees it
    args = (dk ** -0.5,)
    i32 = [pos, seq, tables]
    if latent:
        want = ops.latent_rows(q, kc, *i32, H, dv, page, *args)
        got = ops.latent_rows(dev(q), dev(kc), *map(dev, i32), H, dv, page, *args, singles=2)
    else:
        gate, vp = torch.sigmoid(rnd(n, H, seed=4)), dv
        want, got = torch.zeros(n, H * vp, dtype=dtype), torch.zeros(n, H * vp, dtype=dtype, device=DEV)
        ops.attn_rows(q, kc, vc, *i32, H, G, vp, page, *args, gate, want)
        ops.attn_rows(dev(q), dev(kc), dev(vc), *map(dev, i32), H, G, vp, page, *args, dev(gate), got, singles=2)
    got, odd = got.cpu().float(), sum(lens[:5]) - 1
    keep = [t for t in range(n) if latent or t != odd]
    assert bool(torch.isfinite(got[keep]).all())
    # fp32 scores of up to 220 keys and dk products, exp: a few 2^-24 each; 16-bit results round by 2^-9
    assert rel(got[keep], want[keep].float()) < (4e-3 if dtype == BF else 2e-6)
    if not latent:
        assert bool((got[odd] == float("inf")).all())


@pytest.mark.parametrize("H,G,dk,dv", [(8, 2, 128, 128), (4, 1, 576, 512)])
def test_row_attention_portions_without_keys(H, G, dk, dv, monkeypatch):
    """Rows before position 0 have no keys: a run of them in blocks of their own, or between others, reads nothing and
    leaves the others as they are without it."""
    from llm_map_reduce_summarizer_amd.ops import hip
    monkeypatch.setattr(hip, "PORTION_PAIRS", 0)
    page, lens = 64, [70, 100, 41]
    n = sum(lens)
    kc = dev(rnd(6, G, page, dk, seed=1))
    vc = dev(rnd(6, G, page, dv, seed=2)) if dv == dk else kc
    pos = torch.cat([torch.arange(70), torch.full((100,), -1), torch.arange(41)]).int()
    seq = torch.repeat_interleave(torch.arange(3), torch.tensor(lens)).int()
    tables = dev(torch.tensor([[1, 2], [0, 0], [3, 4]], dtype=torch.int32))
    q, gate = dev(rnd(n, H * dk, seed=3)), dev(torch.ones(n, H))

    def run(rows):
        out = torch.zeros(len(rows), H * dv, device=DEV)
        i = dev(torch.tensor(rows))
        hip._rows_attention(q[i].contiguous(), kc, vc, dev(pos)[i].contiguous(), dev(seq)[i].contiguous(), tables, H, G, dk, dv,
                            dk if vc is kc else dv, dv, dk ** -0.5, gate[i].contiguous(), out, 0, None, "rows")
        return out
    held = [i for i in range(n) if pos[i] >= 0]
    got = run(list(range(n)))
    assert torch.equal(got[held], torch.cat([run(held[:70]), run(held[70:])])) and bool(got[70:170].isnan().all())


@pytest.mark.parametrize("key", [31, 32, 65, 97, 130])
@pytest.mark.parametrize("dk,dv", [(128, 128), (64, 40)])
def test_row_attention_portions_infinite_value_of_a_tile(key, dk, dv, monkeypatch):
    """An infinite value in each of the slots that take turns as flags of a tile: rows before it leave it alone."""
    from llm_map_reduce_summarizer_amd import ops
    from llm_map_reduce_summarizer_amd.ops import hip
    monkeypatch.setattr(hip, "PORTION_PAIRS", 0)
    H, G, n, page = 8, 2, 170, 64
    kc, vc = rnd(4, G, page, dk, seed=1), rnd(4, G, page, dv, seed=2)
    vc[1 + key // page, :, key % page, 3] = float("inf")
    i32 = [torch.arange(n).int(), torch.zeros(n, dtype=torch.int32), torch.tensor([[1, 2, 3]], dtype=torch.int32)]
    q, gate = rnd(n, H * dk, seed=3, std=2.0), torch.sigmoid(rnd(n, H, seed=4))
    got = torch.zeros(n, H * dv, device=DEV)
    ops.attn_rows(dev(q), dev(kc), dev(vc), *map(dev, i32), H, G, dv, page, dk ** -0.5, dev(gate), got, singles=0)
    vc[1 + key // page, :, key % page, 3] = 0
    want = torch.zeros(n, H * dv)
    ops.attn_rows(q, kc, vc, *i32, H, G, dv, page, dk ** -0.5, gate, want)
    hit = torch.zeros(n, H, dv, dtype=torch.bool)
    hit[key:, :, 3] = True
    hit, got = hit.view(n, -1), got.cpu()
    assert bool((got[hit] == float("inf")).all())
    # as above
    assert rel(got[~hit], want[~hit]) < 2e-6


def in_two_groups(monkeypatch):
    """Tiles of portions with two groups of waves on a block's keys, whatever portion_groups says; a list that fills as they run."""
    from llm_map_reduce_summarizer_amd.ops import hip
    fn, ran = hip._fn, []

    def portions(*args):
        ran.append(args[-2])
        return fn("mrsum_attn_portions")(*args[:-2], 2, args[-1])
    monkeypatch.setattr(hip, "_fn", lambda name: portions if name == "mrsum_attn_portions" else fn(name))
    return ran


@pytest.mark.parametrize("H,G,dk,dv", [(8, 2, 48, 32), (6, 2, 128, 100), (5, 5, 64, 64), (70, 1, 16, 8), (70, 1, 100, 128)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_row_attention_portions_in_two_groups(H, G, dk, dv, dtype, monkeypatch):
    """More than one block of heads, keys and values of different widths."""
    ran = in_two_groups(monkeypatch)
    test_row_attention_portions(H, G, dk, dv, dtype, monkeypatch)
    assert ran


@pytest.mark.parametrize("H,G,dk,dv", [(8, 2, 128, 128), (70, 1, 64, 64)])
def test_row_attention_portions_without_keys_in_two_groups(H, G, dk, dv, monkeypatch):
    ran = in_two_groups(monkeypatch)
    test_row_attention_portions_without_keys(H, G, dk, dv, monkeypatch)
    assert ran


@pytest.mark.parametrize("key", [31, 32, 65, 97, 130])
@pytest.mark.parametrize("dk,dv", [(128, 128), (64, 40)])
def test_row_attention_portions_infinite_value_of_a_tile_in_two_groups(key, dk, dv, monkeypatch):
    ran = in_two_groups(monkeypatch)
    test_row_attention_portions_infinite_value_of_a_tile(key, dk, dv, monkeypatch)
    assert ran


@pytest.mark.parametrize("M,N,K,split", [(1, 130, 1024, True), (17, 1023, 2048, True), (129, 2062, 512, True),
                                         (500, 8200, 256, True), (1100, 4096, 128, False), (3, 40000, 64, False)])
def test_gemm32_edges(M, N, K, split, monkeypatch):
    """Rows and columns past the last 128 x 128 tile, 16-row blocks past M, rows of C that are not 16-byte aligned, whole
    tiles and tiles in slices of K behind them."""
    from llm_map_reduce_summarizer_amd.ops import hip
    monkeypatch.setattr(hip, "gemm32_small", lambda *_: False)
    assert (hip.gemm32_splits(M, N, K // 32)[1] > 1) == split
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    got = hip.gemm32(dev(x), dev(w)).double().cpu()
    # each of the K products and sums rounds by at most 2^-24 of the sum of magnitudes
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert got.shape == (M, N) and bool(((got - x.double() @ w.double().T).abs() <= bound).all())


@pytest.mark.parametrize("M", [16, 31, 48, 65, 80, 90, 100, 127, 128, 129, 145, 263, 1040])
@pytest.mark.parametrize("N,K", [(130, 32), (2062, 96), (390, 512)])
def test_gemm32_row_blocks(M, N, K, monkeypatch):
    """Every number of 16-row blocks in a tile, tiles of unequal heights that change from column to column, K-tiles fewer than
    the images in flight and more, whole tiles and (K 512) slices of K."""
    from llm_map_reduce_summarizer_amd.ops import hip
    monkeypatch.setattr(hip, "gemm32_small", lambda *_: False)
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    got = hip.gemm32(dev(x), dev(w)).double().cpu()
    # each of the K products and sums rounds by at most 2^-24 of the sum of magnitudes
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert got.shape == (M, N) and bool(((got - x.double() @ w.double().T).abs() <= bound).all())


@pytest.mark.parametrize("M,N,K", [(3, 130, 22528), (72, 130, 22528), (128, 130, 22528), (70, 1030, 6144)])
def test_gemm32_error_does_not_grow_with_k(M, N, K, monkeypatch):
    """One workgroup adds all of K in chains of 512 products and less, however long K is."""
    from llm_map_reduce_summarizer_amd.ops import hip
    monkeypatch.setattr(hip, "gemm32_small", lambda *_: False)
    monkeypatch.setattr(hip, "gemm32_splits", lambda M, N, kb: (-(-M // 128) * -(-N // 128), 1, 0))
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    y = x.double() @ w.double().T
    err = (hip.gemm32(dev(x), dev(w)).double().cpu() - y).norm() / y.norm()
    # a chain's i-th sum has the size of i of its products and rounds by at most 2^-24 of that, with random signs: sqrt(n / 2) 2^-24
    # of the chain's sum for n products; the sums of the chains in the same way
    assert err <= ((512 + K / 256) / 2) ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("M", [64, 65, 100, 128, 300])
@pytest.mark.parametrize("splits", [1, 3])
def test_gemm32_of_one_chain_and_more(M, splits, monkeypatch):
    """512 products in the longest slice are one chain; with 32 more, which are zeros here, the sums of two: the same bits."""
    from llm_map_reduce_summarizer_amd.ops import hip
    N, tiles = 390, -(-M // 128) * 4
    monkeypatch.setattr(hip, "gemm32_small", lambda *_: False)
    monkeypatch.setattr(hip, "gemm32_splits", lambda M, N, kb: (tiles if splits == 1 else 0, splits, tiles * splits * 16384))
    zeros = lambda t: torch.cat([torch.cat([s, torch.zeros(len(t), 32)], 1) for s in t.split(512, 1)], 1)
    x, w = rnd(M, 512 * splits, seed=1), rnd(N, 512 * splits, seed=2)
    assert torch.equal(hip.gemm32(dev(x), dev(w)), hip.gemm32(dev(zeros(x)), dev(zeros(w))))


@pytest.mark.parametrize("M", [0, 4, 64, 65])
def test_gemm32_of_empty_k(M):
    from llm_map_reduce_summarizer_amd.ops import hip
    got = hip.gemm32(dev(torch.zeros(M, 0)), dev(torch.zeros(130, 0)))
    assert got.shape == (M, 130) and bool((got == 0).all())


@pytest.mark.parametrize("M,N,K", [(65, 16, 32), (64, 130, 192), (33, 65, 288), (257, 1, 128), (520, 8192, 192), (300, 1023, 512)])
def test_gemm32_short_k(M, N, K):
    """The 64 x 64 tiles: rows and columns past the last tile, against 64 bits; the larger tiles give the same up to rounding."""
    from llm_map_reduce_summarizer_amd.ops import hip
    assert hip.gemm32_small(M, N, K // 32)
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    got = hip.gemm32(dev(x), dev(w)).double().cpu()
    # each of the K products and sums rounds by at most 2^-24 of the sum of magnitudes
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert got.shape == (M, N) and bool(((got - x.double() @ w.double().T).abs() <= bound).all())


@pytest.mark.parametrize("M", [5, 130])
@pytest.mark.parametrize("off_x,off_w", [(1, 0), (0, 3), (2, 1)])
def test_gemm32_unaligned_storage(M, off_x, off_w):
    """Contiguous operands that begin anywhere in their storage."""
    from llm_map_reduce_summarizer_amd.ops import hip
    N, K = 200, 256
    x, w = dev(rnd(M * K + 8, seed=1)), dev(rnd(N * K + 8, seed=2))
    x, w = x[off_x: off_x + M * K].view(M, K), w[off_w: off_w + N * K].view(N, K)
    assert torch.equal(hip.gemm32(x, w), hip.gemm32(x.clone(), w.clone()))


# row tiles of every height (2 - 5 units of 32 rows), unequal ones, rows and columns past the last tile, whole tiles and slices, one
# K-tile in a slice, odd numbers of them, chains of 16 and one more
TERMS = [(65, 130, 512, (1, 1, 1)), (96, 390, 544, (1, 2, 1)), (160, 256, 1056, (1, 0, 16)), (161, 1023, 608, (2, 3, 5)),
         (250, 2062, 544, (4, 9, 2)), (300, 4100, 512, (3, 0, 3)), (903, 515, 96, (6, 18, 1))]


@pytest.mark.parametrize("M,N,K,plan", TERMS)
def test_gemm32_in_terms(M, N, K, plan, monkeypatch):
    """W of bf16 values: three exact terms of X, sums in fp32.  W with one value that has more bits, in the first K-tile or the
    last: what the fp32 instruction gives."""
    from llm_map_reduce_summarizer_amd.ops import hip
    scratch = (plan[0] * -(-N // 256) - plan[1]) * plan[2] * 40960
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2, dtype=BF).float()
    x[3], x[5] = x[3] * 2.0 ** -90, x[5] * 2.0 ** 90
    full = {}
    for at in ((0, 0), (N - 1, K - 1)):
        v = w.clone()
        v[at] += 2.0 ** -20 * v[at]
        full[at] = v
    monkeypatch.setattr(hip, "gemm32_small", lambda *_: False)
    monkeypatch.setattr(hip, "gemm32_terms", lambda *_: None)
    want = {at: hip.gemm32(dev(x), dev(v)) for at, v in full.items()}
    monkeypatch.setattr(hip, "gemm32_terms", lambda *_: (*plan, scratch))
    got = hip.gemm32(dev(x), dev(w)).double().cpu()
    # a sum rounds by at most 2^-24 of the sum of magnitudes, and there are at most K of them
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert got.shape == (M, N) and bool(((got - x.double() @ w.double().T).abs() <= bound).all())
    for at, v in full.items():
        assert torch.equal(hip.gemm32(dev(x), dev(v)), want[at])


# every tile height over more than one chain of 16 K-tiles, whole and in slices, odd numbers of K-tiles, heights side by side
HEIGHTS = [(50, 300, 1056, (1, 2, 1)), (50, 300, 1056, (1, 0, 2)), (96, 257, 1280, (1, 2, 1)), (96, 257, 1280, (1, 1, 3)),
           (120, 256, 1120, (1, 1, 1)), (120, 256, 1120, (1, 0, 5)), (160, 300, 1568, (1, 2, 1)), (160, 300, 1568, (1, 0, 4)),
           (300, 520, 1088, (3, 9, 1)), (300, 520, 1088, (3, 4, 2)), (903, 515, 96, (6, 18, 1))]


def terms_only(hip, monkeypatch, N, plan):
    """gemm32 in terms by ``plan``; and a function that gives what the fp32 instruction does."""
    scratch = (plan[0] * -(-N // 256) - plan[1]) * plan[2] * 40960
    monkeypatch.setattr(hip, "gemm32_small", lambda *_: False)
    monkeypatch.setattr(hip, "gemm32_terms", lambda *_: (*plan, scratch))

    def instruction(x, w):
        with monkeypatch.context() as m:
            m.setattr(hip, "gemm32_terms", lambda *_: None)
            return hip.gemm32(x, w)
    return instruction


@pytest.mark.parametrize("bits,per_row", [(21, 6), (24, 1)])
@pytest.mark.parametrize("M,N,K,plan", HEIGHTS)
def test_gemm32_in_terms_leaves_no_bit_out(M, N, K, plan, bits, per_row, monkeypatch):
    """X of integers of so many bits and W of few ones: every product and every sum, in any order, is an integer below 2^24 and
    exact, so the result is, and a term left out is seen."""
    from llm_map_reduce_summarizer_amd.ops import hip
    terms_only(hip, monkeypatch, N, plan)
    g = torch.Generator().manual_seed(5)
    x = torch.randint(1 << (bits - 1), 1 << bits, (M, K), generator=g) | 1
    x *= torch.randint(0, 2, (M, K), generator=g) * 2 - 1
    w = torch.zeros(N, K, dtype=torch.int64)
    w.scatter_(1, torch.rand(N, K, generator=g).argsort(1)[:, :per_row], 1)
    w *= torch.randint(0, 2, (N, K), generator=g) * 2 - 1
    want = (x.double() @ w.double().T).float()
    assert torch.equal(hip.gemm32(dev(x.float()), dev(w.float())).cpu(), want)
    # the two upper terms of X alone give other values nearly everywhere
    top = x.float()
    for shift in (2.0 ** (bits - 8), 2.0 ** (bits - 16)):
        hi = torch.trunc(top / shift) * shift
        top = top - hi
    assert float(((x.double() - top.double()) @ w.double().T != want).double().mean()) > 0.8


@pytest.mark.parametrize("kind", ["bit", "inf", "subnormal"])
def test_gemm32_in_terms_finds_each_column_of_w(kind, monkeypatch):
    """Two waves share a tile's columns and look at half of them each: one value that is not its bf16 term, in every block of
    16 columns, in the first K-tile, in the one behind a chain and in the last."""
    from llm_map_reduce_summarizer_amd.ops import hip
    M, N, K = 70, 256, 576
    instruction = terms_only(hip, monkeypatch, N, (1, 1, 1))
    x, w = dev(rnd(M, K, seed=1)), dev(rnd(N, K, seed=2, dtype=BF).float())
    got = hip.gemm32(x, w)
    assert not torch.equal(got, instruction(x, w)) and rel(got, x.cpu().double() @ w.cpu().double().T) < 1e-6
    for n in range(0, N, 16):
        for k in (n % 32, 16 * 32 + 5, K - 1 - n % 3):
            v = w.clone()
            at = n + (n // 16 * 5) % 16, k
            v[at] = {"bit": v[at] * (1 + 2.0 ** -20), "inf": float("inf"), "subnormal": 2.0 ** -130}[kind]
            assert torch.equal(hip.gemm32(x, v), instruction(x, v)), (n, k)


@pytest.mark.parametrize("M,N,K,plan", [(160, 1500, 2080, (1, 6, 1)), (300, 1024, 1600, (3, 12, 1)), (500, 700, 3200, (4, 6, 3))])
@pytest.mark.parametrize("n0,n1,k", [(0, 256, 0), (300, 301, 700), (500, 700, 520), (699, 700, 1599)])
def test_gemm32_in_terms_stops_with_its_neighbours(M, N, K, plan, n0, n1, k, monkeypatch):
    """Some rows of W have more bits from some column on: tiles that see it, at their start, behind a chain or at their end, and
    tiles that hear of it from others, whole and in slices, and again when the call is replayed."""
    from llm_map_reduce_summarizer_amd.ops import hip
    instruction = terms_only(hip, monkeypatch, N, plan)
    x, w = dev(rnd(M, K, seed=1)), dev(rnd(N, K, seed=2, dtype=BF).float())
    clean = hip.gemm32(x, w)
    v = w.clone()
    v[n0:n1, k:] *= 1 + 2.0 ** -20
    want = instruction(x, v)
    assert not torch.equal(clean, want)
    buf = w.clone()
    hip.gemm32(x, buf)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = hip.gemm32(x, buf)
    for src, res in ((v, want), (w, clean), (v, want), (v, want), (w, clean)):
        buf.copy_(src)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, res) and torch.equal(hip.gemm32(x, src), res)


@pytest.mark.parametrize("at", [(0, 0), (8191, 2047), (8999, 4095)])
@pytest.mark.parametrize("value,held", [(1.0, True), (0.0, True), (-0.0, True), (2.0 ** -126, True), (1 + 2.0 ** -8, False), (3.0e38, False),
                                        (2.0 ** -127, False), (-2.0 ** -149, False), (float("inf"), False), (float("nan"), False)])
def test_weights_of_bf16_values(at, value, held):
    from llm_map_reduce_summarizer_amd.ops import hip
    w = torch.randn(9000, 4096, generator=torch.Generator(DEV).manual_seed(1), device=DEV).to(BF).float()
    w[at] = value
    odd = w.view(-1)[1:8191].view(1, -1)  # not on 16 bytes, no multiple of four
    odd[0, -1] = value
    assert hip.bf16_values(w, w[:0], odd, w[8998:8999], w[8999:, :]) == [held, True, held, True, held or at[0] != 8999]


def entries(hip, monkeypatch):
    """Names of the entry points called from here on."""
    names, fn = [], hip._fn
    monkeypatch.setattr(hip, "_fn", lambda name: names.append(name) or fn(name))
    return names


def test_gemm32_of_weights_known_to_have_more_bits(monkeypatch):
    """They run on the fp32 instruction alone, as before there were terms; a mark that no longer holds costs no bit."""
    from llm_map_reduce_summarizer_amd import ops
    from llm_map_reduce_summarizer_amd.ops import hip
    x, w = dev(rnd(300, 4096, seed=1)), dev(rnd(4096, 4096, seed=2))
    names = entries(hip, monkeypatch)
    got = hip.gemm32(x, w)
    assert names == ["mrsum_gemm32_terms"]
    ops.mark_values(w)
    assert w.bf16_values is False and torch.equal(ops.project(x, w, "o")[0], got) and torch.equal(ops.logits32(x, w), got)
    assert names[1:] == ["mrsum_bf16_values"] + ["mrsum_gemm32"] * 2
    v = w.to(BF).float()
    ops.mark_values(v)
    assert v.bf16_values is True
    v.copy_(w)
    assert torch.equal(hip.gemm32(x, v), got)
    w.copy_(w.to(BF).float())
    assert rel(hip.gemm32(x, w).cpu(), x.cpu().double() @ w.cpu().double().T) < 1e-6


@pytest.mark.parametrize("model", ["tiny-merulorn", "tiny-muzozen"])
@pytest.mark.parametrize("more", [False, True])
def test_models_know_which_weights_are_bf16_values(model, more, monkeypatch):
    from llm_map_reduce_summarizer_amd.engine.config import get_model_config
    from llm_map_reduce_summarizer_amd.engine.hybrid import HybridModel
    plain = HybridModel._random

    def random(self, seed):
        get = plain(self, seed)
        return lambda name, shape: get(name, shape).float() * (1 + 2.0 ** -12) if more else get(name, shape)
    monkeypatch.setattr(HybridModel, "_random", random)
    m = HybridModel(get_model_config(model), torch.device(DEV), F32)
    found = [m.lm_head] + [t for la in m.layers for t in (la.w.w_in, la.w.w_o)]
    found += [la.w.w_gu for la in m.layers if hasattr(la.w, "w_gu")] + [la.latent.w.w_uq for la in m.layers if la.latent is not None]
    assert len(found) > 4 and [t.bf16_values for t in found] == [not more] * len(found)
    half = HybridModel(get_model_config(model), torch.device(DEV), BF)
    assert not hasattr(half.lm_head, "bf16_values")


@pytest.mark.parametrize("M,K,tiles,at", [(70, 512, 1, (0, 0)), (70, 512, 1, (69, 511)), (70, 608, 1, (33, 607)), (96, 544, 1, (95, 543)),
                                          (161, 1056, 2, (97, 1055)), (160, 9632, 1, (159, 9631)), (160, 9632, 1, (3, 7000))])
def test_gemm32_in_terms_of_values_finer_than_bf16(M, K, tiles, at, monkeypatch):
    """One value of X whose lowest bits are below bf16's: what the fp32 instruction gives.  Values down to 2^-110 are the sums of
    their terms, whose own values are subnormal then."""
    from llm_map_reduce_summarizer_amd.ops import hip
    N = 256
    instruction = terms_only(hip, monkeypatch, N, (tiles, tiles, 1))
    x, w = dev(rnd(M, K, seed=1)), torch.zeros(N, K)
    w[torch.arange(N), torch.randint(0, K, (N,), generator=torch.Generator().manual_seed(3))] = 1.0
    w[7], w[7, at[1]] = 0.0, 1.0
    w, x[at] = dev(w), 2.0 ** -111 * (1 + 2.0 ** -23)
    assert torch.equal(hip.gemm32(x, w), instruction(x, w))
    small = (torch.randint(1 << 23, 1 << 24, (M, K), generator=torch.Generator().manual_seed(4)).double() * 2.0 ** -133).float()
    got = hip.gemm32(dev(small), w).double().cpu()
    assert torch.equal(got, small.double() @ w.double().cpu().T)


def test_gemm32_in_terms_of_infinities():
    """Infinities and NaN in X and W make what fp32 products and sums make of them."""
    from llm_map_reduce_summarizer_amd.ops import hip
    M, N, K = 300, 4096, 4096
    assert hip.gemm32_terms(M, N, K // 32)
    inf, nan = float("inf"), float("nan")
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2, dtype=BF).float()
    x[7, 9], x[8, 4095], x[299, 0] = inf, -inf, nan
    x[20] = torch.full((K,), 1, dtype=torch.int32).add_(0x7f800000).view(F32)  # NaN whose bits are all low
    for odd in (False, True):
        if odd:
            w[11, 5], w[4095, 4095], w[77, 2048] = inf, -inf, nan
        want, got = x.double() @ w.double().T, hip.gemm32(dev(x), dev(w)).cpu()
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
        assert torch.equal(got[want.isinf()].double(), want[want.isinf()])
        ok = want.isfinite()
        assert float((got.double() - want)[ok].norm() / want[ok].norm()) < 1e-6


def test_gemm32_in_terms_of_many_rows(monkeypatch):
    """Terms beyond their buffer's size are made for a part of the rows at a time; replays of a captured product give the same."""
    from llm_map_reduce_summarizer_amd.ops import hip
    M, N, K = 700, 1024, 1024
    x, w = dev(rnd(M, K, seed=1)), dev(rnd(N, K, seed=2, dtype=BF).float())
    monkeypatch.setattr(hip, "gemm32_terms", lambda m, n, kb: (-(-m // 160), -(-m // 160) * 4, 1, 0))
    want = hip.gemm32(x, w)
    monkeypatch.setattr(hip, "GEMM32_TERMS_BYTES", 300 * K * 6)
    assert torch.equal(hip.gemm32(x, w), want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = hip.gemm32(x, w)
    for scale in (1, 2, 4):
        got.zero_()
        x.mul_(scale)
        want = want * scale  # powers of two
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.parametrize("M", [1, 16, 17, 33, 48, 49])
@pytest.mark.parametrize("K,splits", [(512, 1), (4096, 1), (4096, 3)])
def test_gemm32_of_weights_that_no_cache_holds(M, K, splits, monkeypatch):
    """Beyond 256 MiB W is read past the caches, for up to 48 rows: the bits of two products of its halves."""
    from llm_map_reduce_summarizer_amd.ops import hip
    N = (1 << 26) // K + 3 * 128 + 5
    tiles = lambda n: -(-M // 128) * -(-n // 128)  # noqa: E731
    monkeypatch.setattr(hip, "gemm32_small", lambda *_: False)
    monkeypatch.setattr(hip, "gemm32_splits", lambda m, n, kb: (tiles(n), 1, 0) if splits == 1 else (0, splits, tiles(n) * splits * 16384))
    x = dev(rnd(M, K, seed=1))
    w = torch.randn(N, K, generator=torch.Generator(DEV).manual_seed(2), device=DEV)
    got, half = hip.gemm32(x, w), N // 256 * 128
    assert torch.equal(got, torch.cat([hip.gemm32(x, w[:half]), hip.gemm32(x, w[half:])], 1))
    assert rel(got.cpu(), (x.double() @ w.double().T).cpu()) < 1e-6


def test_gemm32_deep():
    """K beyond what 31-bit offsets over a tile's rows reach."""
    from llm_map_reduce_summarizer_amd.ops import hip
    K = hip.GEMM32_MAX_K + 96
    x, w = rnd(2, K, seed=1), rnd(3, K, seed=2)
    got, want = hip.gemm32(dev(x), dev(w)).double().cpu(), x.double() @ w.double().T
    # K roundings, each at most 2^-24 of a sum of the size sqrt(K), add up to sqrt(K) of one: four times that
    assert bool(((got - want).abs() <= 4 * K ** 0.5 * 2.0 ** -24 * K ** 0.5).all())


def test_gemm32_shapes():
    from llm_map_reduce_summarizer_amd.ops import hip
    for Mr, N, K in ((1, 16, 32), (70, 130, 96), (64, 64, 128), (129, 77, 256)):
        x, w = rnd(Mr, K), rnd(N, K, seed=1)
        assert rel(hip.gemm32(dev(x), dev(w)), x.double() @ w.double().T) < 1e-6


# ------------------------------------------------------------------ whole models
@pytest.mark.parametrize("name", sorted(M.CONFIGS))
@pytest.mark.parametrize("dtype", DTYPES)
def test_prompt_and_token_by_token(name, dtype, tmp_path):
    eng = M.engine(name, tmp_path, DEV, dtype)
    ids = M.tokens(name, 140)
    want = M.expected(name, ids)
    M.check(M.feed(eng, "a", ids, [140]), want, dtype, "one portion")
    M.check(M.feed(eng, "b", ids, [1] * 140), want, dtype, "token by token")
    M.check(M.feed(eng, "c", ids, M.cuts(140, [2, 3, 64, 1, 17])), want, dtype, "portions")


@pytest.mark.parametrize("name", ["mixed", "wide"])
@pytest.mark.parametrize("dtype", DTYPES)
def test_unequal_requests_share_batches_and_reuse_slots(name, dtype, tmp_path):
    lengths = {"a": 131, "b": 5, "c": 64, "d": 1, "e": 90, "f": 65}
    eng = M.engine(name, tmp_path, DEV, dtype, max_num_seqs=3, kv_pages=8)
    reqs = {r: M.tokens(name, n, seed=i) for i, (r, n) in enumerate(lengths.items())}
    got = M.feed_mixed(eng, reqs, M.mixed_plan(lengths, [1, 30, 2, 1, 64, 1], live=3))
    for r, ids in reqs.items():
        M.check(got[r], M.expected(name, ids), dtype, r)


@pytest.mark.parametrize("dtype", DTYPES)
def test_long_prompt_then_long_decoding(dtype, tmp_path):
    """A prompt of several runs of the scan, then 100 decoded tokens across page borders."""
    eng = M.engine("wide", tmp_path, DEV, dtype, max_model_len=1024)
    ids = M.tokens("wide", 700)
    M.check(M.feed(eng, "a", ids, [600] + [1] * 100), M.expected("wide", ids), dtype)


@pytest.mark.parametrize("name", ["mixed", "wide"])
@pytest.mark.parametrize("dtype", DTYPES)
def test_greedy_generation_with_graphs(name, dtype, tmp_path):
    """generate(): packed prefill, hipGraph decode replayed over growing, shrinking and refilled batches (several
    captures, eager work between replays), sliced prompts, requests joining a running batch."""
    from llm_map_reduce_summarizer_amd.engine.engine import SamplingParams
    eng = M.engine(name, tmp_path, DEV, dtype, prefill_chunk=64, max_num_seqs=3)
    prompts = [M.tokens(name, n, seed=n) for n in (3, 130, 64, 1, 77)]
    slack = 0.15 if dtype == BF else 1e-4
    for _ in range(2):
        outs = eng.generate(prompts, [SamplingParams(n, 0.0, 1) for n in (30, 12, 6, 20, 2)])
        assert [len(o.token_ids) for o in outs] == [30, 12, 6, 20, 2]
        for p, o in zip(prompts, outs):
            M.check_greedy(name, p, o.token_ids, slack)
    fed = []

    def feeder(done):
        if not fed:
            fed.append(1)
            return [(p, SamplingParams(7, 0.0, 1)) for p in prompts[1:3]]
        return []
    outs = eng.generate(prompts[:1], [SamplingParams(25, 0.0, 1)], feeder=feeder)
    for p, o in zip([prompts[0]] + prompts[1:3], outs):
        M.check_greedy(name, p, o.token_ids, slack)
    assert eng.stats["graph_captures"] >= 2 and eng.kv.state.alloc.available() == 3


def test_graph_capture_leaves_live_state_alone(tmp_path):
    """The eager warm-up before a capture must not advance the recurrent state of the rows it runs on."""
    from llm_map_reduce_summarizer_amd.engine.engine import SamplingParams
    prompts = [M.tokens("wide", n, seed=n) for n in (50, 20)]
    outs = []
    for graphs in (False, True):
        eng = M.engine("wide", tmp_path, DEV, F32, use_graphs=graphs)
        outs.append([o.token_ids for o in eng.generate(prompts, [SamplingParams(40, 0.0, 1)] * 2)])
    assert outs[0] == outs[1]


def test_trace_runner_on_the_gpu(tmp_path, monkeypatch, capsys):
    import io
    import json
    from llm_map_reduce_summarizer_amd import trace
    path = M.checkpoint("mixed", str(tmp_path / "m"))
    ids = M.tokens("mixed", 70)
    steps = [{"step": 0, "entries": [{"id": "x", "tokens": ids[:66], "want": [0, 65]}], "end": []},
             {"step": 1, "entries": [{"id": "x", "tokens": ids[66:67], "want": [0]},
                                     {"id": "y", "tokens": ids[:20], "want": [19]}], "end": ["x", "y"]}]
    monkeypatch.setattr("sys.stdin", io.StringIO("".join(json.dumps(s) + "\n" for s in steps)))
    assert trace.main(["--model", path, "--dtype", "bfloat16", "--out", str(tmp_path), "--max-tokens", "192"]) == 0
    assert "done 1" in capsys.readouterr().out
    got = torch.cat([torch.frombuffer(bytearray((tmp_path / ("%d.f32" % k)).read_bytes()), dtype=F32).view(2, -1)
                     for k in (0, 1)])
    M.check(got, M.expected("mixed", ids)[[0, 65, 66, 19]], BF)


@pytest.mark.parametrize("H,G,d,pitch", [(8, 2, 128, 128), (3, 3, 64, 60), (5, 1, 100, 100), (2, 1, 20, 20)])
@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("groups", [1, 2])
def test_portion_attention_of_key_groups(H, G, d, pitch, dtype, groups):
    """Walks of 1 key to several tiles, odd and even, sequences that share a block, and values that are not finite behind the keys
    of a row: the groups' sums meet to what one softmax over all keys gives."""
    from llm_map_reduce_summarizer_amd.ops.hip import _fn, _p, _stream
    portions = [(3, 0), (70, 0), (1, 31), (5, 60), (40, 100), (2, 0), (33, 223)]
    T, ends = sum(n for n, _ in portions), [n + b for n, b in portions]
    pages = [-(-e // 64) for e in ends]
    q, kc, vc = rnd(T, H * d), rnd(sum(pages), G, 64, d, seed=1), rnd(sum(pages), G, 64, d, seed=2)
    perm, tables, at = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(3)), [], 0
    for p in pages:
        tables.append(perm[at: at + p].tolist())
        at += p
    vc[tables[1][1], :, 5] = float("inf")  # key 69: the last row of the second portion alone has it
    vc[tables[4][1], 0, 63, 0] = float("nan")  # key 127: rows 27 .. of the fifth
    q, kc, vc = (t.to(dtype) for t in (q, kc, vc))
    bt = torch.zeros(len(portions), max(pages), dtype=torch.int32)
    for i, t in enumerate(tables):
        bt[i, :len(t)] = torch.tensor(t)
    pos = torch.cat([torch.arange(b, b + n) for n, b in portions]).int()
    seq = torch.cat([torch.full((n,), i) for i, (n, _) in enumerate(portions)]).int()
    gate = rnd(T, H, seed=4)
    args = [dev(t) for t in (q, kc, vc, pos, seq, bt, gate)]
    out = torch.full((T, H * pitch + 8), 7.0, dtype=dtype, device=DEV)
    assert _fn("mrsum_attn_portions")(*map(_p, args[:6]), bt.stride(0), T, H, G, d, d, d, pitch, d ** -0.5, _p(args[6]), _p(out),
                                      out.stride(0), 1 if dtype == F32 else 0, groups, _stream()) == 0
    got, row = out.cpu(), 0
    assert (got[:, H * pitch:] == 7).all()
    for (n, b), t in zip(portions, tables):
        K, V = (c[t].double().permute(1, 0, 2, 3).reshape(G, -1, d).repeat_interleave(H // G, 0) for c in (kc, vc))
        for r in range(n):
            w = torch.softmax((K[:, :b + r + 1] @ q[row].double().view(H, d, 1)).squeeze(-1) * d ** -0.5, -1)
            want = (w[:, None] @ V[:, :b + r + 1]).squeeze(1)[:, :pitch] * gate[row].double()[:, None]
            have = got[row, :H * pitch].view(H, pitch).double()
            good = want.isfinite()
            assert torch.equal(good, have.isfinite()), (row, r)
            # fp32: sums of up to 256 terms in eight chains; bf16: the output's rounding
            if good.any():
                assert rel(have[good], want[good]) < (4e-3 if dtype == BF else 3e-6)
            row += 1
