"""Host-side work lists and launch plans of the HIP ops (no GPU needed): the prefill-attention item list
covers every query row of every sequence exactly once at each GQA ratio, heaviest blocks first, and the
decode-attention split plan keeps its measured choices (ops/hip.py)."""
import glob
import importlib.util
import json
import os
import re

import numpy as np
import pytest
import torch

from llm_map_reduce_summarizer_amd.ops import hip

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("group", [1, 2, 4, 8, 3, 5, 16])
def test_prefill_items_cover_every_row_once(group):
    seqlens = [1, 63, 64, 65, 300, 4096]
    bm = hip.prefill_block_m(group)
    # packed GQA ratios: 256 / G positions per workgroup; others: per-query-head fallback, 256 positions
    assert bm == (256 // group if group in (1, 2, 4, 8) else 256)
    items = hip.prefill_items(seqlens, group).tolist()
    assert len(items) == sum(-(-n // bm) for n in seqlens)
    seen = {s: [0] * n for s, n in enumerate(seqlens)}
    for s, qb in items:
        assert qb % bm == 0 and 0 <= qb < seqlens[s]
        for r in range(qb, min(qb + bm, seqlens[s])):
            seen[s][r] += 1
    assert all(c == 1 for rows in seen.values() for c in rows)
    starts = [qb for _, qb in items]
    assert starts == sorted(starts, reverse=True)  # heaviest (latest) blocks first


def test_prefill_block_m_rejects_bad_ratios():
    for g in (0, 65):
        with pytest.raises(ValueError):
            hip.prefill_block_m(g)


def test_decode_groups():
    assert hip.decode_groups(32, 8) == 8 and hip.decode_groups(64, 8) == 8 and hip.decode_groups(16, 1) == 1
    assert hip.decode_groups(24, 8) == 24  # ratio 3: one group per query head
    with pytest.raises(ValueError):
        hip.decode_groups(24, 7)


def test_decode_attn_plan_measured_choices():
    # a TP shard's single kv head at B=20, 4k context: 12 fused splits (profiles/r3_plans_insitu_tp8_b39_b20.jsonl)
    assert hip.decode_attn_plan(20, 1, 4096) == (12, True)
    # the same batch over 8 kv heads (TP=1) keeps at most 8 fused splits
    s, fused = hip.decode_attn_plan(20, 8, 4096)
    assert fused is False or s <= 8
    # B=1 at TP=8 (one kv head, 4k): one workgroup per page, separate merge
    s, fused = hip.decode_attn_plan(1, 1, 4096)
    assert not fused and s == 64


@pytest.mark.parametrize("batch,ctx,splits", [(17, 4608, 3), (39, 4608, 4), (39, 6144, 4), (64, 2048, 4), (92, 4608, 4), (300, 4608, 4),
                                              (20, 128, 1), (20, 32768, 4), (92, 12288, 1)])
def test_decode_attn_plan_of_many_rows_keeps_its_order_of_sums(batch, ctx, splits):
    """Splits are the order in which a row's sums are added, and the bytes that later layers store."""
    assert hip.decode_attn_plan(batch, 8, ctx) == (splits, False)
    for kv8 in ("fp8v", "fp8"):
        assert hip.decode_attn_plan(batch, 8, ctx, kv8=kv8) == (splits, False)


def test_decode_attn_plan_class1_six_fused_splits():
    # the <= 12k context class (level-1 reduce at ~6k), per graph bucket: 6 fused splits, in situ
    # (profiles/r4_attn_plans_insitu_class1.jsonl): batch 5 (bucket 8) and batch 10 (bucket 16) faster than 4
    assert hip.decode_attn_plan(8, 8, 12288) == (6, True)
    assert hip.decode_attn_plan(16, 8, 12288) == (6, True)
    # the final reduce (B=1, ~13k, <= 32k class) keeps 32 separate splits (best of 16-64 / fused in situ)
    assert hip.decode_attn_plan(1, 8, 32768) == (32, False)
    # a TP shard's single kv head beyond 6k (config 5's 32k at TP=8): one workgroup per 2 pages, up to 128
    # splits (70B fp8 shard step at 32k: 128 splits 4.80 ms vs 64 5.07, 250 5.10, 32 5.66; r5_attn_plans*.jsonl)
    assert hip.decode_attn_plan(1, 1, 32768) == (128, False)
    assert hip.decode_attn_plan(1, 1, 12288) == (96, False)
    assert hip.decode_attn_plan(16, 1, 32768) == (48, False)
    assert all(hip.decode_attn_plan(b, h, c)[0] <= hip.MAX_SPLITS for b in (1, 2, 16, 64) for h in (1, 2, 8)
               for c in (4096, 12288, 32768, 131072))
    # TP shards keep their measured cap of 4 in the longer classes
    assert hip.decode_attn_plan(20, 1, 12288)[0] <= 4


def test_skinny_waves_rule():
    # 8-wave workgroups where the grid is about one workgroup per CU or less (TP-shard N / 16 tiles)
    assert hip.skinny_waves(3584, 1, 1) == 8      # 8B TP=8 gate_up: 224 workgroups
    assert hip.skinny_waves(4096, 1, 1) == 8      # o / down producers: 256
    assert hip.skinny_waves(7168, 1, 1) == 8      # 70B TP=8 gate_up: 448
    assert hip.skinny_waves(57344, 1, 1) == 4     # 70B TP=1 gate_up: 3584
    assert hip.skinny_waves(4096, 1, 4) == 4      # split-K slabs: 1024
    assert hip.skinny_waves(4096, 1, 1, M=10) == 4  # more than one row: 4 waves (measured 0.3-1 % faster)


def test_fp8_tp_push_producer_rule(monkeypatch):
    # 70B fp8 TP=8 shard: o (K 1024) on the fp8 register-streaming producer at every decode row count up to
    # 16, down (K 3584) only at one row (in situ, profiles/r5_fp8_skinny_push_ab.jsonl); TP=1 keeps the stream
    # producer
    import torch
    from llm_map_reduce_summarizer_amd import ops
    from llm_map_reduce_summarizer_amd.ops.reference import Fp8Weight
    monkeypatch.setattr(hip, "skinny_fp8_resid_capacity", lambda: 1024)

    def w(N, K):
        return Fp8Weight(torch.empty(N, K, dtype=torch.float8_e4m3fn, device="meta"),
                         torch.empty(N, dtype=torch.float32, device="meta"))

    def a(M, K):
        return torch.empty(M, K, dtype=torch.bfloat16, device="meta")

    assert ops._resid_plan(hip, a(1, 1024), w(8192, 1024), "o", tp=True) == ("skinny",)
    assert ops._resid_plan(hip, a(10, 1024), w(8192, 1024), "o", tp=True) == ("skinny",)
    assert ops._resid_plan(hip, a(1, 3584), w(8192, 3584), "down", tp=True) == ("skinny",)
    assert ops._resid_plan(hip, a(10, 3584), w(8192, 3584), "down", tp=True)[0] == "stream"
    assert ops._resid_plan(hip, a(1, 8192), w(8192, 8192), "o", tp=False)[0] == "stream"
    assert ops._resid_plan(hip, a(1, 1024), w(8192, 1024), "o", tp=True, force="stream")[0] == "stream"


def test_narrow_gate_up_split_rules():
    # fp8: a gate_up too narrow for one stream tile per CU takes the split-K SwiGLU (70B TP=8 shard, every decode
    # row count: profiles/r6_fp8_swiglu_split_insitu.jsonl); TP=1 / TP=4 at <= 8 rows stay on the register-
    # streaming kernel (N x K >= 64 M), and wider gate_ups keep one tile per column
    assert hip.stream_config_fp8(7168, 8192, swiglu=True, M=1) == (7, 4)
    assert hip.stream_config_fp8(7168, 8192, swiglu=True, M=39) == (7, 4)
    assert hip.stream_config_fp8(14336, 8192, swiglu=True, M=1) is None
    assert hip.stream_config_fp8(57344, 8192, swiglu=True, M=1) is None
    assert hip.stream_config_fp8(57344, 8192, swiglu=True, M=16) == (7, 1)
    # bf16: the TP=4 shard's 7168-row gate_up splits at one row too (one-round grid), the TP=8 shard's 3584 rows
    # stay on the register-streaming kernel up to 16 rows, the TP=2 shard's 14336 rows on one tile per column
    # (profiles/r6_bf16_swiglu_split_insitu.jsonl)
    assert hip.plan("gate_up", 1, 7168, 4096) == ("stream_split", 7, 4)
    assert hip.plan("gate_up", 10, 7168, 4096) == ("stream_split", 7, 4)
    assert hip.plan("gate_up", 1, 3584, 4096)[0] == "skinny"
    assert hip.plan("gate_up", 1, 14336, 4096) == ("stream", 4, 1)


@pytest.mark.parametrize("portions,hkv,tiles", [
    # 32 heads of 128: row kernel and tiles, us (profiles/row_attention_portions.jsonl)
    ([(2, 1998)] * 32, 32, False),  # 769, 6117: 32 contexts in one workgroup's chain
    ([(2, 1998)] * 32, 8, False),   # 636, 1533
    ([(8, 1992)] * 32, 8, True),    # 1478, 404
    ([(16, 584)] * 8, 32, False),   # 236, 255
    ([(32, 568)] * 8, 32, True),    # 431, 134
    ([(900, 0)], 8, True),          # 1018, 107
    ([(900, 0), (2, 30)], 8, True)])
def test_row_attention_of_short_portions(portions, hkv, tiles, monkeypatch):
    """Prompt portions go to the tiled kernel where it leads: not where a workgroup would walk many contexts."""
    ran = []
    monkeypatch.setattr(hip, "_fn", lambda name: lambda *a: ran.append((name, a[7])) or 0)
    monkeypatch.setattr(hip, "_stream", lambda: 0)
    rows, one = 3 + sum(n for n, _ in portions), torch.zeros(1, dtype=torch.int32)
    t = torch.zeros(rows, 32 * 128)
    hip._rows_attention(t, t, t.clone(), one, one, one[None], 32, hkv, 128, 128, 128, 128, 1.0, None, t, 3, portions, "")
    assert ran == ([("mrsum_attn_rows", 3), ("mrsum_attn_portions", rows - 3)] if tiles else [("mrsum_attn_rows", rows)])


@pytest.mark.parametrize("M,N,K,small", [
    # us in 128 x 128 and 64 x 64 tiles (profiles/gemm32_short_k.jsonl)
    (256, 4096, 256, True),    # 20, 13
    (300, 2048, 192, True),    # 16, 8
    (520, 8192, 192, True),    # 29, 23
    (64, 4096, 256, True),     # 12, 13
    (900, 16384, 128, True),   # 43.3, 42.9 (903 rows)
    (1500, 8192, 256, False),  # 58, 64
    (300, 4096, 768, False),   # 32, 37
    (8, 16384, 256, False),    # 6, 13
    (300, 16384, 192, True),   # 28, 23
    (700, 8192, 192, True),    # 31, 26
    (64, 4096, 128, True),     # 8, 6
    (100, 1024, 384, True),    # 15, 14
    (40, 16384, 256, False),   # 11, 13
    (903, 4096, 4096, False)])
def test_fp32_gemm_of_short_k(M, N, K, small):
    assert hip.gemm32_small(M, N, K // 32) == small


def test_wide_heads_keep_the_outputs_they_took(monkeypatch):
    """The tile GEMM takes a head's 65 - 128 rows only into rows that it can store; others stay with the stream GEMM."""
    ran = []
    monkeypatch.setattr(hip, "gemm", lambda x, w, out=None, **kw: ran.append("tile") or out)
    monkeypatch.setattr(hip, "_stream_gemm", lambda x, w, out, *a, **kw: ran.append("stream") or out)
    M, N, K = 66, 49152, 256
    x, w, room = (torch.empty(n, dtype=torch.bfloat16) for n in (M * K, N * K, M * N + 4))
    x, w = x.view(M, K), w.view(N, K)
    assert hip.tile_head(M, N)
    for off in (0, 4, 1, 2):  # elements of 2 bytes
        hip.linear(x, w, out=room[off: off + M * N].view(M, N))
    hip.linear(x, w)
    assert ran == ["tile", "tile", "stream", "stream", "tile"]


def recorded(name):
    """Lines of a record under profiles/; some machines get the tree without them."""
    path = os.path.join(ROOT, "profiles", name)
    if not os.path.exists(path):
        pytest.skip("no " + name)
    with open(path) as f:
        return [json.loads(line) for line in f if not line.startswith("#")]


def test_tile_gemm_plan_by_its_record():
    """What the rule takes was timed, is what the record says, and is near the best of each shape: 20 % at most, 1 % on average
    (whether or not the rule was fitted to the shape)."""
    losses = {True: [], False: []}
    for e in recorded("gemm_rows.jsonl"):
        _, splits, _, rows = hip.gemm_splits(e["M"], e["N"], e["K"] // 64)
        took = "%d/%d" % (rows, splits)
        assert took == e["rule"] and took in e["us"], e
        losses[e["fit"]].append(e["us"][took] / min(e["us"].values()) - 1)
        assert losses[e["fit"]][-1] <= 0.2, e
    assert len(losses[True]) > 400 and len(losses[False]) > 100 and all(sum(v) / len(v) <= 0.012 for v in losses.values())


def test_fp32_gemm_slices_by_their_record():
    """What the rule takes was timed, is what the record says, and is near the best of each shape: 12 % at most (16 rows of 4096 x
    22528, whose slices are bound by reads that the rule does not tell apart), 1 % on average."""
    losses = []
    for e in recorded("gemm32_slices.jsonl"):
        _, rest, splits, _ = hip._gemm32_plan(e["M"], e["N"], e["K"] // 32)
        took = "%d/%d" % (rest if splits > 1 else 0, splits)
        assert took == e["rule"] and took in e["us"], e
        losses.append(e["us"][took] / min(e["us"].values()) - 1)
        assert losses[-1] <= 0.12, e
    assert len(losses) > 500 and sum(losses) / len(losses) <= 0.01


def test_fp32_gemm_of_short_k_by_its_record():
    """The rule is the record's, and takes what is 0.5 % from the faster of the two on average, 28 % at most (33 x 4096 x 32, 1 us)."""
    losses = []
    for e in recorded("gemm32_short_k.jsonl"):
        assert hip.gemm32_small(e["M"], e["N"], e["K"] // 32) == e["rule"], e
        if e["K"] <= 512:
            losses.append((e["small"] if e["rule"] else e["large"]) / min(e["small"], e["large"]) - 1)
            assert losses[-1] <= 0.29, e
    assert len(losses) > 1300 and sum(losses) / len(losses) <= 0.006


def test_fp32_gemm_in_terms_by_its_record():
    """The plan is the record's and near the best of each shape; the rule takes terms only where they are no slower than the fp32
    instruction, and loses 0.9 % on average against the best plan of the two, 16 % at most.  (W of 24 bits costs up to 60 us
    and 33 %, or 10 %.)"""
    plans, losses = [], []
    for e in recorded("gemm32_terms.jsonl"):
        plan = hip.gemm32_terms(e["M"], e["N"], e["K"] // 32)
        assert (plan is not None) == e["rule"], e
        best = min(e["us"].values())
        took = e["fp32"]
        if e["M"] > 64:
            assert "%d/%d/%d" % hip._gemm32_terms_plan(e["M"], e["N"], e["K"] // 32)[:3] == e["plan"], e
            plans.append(e["us"][e["plan"]] / best - 1)
            assert plans[-1] <= 0.14, e
        if e["rule"]:
            assert "%d/%d/%d" % plan[:3] == e["plan"]
            took = e["us"][e["plan"]]
            assert took <= e["fp32"] and e["bits24"] <= e["fp32"] + max(min(60, 0.33 * e["fp32"]), 0.1 * e["fp32"]), e
        if e["M"] > 64:
            losses.append(took / min(best, e["fp32"]) - 1)
            assert losses[-1] <= 0.16, e
    assert len(plans) > 500 and sum(plans) / len(plans) <= 0.007 and sum(losses) / len(losses) <= 0.009


@pytest.mark.parametrize("M,K,tiles,whole,splits", [(32, 512, 1, 1, 1), (65, 0, 1, 1, 1), (65, 512, 2, 1, 1), (161, 512, 1, 1, 1),
                                                    (65, 512, 1, 0, 17), (65, 512, 1, 2, 1), (65, 528, 1, 1, 1), (65, 512, 0, 0, 1)])
def test_fp32_terms_refuse_what_their_tiles_cannot_hold(M, K, tiles, whole, splits):
    invalid, buffer = 1, 1 << 20  # hipErrorInvalidValue; never read
    assert hip._fn("mrsum_gemm32_terms")(buffer, K, buffer, K, buffer, 16, M, 16, K, tiles, whole, splits, 1, 1, buffer, buffer,
                                         None) == invalid


def test_fp32_tiles_refuse_an_empty_k():
    """The tiles ask for their first K-tile before they look whether there is one; the entry point refuses K 0 on the host."""
    invalid = 1  # hipErrorInvalidValue
    assert hip._fn("mrsum_gemm32")(None, 0, None, 0, None, 16, 4, 16, 0, 0, 1, None, None) == invalid


def c_parameters():
    """Entry point -> number of its parameters, from the kernels' sources."""
    found = {}
    for f in glob.glob(os.path.join(ROOT, "llm_map_reduce_summarizer_amd", "csrc", "kernels", "*.hip")):
        with open(f) as fh:
            for name, pars in re.findall(r"MRSUM_API int (\w+)\(([^)]*)\)\s*\{", fh.read()):
                found[name] = len([p for p in pars.split(",") if p.strip()])
    return found


@pytest.mark.parametrize("rows,heads,vdim,chunks", [
    # token by token and in chunks, us (state 128)
    ([24], 128, 64, False),        # 10.7, 15.2
    ([64], 128, 64, True),         # 19.2, 16.8
    ([900], 128, 64, True),        # 228, 76
    ([40] * 8, 128, 64, False),    # 51, 59
    ([80] * 8, 128, 64, False),    # 87, 95
    ([128] * 8, 128, 64, True),    # 128, 99
    ([1200] * 4, 128, 64, True),   # 559, 340
    ([900], 24, 64, True),         # 209, 72
    ([64] * 40, 128, 128, False),  # 519, 556
    ([], 128, 64, False)])
def test_fp32_scan_in_chunks(rows, heads, vdim, chunks):
    assert hip.ssm_chunk32_rows(rows, heads, vdim) == chunks


@pytest.mark.parametrize("rows,heads,state,chunks", [
    ([40], 128, 128, False),     # 15.3, 16.1
    ([48], 128, 128, False),     # 15.2, 16.2
    ([48], 24, 128, False),      # 14.3, 15.2
    ([56], 128, 128, True),      # 18.7, 16.5
    ([65], 24, 128, True),       # 21.2, 19.6
    ([64] * 4, 24, 128, True),   # 19.3, 16.8
    ([64] * 4, 128, 128, False), # 35.6, 37.0
    ([48], 128, 96, False),      # 14.5, 14.5
    ([48], 128, 64, True),       # 12.4, 11.6
    ([48], 128, 16, True)])      # 12.2, 10.6
def test_fp32_scan_steps_sixteen_rows_at_a_time(rows, heads, state, chunks):
    """us on the GPU, stepped and in chunks, heads of 64."""
    assert hip.ssm_chunk32_rows(rows, heads, 64, state) == chunks


def test_signatures_match_the_kernels():
    """ctypes checks nothing: a signature with another number of arguments reads the rest from the stack."""
    pars = c_parameters()
    assert {n: len(t) for n, t in hip._SIGS.items()} == {n: pars[n] for n in hip._SIGS}


def test_gemm_clock_passes_what_the_gemm_takes():
    spec = importlib.util.spec_from_file_location("gemm_clock", os.path.join(ROOT, "tools", "gemm_clock.py"))
    tool = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(tool)
    x, w, c = torch.zeros(3, 64), torch.zeros(16, 64), torch.zeros(3, 16)
    args = [a.value for a in tool.gemm_args(x, w, c, 99)]
    assert len(args) == c_parameters()["mrsum_gemm"] and args[6:9] == [3, 16, 64]
    # GLU parameters, no tiles in slices, the stream
    assert args[15:] == [float("inf"), 1.0, 0.0, 0, 1, None, 0, 99]


@pytest.mark.parametrize("group_m", [None, 4, 4 | 256, 4 | 512, 255 << 9, -1])
def test_tile_rows_are_those_of_the_plan(group_m, monkeypatch):
    """The caller's raster choice shares a word with the tile's rows, which the scratch of the slices is sized for."""
    M, N, K = 305, 4096, 4096
    whole, splits, room, rows = hip.gemm_splits(M, N, K // 64)
    assert splits > 1 and rows < 256
    passed = []
    monkeypatch.setattr(hip, "_fn", lambda name: lambda *a: passed.append(a) or 0)
    monkeypatch.setattr(hip, "_stream", lambda: 0)
    hip._gemm(None, K, None, K, torch.zeros(M, N, dtype=torch.bfloat16), M, N, K, 0, hip.GEMM_EPI_BF16, None, None, group_m)
    word = passed[0][13]
    assert word >> 9 == rows // 32 and word & 511 == (4 if group_m is None else group_m) & 511
    assert passed[0][18:20] == (whole, splits)


@pytest.mark.parametrize("lens", [[1], [300, 64], [0, 65, 4096, 4096, 1, 700], [64] * 40])
def test_block_items_of_few_and_many_blocks(lens):
    """Work lists built from tuples (few blocks) and from arrays are the same list: latest blocks first, then by sequence."""
    want = sorted(((-qb, i) for i, n in enumerate(lens) for qb in range(0, n, 64)), key=lambda e: e[0])
    got = hip.block_items(lens, 64)
    assert got.dtype == torch.int32 and got.tolist() == [[i, -qb] for qb, i in want]


def test_token_ids_of_one_and_many():
    from llm_map_reduce_summarizer_amd.engine.engine import _token_ids
    for toks in ([7], (7,), [7, 9], range(3), np.arange(4)):
        ids = _token_ids(toks, 10)
        assert ids.dtype == np.int32 and ids.tolist() == list(toks)
    for toks in ([], [10], [-1], [3, 10], [2 ** 70], [-(2 ** 70)]):
        with pytest.raises(ValueError):
            _token_ids(toks, 10)


def test_portion_groups_by_chain_and_load():
    """On both sides of each line: a chain of 48 keys, all walks on 333 workgroups (960 of heads up to 64), width 128."""
    from llm_map_reduce_summarizer_amd.ops.hip import portion_groups
    for portions, hq, hkv, d, want in ((((48, 0),), 32, 8, 128, 1), (((49, 0),), 32, 8, 128, 2), (((45, 4),), 32, 8, 128, 2),
                                       (((1008, 0),), 32, 8, 128, 2), (((1264, 0),), 32, 8, 128, 2), (((1265, 0),), 32, 8, 128, 1),
                                       (((1024, 0),), 32, 8, 64, 2), (((2032, 0),), 32, 8, 64, 2), (((3760, 0),), 32, 8, 64, 2),
                                       (((3761, 0),), 32, 8, 64, 1), (((900, 0),), 32, 8, 132, 1), (((24, 76),) * 32, 32, 8, 128, 1),
                                       (((16, 100),) * 64, 32, 8, 128, 1), (((40, 300),) * 12, 32, 8, 128, 2),
                                       (((100, 0),) * 24, 32, 8, 64, 1), (((400, 0),), 64, 1, 128, 2)):
        assert portion_groups(portions, hq, hkv, d, d) == want, (portions, hq, hkv, d)


def test_new_portions_are_walked_once():
    """Whether they run in tiles and in how many groups are two questions about one walk over them."""
    portions = tuple((7 + i, 1000 + 3 * i) for i in range(20))
    before = hip._portion_walks.cache_info().misses
    hip.portions_in_tiles(portions, 32, 8, 128, 128)
    hip.portion_groups(portions, 32, 8, 128, 128)
    assert hip._portion_walks.cache_info().misses == before + 1


def test_delta_splits_by_their_record():
    """The rule takes what is 0.2 % from the best of the forms on average, 10 % at most."""
    losses = []
    for e in recorded("delta_splits.jsonl"):
        form = hip.delta_waves(e["vdim"], e["dim"], e["heads"] * len(e["lens"]), tuple(-(-n // 64) for n in e["lens"]))
        losses.append(e["us"]["%d/%d" % form] / min(e["us"].values()) - 1)
        assert losses[-1] <= 0.1, e
    assert len(losses) > 1400 and sum(losses) / len(losses) <= 0.002


def test_portion_groups_by_their_record():
    """The rule takes what is 0.3 % from the better of the two on average, 13 % at most."""
    losses = []
    for e in recorded("row_attention_groups.jsonl"):
        us = e["us"][hip.portion_groups(tuple(map(tuple, e["portions"])), *e["heads"]) - 1]
        losses.append(us / min(e["us"]) - 1)
        assert losses[-1] <= 0.13, e
    assert len(losses) > 800 and sum(losses) / len(losses) <= 0.003


def test_portions_in_tiles_by_their_record():
    """The rule takes what is 0.9 % from the better of the two on average, 69 % at most (40 % in fp32)."""
    losses = []
    for e in recorded("row_attention_portions.jsonl"):
        p = e["portions"]
        p = tuple((n, first) for count, n, first in p for _ in range(count)) if e["form"] == "sweep" else tuple(map(tuple, p))
        half = e["dtype"] == "bf16" if e["form"] == "types" else 128 < max(e["heads"][2:]) <= 256
        took = e["tiles_us"] if hip.portions_in_tiles(p, *e["heads"], half) else e["rows_us"]
        losses.append(took / min(e["tiles_us"], e["rows_us"]) - 1)
        assert losses[-1] <= (0.69 if half else 0.41), e
    assert len(losses) > 1800 and sum(losses) / len(losses) <= 0.0086
