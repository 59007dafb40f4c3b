#!/usr/bin/env python3
"""In-kernel clock of the bf16 prefill GEMM (gemm_bf16.hip) under sustained load, against its wall-clock TF/s and
hipBLASLt's (torch.matmul) on the same shapes.

MFMA-dense loops on random data run well under the 2.4 GHz the 2.5 PF/s bf16 peak is quoted at
(MI355X_MICROARCH.md, 'DVFS give-back'), so the useful ceiling of a GEMM is peak x (held clock / 2.4 GHz).
A diagnostic build of it (-DMRSUM_CLOCK_STAMPS: s_memtime / s_memrealtime around each workgroup,
stored by one lane to a buffer nothing else reads) measures that clock after >= 2 s of back-to-back
launches.  The production library is not touched: ``--build`` writes _native/diag/libmrsum_gemm_clock.so."""
import argparse
import ctypes
import json
import os
import statistics
import subprocess
import sys
import time

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
KERNELS = os.path.join(ROOT, "llm_map_reduce_summarizer_amd", "csrc", "kernels")
SRC = [os.path.join(KERNELS, f) for f in ("gemm.hip", "gemm_bf16.hip")]
LIB = os.path.join(ROOT, "llm_map_reduce_summarizer_amd", "_native", "diag", "libmrsum_gemm_clock.so")
SHAPES = {"qkv": (6144, 4096), "o": (4096, 4096), "gate_up": (28672, 4096), "down": (4096, 14336)}


def build():
    from llm_map_reduce_summarizer_amd import _stamp
    os.makedirs(os.path.dirname(LIB), exist_ok=True)
    flags = [f for f in _stamp.HIP_FLAGS if not f.startswith("-Rpass")]
    subprocess.check_call(["/opt/rocm/bin/hipcc"] + flags + ["-shared", "-DMRSUM_CLOCK_STAMPS"] + SRC + ["-o", LIB])
    print("built", LIB)


def gemm_args(x, w, c, stream):
    """Arguments of mrsum_gemm for c = x w^T in bf16, every tile whole; refused if the entry point takes others."""
    from llm_map_reduce_summarizer_amd.ops import hip
    (M, K), N = x.shape, w.shape[0]
    args = (x.data_ptr(), K, w.data_ptr(), K, c.data_ptr(), N, M, N, K, 0, hip.GEMM_EPI_BF16, None, None, 0, 0,
            *hip.SWIGLU, 0, 1, None, 0, stream)
    types = hip._SIGS["mrsum_gemm"]
    if len(args) != len(types):
        raise TypeError("mrsum_gemm takes %d arguments, not %d" % (len(types), len(args)))
    return [t(v) for t, v in zip(types, args)]


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--build", action="store_true")
    ap.add_argument("--M", type=int, default=16384)
    ap.add_argument("--roles", default="qkv,o,gate_up,down")
    ap.add_argument("--seconds", type=float, default=2.5)
    a = ap.parse_args()
    if a.build:
        return build()
    import torch
    from llm_map_reduce_summarizer_amd.ops import hip
    lib = ctypes.CDLL(LIB)
    lib.mrsum_gemm.argtypes = hip._SIGS["mrsum_gemm"]
    lib.mrsum_gemm_stamps.argtypes = [ctypes.c_void_p, ctypes.c_int]
    dev = torch.device("cuda:0")
    stream = torch.cuda.current_stream().cuda_stream
    for role in a.roles.split(","):
        N, K = SHAPES[role]
        M = a.M
        g = torch.Generator(device="cpu").manual_seed(1)
        x = (torch.randn(M, K, generator=g) * 0.5).to(torch.bfloat16).to(dev)
        w = (torch.randn(N, K, generator=g) * 0.02).to(torch.bfloat16).to(dev)
        c = torch.empty(M, N, dtype=torch.bfloat16, device=dev)

        args = gemm_args(x, w, c, stream)

        def run():
            rc = lib.mrsum_gemm(*args)
            assert rc == 0, rc

        flop = 2.0 * M * N * K
        res = {"role": role, "M": M, "N": N, "K": K}
        for name, fn in (("own", run), ("hipblaslt", lambda: torch.matmul(x, w.t(), out=c))):
            t_end = time.time() + a.seconds
            n = 0
            while time.time() < t_end:  # sustained load first: the clock it holds, not the idle one
                for _ in range(10):
                    fn()
                torch.cuda.synchronize()
                n += 10
            ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            ev0.record()
            for _ in range(20):
                fn()
            ev1.record()
            torch.cuda.synchronize()
            us = ev0.elapsed_time(ev1) * 1000 / 20
            res[name + "_us"] = round(us, 1)
            res[name + "_tflops"] = round(flop / us / 1e6, 1)
            if name == "own":
                buf = (ctypes.c_ulonglong * (2 * 4096))()
                nw = lib.mrsum_gemm_stamps(buf, 2 * 4096)
                clk = [buf[2 * i] / buf[2 * i + 1] * 0.1 for i in range(nw // 2) if buf[2 * i + 1]]
                res["own_clock_ghz_median"] = round(statistics.median(clk), 3)
                res["own_clock_ghz_min_max"] = [round(min(clk), 3), round(max(clk), 3)]
                # the dense bf16 peak (2.5 PF/s at 2.4 GHz) scaled to the clock held
                res["peak_at_held_clock_tflops"] = round(2500 * statistics.median(clk) / 2.4, 1)
                res["own_pct_of_held_clock_peak"] = round(100 * res["own_tflops"] / res["peak_at_held_clock_tflops"], 1)
        print(json.dumps(res), flush=True)


if __name__ == "__main__":
    sys.exit(main())
