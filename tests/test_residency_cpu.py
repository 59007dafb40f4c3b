"""Workgroups that fit a compute unit by their registers and LDS, as the compiler reports them, where launch rules count on them."""

import functools
import os
import re
import subprocess

import pytest

from llm_map_reduce_summarizer_amd import _stamp

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")


@functools.lru_cache(maxsize=None)
def reported(source):
    """Mangled name -> (registers of a wave, LDS bytes of a workgroup)."""
    r = subprocess.run([HIPCC, *_stamp.HIP_FLAGS, "-c", os.path.join(_stamp.CSRC, "kernels", source), "-o", os.devnull],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, check=True)
    out, name, seen = {}, None, {}
    for line in r.stdout.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            name, seen = m[1], {}
        m = re.search(r" (VGPRs|AGPRs|LDS Size \[bytes/block\]): (\d+)", line)
        if m and name:
            seen[m[1]] = int(m[2])
            if len(seen) == 3:
                out[name] = (-(-seen["VGPRs"] // 4) * 4 + seen["AGPRs"], seen["LDS Size [bytes/block]"])
    return out


def workgroups(source, kernel, threads):
    """How many workgroups of ``threads`` a CU holds: 512 registers a lane and SIMD in pieces of 8, 160 KiB of LDS."""
    found = [v for k, v in reported(source).items() if kernel in k]
    assert len(found) == 1, (kernel, found)
    regs, lds = found[0]
    waves = 4 * min(8, 512 // (-(-regs // 8) * 8))
    return min(waves // (threads // 64), 160 * 1024 // max(lds, 1))


def test_delta_workgroups_as_their_plan_counts_them():
    """Every form of the chunked delta rule: as many workgroups on a CU as ops/hip.py has in DELTA_FORMS."""
    from llm_map_reduce_summarizer_amd.ops.hip import DELTA_FORMS
    for dim, forms in DELTA_FORMS.items():
        for (blocks, pair), (_, fit) in forms.items():
            kernel = "delta_chunk_%skernelILi%dELi%dE" % ("pair_" if pair else "", dim // 32, blocks)
            assert workgroups("delta_chunk.hip", kernel, 64 * blocks * (1 + pair)) == fit, (dim, blocks, pair)


def test_delta_pairs_of_narrow_heads():
    assert workgroups("delta_chunk.hip", "delta_chunk_pair_kernelILi1ELi4E", 512) == 2


@pytest.mark.parametrize("PW,NB,scan_wave,want", [(1, 8, 0, 2), (1, 4, 0, 4), (1, 4, 1, 3), (1, 1, 1, 4), (1, 2, 1, 4), (2, 1, 1, 3),
                                                  (2, 2, 1, 3), (2, 4, 1, 2)])
def test_state_passes_of_the_chunked_scan(PW, NB, scan_wave, want):
    """Two of each run at a time, which is what segments are cut for (SSM_WGS), and all of 768 with a wave that only scans; of
    64 x 128 states all that there can be without it."""
    kernel = "ssm_chunk_kernelILi%dELi%dELb1ELb%dE" % (PW, NB, scan_wave)
    assert workgroups("ssm_chunk.hip", kernel, 320 if scan_wave else 256) >= want
