"""Compile-only check of the register allocation of the hot kernels: a tile kernel that spills
VGPRs to scratch runs several times slower and no numerics test notices.  Needs hipcc, no GPU."""
import concurrent.futures
import os
import re
import shutil
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cudaintro_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")
FLAGS = ["-O3", "-std=c++17", "--offload-arch=gfx950", "-fvisibility=hidden", "-Xclang",
         "-target-feature", "-Xclang", "-packed-fp32-ops", "-ffp-contract=off", "-Wno-inline-asm",
         f"-I{os.path.join(ROOT, 'include')}", f"-I{CSRC}", "--offload-device-only", "-S"]


FILES = ("gemm_16b.hip", "gemm_i8.hip", "gemm_f32.hip", "gemm_any_tile.hip", "gemm_skinny.hip", "gemm_kwaves.hip",
         "gemm_panel.hip", "gemm_f32_small.hip", "probe.hip", "probe_paired.hip")


@pytest.fixture(scope="module")
def assembly():
    """{file: its gfx950 assembly}, each compiled once."""
    def compiled(d, name):
        out = os.path.join(d, name + ".s")
        subprocess.run([HIPCC, *FLAGS, os.path.join(CSRC, name), "-o", out], check=True,
                       stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
        with open(out) as f:
            return f.read()
    with tempfile.TemporaryDirectory() as d, concurrent.futures.ThreadPoolExecutor(8) as pool:
        return dict(zip(FILES, pool.map(lambda name: compiled(d, name), FILES)))


def kernels(text):
    """(name, code) of every kernel of an assembly file."""
    for body in re.split(r"\n(?=_Z\w+:)", text):
        code = body.split(".Lfunc_end")[0]
        if "s_endpgm" in code:
            yield body.split(":", 1)[0], code


def spill_counts(text):
    res, name = {}, None
    for line in text.split("\n"):
        m = re.match(r"\s+\.name:\s+(\S+)", line)
        if m:
            name = m.group(1)
        m = re.match(r"\s+\.vgpr_spill_count:\s+(\d+)", line)
        if m and name:
            res[name] = int(m.group(1))
    return res


@pytest.mark.skipif(HIPCC is None, reason="hipcc not installed")
def test_hot_kernels_do_not_spill(assembly):
    spills = {k: v for text in assembly.values() for k, v in spill_counts(text).items()}
    assert len(spills) > 60          # every template instance was seen
    assert sum("kwaves_kernelINS" in k for k in spills) >= 10
    assert sum("panel_kernel" in k for k in spills) == 10
    assert sum("mfma_tile_kernelINS0_7MathF32E" in k for k in spills) >= 63    # seven heights, both forms
    for name, n in spills.items():
        if re.search(r"EpiDequantX4ILb[01]ELb1", name):
            assert n <= 160, (name, n)     # accumulator-dump variants (a test aid)
        elif "issue_cost_kernel" in name:
            assert n <= 12, (name, n)      # (set-up values, spilled once outside the timed loop)
        elif re.search(r"MathI8ELi2ELi4ELi4ENS_12EpiDequantX4ILb[01]ELb0EEELi2ELb1E", name):
            assert n <= 2, (name, n)       # (256-row tiles at any alignment with scales: in the epilogue)
        else:
            assert n == 0, (name, n)


@pytest.mark.skipif(HIPCC is None, reason="hipcc not installed")
def test_cross_workgroup_exchange_uses_agent_scope_accesses(assembly):
    """The decode kernels' K ranges meet through memory written by one workgroup and read by
    another, possibly on another XCD whose L2 is not coherent with the writer's.  The code relies
    on every such access being an agent-scope atomic, which gfx950 encodes as a load / store with
    the sc1 bit (served at the memory-side point of coherence, never by the local L2), and on
    there being NO whole-cache write-back or invalidate in those kernels (55 us per call).  A
    compiler that stopped encoding either would break results only under particular timing; this
    checks the generated code instead."""
    seen = 0
    for name, body in kernels(assembly["gemm_skinny.hip"]):
        if "skinny_kn16_kwaves_kernel" not in name and "skinny_kernelI" not in name:
            continue
        if re.search(r"skinny_kernelI.*ELi1EEEviii", name):
            continue                       # one K range: nothing is exchanged
        seen += 1
        assert not re.search(r"\bbuffer_wbl2\b|\bbuffer_inv\b", body), name
        # partial sums: 8-byte agent-scope stores and loads; the arrival counter: an atomic add
        assert re.search(r"global_store_dwordx2 .* sc1", body), name
        assert re.search(r"global_load_dwordx2 .* sc1", body), name
        assert re.search(r"global_atomic_(add|swap)", body), name
    assert seen >= 12


@pytest.mark.skipif(HIPCC is None, reason="hipcc not installed")
def test_kernel_of_small_outputs_exchanges_at_agent_scope(assembly):
    """The same for the K ranges of gemm_kwaves.hip: 8-byte sc1 stores and loads for the sums, an
    atomic add for the arrivals, every store acknowledged (vmcnt 0) before it, no whole-cache operation."""
    seen = 0
    for name, code in kernels(assembly["gemm_kwaves.hip"]):
        if "kwaves_kernelINS" not in name:
            continue
        seen += 1
        assert not re.search(r"\bbuffer_wbl2\b|\bbuffer_inv\b", code), name
        words = 2 if "MathF32E" in name else 4          # 8-byte words of a thread's sums
        stores = [m.end() for m in re.finditer(r"global_store_dwordx2 .* sc1", code)]
        assert len(stores) == words, (name, len(stores))
        assert len(re.findall(r"global_load_dwordx2 .* sc1", code)) >= 8 * words, name
        add = code.index("global_atomic_add")
        assert stores[-1] < add and "vmcnt(0)" in code[stores[-1]:add], name
    assert seen >= 10


@pytest.mark.skipif(HIPCC is None, reason="hipcc not installed")
def test_fp32_tiles_have_both_kinds_of_stores(assembly):
    """The fp32 tile kernel stores rows of whole lines with streaming stores and others with plain ones
    (tile_plan.h, store_streams; tiles of 64 rows stream all).  The compiler may join two branches that
    end in the same stores, and the joined ones are plain: half of the 16-byte stores of each instance
    must carry the nt bit (64 rows: all)."""
    seen = 0
    for name, code in kernels(assembly["gemm_f32.hip"]):
        if "mfma_tile_kernelINS0_7MathF32E" not in name:
            continue
        stores = re.findall(r"global_store_dwordx4 .*", code)
        seen += 1
        tall = "MathF32ELi3ELi4ELi2E" not in name
        assert stores and (1 + tall) * sum(" nt" in s for s in stores) == len(stores), (name, len(stores))
    assert seen >= 42      # seven heights x (partial sums, plain, four epilogues)
