"""ISA checks of kernels whose waits or range checks rest on the instructions
the compiler makes, on the CPU (hipcc cross-compiles gfx950).

layer.hip, the decode-step in-projection (gdn_decode_skinny_kernel<0, *>): the
kernel copies x and gamma to LDS with global_load_lds, then issues the
epilogue's EPI small loads (conv taps, cache window, x_n history) and its
MAXSTEPS weight loads, then waits with vmcnt(MAXSTEPS + EPI): vector memory
operations retire in issue order, so that wait covers the LDS copies only if
exactly MAXSTEPS + EPI vector memory operations sit between the last copy and
the wait.  A compiler that moved another load (or a spill) into that window
would let RMSNorm read LDS before the copy lands; this test fails first.
"""

import os
import re
import shutil
import subprocess

import pytest

HIPCC = "/opt/rocm/bin/hipcc"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gdn_18646_amd", "csrc")

VMEM = re.compile(r"^\s*(buffer|global|scratch|flat)_(load|store|atomic)")


def _assembly(source, tmp_path_factory, *flags):
    if not shutil.which(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("isa") / "out.s"
    cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", *flags, "--cuda-device-only", "-S", os.path.join(CSRC, source), "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True, timeout=600)
    return out.read_text()


@pytest.fixture(scope="module")
def layer_asm(tmp_path_factory):
    return _assembly("layer.hip", tmp_path_factory)


@pytest.fixture(scope="module")
def prefill_asm(tmp_path_factory):
    return _assembly("prefill.hip", tmp_path_factory, "-mllvm", "-amdgpu-mfma-vgpr-form")


def _function(asm, symbol):
    start = asm.index(f"\n{symbol}:")
    return asm[start:asm.index("\n.Lfunc_end", start)].splitlines()


@pytest.mark.parametrize("maxsteps", [8, 16])
def test_in_proj_dma_wait_covers_only_the_weight_loads(layer_asm, maxsteps):
    sym = f"_ZN12_GLOBAL__N_124gdn_decode_skinny_kernelILi0ELi{maxsteps}EEEvNS_12SkinnyParamsE"
    body = _function(layer_asm, sym)
    last_dma = max(i for i, ln in enumerate(body) if "global_load_lds_dwordx4" in ln)
    wait = next(i for i in range(last_dma, len(body)) if re.search(r"s_waitcnt vmcnt\(\d+\)", body[i]))
    n = int(re.search(r"vmcnt\((\d+)\)", body[wait]).group(1))
    between = [ln.strip() for ln in body[last_dma + 1:wait] if VMEM.match(ln)]
    epi = 9  # kEpiLoads in layer.hip: 7 global_load_ushort + 2 global_load_dwordx4
    assert n == maxsteps + epi, f"first wait after the copies is vmcnt({n}), expected vmcnt({maxsteps + epi})"
    assert len(between) == maxsteps + epi, between
    assert sum(ln.startswith("buffer_load_dwordx4") for ln in between) == maxsteps, between
    assert all(ln.startswith(("buffer_load_dwordx4", "global_load_ushort", "global_load_dwordx4")) for ln in between)
    assert not any("scratch_" in ln for ln in body), "the kernel spills"


def test_tile_kernels_keep_their_ring_waits_and_do_not_spill(layer_asm):
    """The decode-step tile kernels (gdn_decode_tile_kernel<MODE, NC, TN>)
    order their LDS ring by explicit vmcnt waits that count the copies a
    slice issues (two per wave: one of A, one of W, also for 32-wide tiles,
    whose W copy runs on lanes 0..31 of every wave): vmcnt(6) after the four
    slots are issued and vmcnt(4) in the loop.  Every instantiation must keep
    both waits, issue its copies as global_load_lds_dwordx4 only, and not
    spill (a spill's scratch access inside the loop would shift the count)."""
    syms = sorted(set(re.findall(r"^(_ZN12_GLOBAL__N_122gdn_decode_tile_kernel\w+):", layer_asm, re.M)))
    assert len(syms) == 9, syms  # in-projection NC 0..3 x TN 32, 64; out-projection TN 32
    for sym in syms:
        body = _function(layer_asm, sym)
        text = "\n".join(body)
        assert "scratch_" not in text, f"{sym} spills"
        waits = re.findall(r"s_waitcnt vmcnt\((\d+)\)", text)
        assert "6" in waits and "4" in waits, (sym, waits)
        assert any("global_load_lds_dwordx4" in ln for ln in body), sym
        assert not any(re.search(r"global_load_lds_dword(x2|x3)?\s", ln) for ln in body), sym


def test_intra_kernel_loads_are_range_checked_whole(prefill_asm):
    """gdn_prefill_intra_kernel takes K and Q rows past a sequence's end as
    zeros from the buffer resource's range check.  That check covers the lane
    and the immediate offset but not the scalar one, so no load may carry part
    of its row in a scalar offset (it would read the rows behind the tensor's
    sequence, or behind the tensor).  16 loads of K, and 16 of Q in the
    instantiation that forms Aq."""
    syms = sorted(set(re.findall(r"^(_ZN12_GLOBAL__N_124gdn_prefill_intra_kernel\w+):", prefill_asm, re.M)))
    assert len(syms) == 2, syms
    for sym, n in zip(syms, (16, 32)):  # <false>, <true>
        loads = [ln.split(";")[0] for ln in _function(prefill_asm, sym) if "buffer_load" in ln]
        assert len(loads) == n, (sym, loads)
        for ln in loads:
            assert re.search(r"buffer_load_dwordx4 v\[\d+:\d+\], v\d+, s\[\d+:\d+\], 0 offen", ln), (sym, ln)
