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

from tests.proj_tiles import ARGS

HIPCC = "/opt/rocm/bin/hipcc"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gdn_18646_amd", "csrc")

VMEM = re.compile(r"^\s*(buffer|global|scratch|flat)_(load|store|atomic)")


def _assembly(source, tmp_path_factory, *flags):
    if not shutil.which(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("isa") / "out.s"
    cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", *flags, "--cuda-device-only", "-S", "-I", CSRC, os.path.join(CSRC, source), "-o", str(out)]
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


@pytest.fixture(scope="module")
def proj_asm(tmp_path_factory):
    """Every tile of the projection kernel (equal lengths)."""
    src = tmp_path_factory.mktemp("isa") / "tiles.hip"
    lines = [f"template __global__ void gdn_proj_conv_mfma_kernel<gdn_proj::{t}, 0>(gdn_proj::ProjParams, int, int);"
             for t in ARGS]
    src.write_text('#include "proj_mfma.hpp"\nnamespace {\n' + "\n".join(lines) + "\n}\n")
    return _assembly(str(src), tmp_path_factory)


def _tile_function(asm, args):
    cw, tw, wmt, wnt, ns, per_cu, phased, ks, kd = args
    t = f"8ProjTileILi{cw}ELi{tw}ELi{wmt}ELi{wnt}ELi{ns}ELi{per_cu}ELb{phased}ELi{ks}ELi{kd}EEE"
    return _function(asm, f"_ZN12_GLOBAL__N_125gdn_proj_conv_mfma_kernelINS_{t}Li0EEEvN8gdn_proj10ProjParamsEii")


def _events(body):
    """The copies into LDS ('c'), other vector memory operations ('m'), vmcnt waits (n) and barriers ('b')."""
    ev = []
    for ln in body:
        wait = re.match(r"\s*s_waitcnt .*vmcnt\((\d+)\)", ln)
        if "global_load_lds_dwordx4" in ln:
            ev.append("c")
        elif VMEM.match(ln):
            ev.append("m")
        elif wait:
            ev.append(int(wait.group(1)))
        elif re.match(r"\s*s_barrier", ln):
            ev.append("b")
    return ev


def _blocks(body):
    """Basic blocks: [(lines, successors)], a successor's last line of a conditional branch first."""
    starts, label = {0}, {}
    for i, ln in enumerate(body):
        if m := re.match(r"(\.LBB\w+):", ln):
            label[m.group(1)] = i
            starts.add(i)
        if re.match(r"\s*s_(c?branch|endpgm)", ln):
            starts.add(i + 1)
    starts = sorted(x for x in starts if x < len(body))
    index = {i: k for k, i in enumerate(starts)}
    blocks = []
    for k, i in enumerate(starts):
        lines = body[i:starts[k + 1] if k + 1 < len(starts) else len(body)]
        m = re.match(r"\s*s_(c?branch\w*) (\.LBB\w+)", lines[-1])
        after = [k + 1] if k + 1 < len(starts) else []
        if m:
            succ = [index[label[m.group(2)]]] + (after if m.group(1) != "branch" else [])
        else:
            succ = [] if "s_endpgm" in lines[-1] else after
        blocks.append((lines, succ))
    return blocks


def _copy_loop(body):
    """The blocks of the loop that issues copies, and all blocks."""
    blocks = _blocks(body)

    def reach(k):
        seen, todo = set(), list(blocks[k][1])
        while todo:
            x = todo.pop()
            if x not in seen:
                seen.add(x)
                todo += blocks[x][1]
        return seen

    copying = [k for k, (lines, _) in enumerate(blocks) if "c" in _events(lines)]
    loops = []
    for k in copying:
        forward = reach(k)
        if k in forward:
            loops.append(frozenset(x for x in forward if k in reach(x)))
    assert len(set(loops)) == 1, loops
    return loops[0], blocks


@pytest.mark.parametrize("tile", [t for t, a in ARGS.items() if a[6]])
def test_phased_projection_tiles_keep_their_counted_waits(proj_asm, tile):
    """The two-group loop of the projection kernel refills a stage's buffer
    region by region (first and second part of the tokens and columns, in the
    order X0, W0, W1, X1) and waits, before the barrier that opens a phase, for
    the region the next phase reads, by counting the copies issued after it.
    The counts hold only for these copies in this order: none moved over a
    wait, merged or dropped, in the loop and in the stages after the last issued
    one, no other vector memory operation in the loop, and no spill."""
    cw, tw, wmt, wnt, ns, *_ = ARGS[tile]
    m0, x0 = wmt // 2, (wnt + 1) // 2
    groups = [2 * tw * x0, 2 * cw * m0, 2 * cw * (wmt - m0), 2 * tw * (wnt - x0)]  # 8-row copies, split over 8 waves
    n = [g // 8 + g % 8 // 4 for g in groups]
    every = sum(n)
    body = _tile_function(proj_asm, ARGS[tile])
    assert not any("scratch_" in ln for ln in body), "the kernel spills"
    loop, blocks = _copy_loop(body)
    # once round the loop; a branch over a copy of half the lanes (execz) is never taken, every wave has them
    k = start = min(loop)
    got = []
    while True:
        lines, succ = blocks[k]
        got += _events(lines)
        inside = [x for x in succ if x in loop]
        if "s_cbranch_execz" in lines[-1]:
            inside = inside[1:]
        assert len(inside) == 1, lines[-1]
        k = inside[0]
        if k == start:
            break
    want = (["c"] * n[3] + [n[3] + (ns - 1) * every, "b", "b"] + ["c"] * n[0] + [n[0] + (ns - 1) * every, "b", "b"]
            + ["c"] * n[1] + ["b", "b"] + ["c"] * n[2] + [n[2] + (ns - 1) * every, "b", "b"])
    assert any(got == want[i:] + want[:i] for i in range(len(want))), got
    # the ring's filling (all but X1 of its last stage, which the first stage of the drain issues) and its wait
    events = _events(body)
    assert events.count("c") == (ns + 1) * every
    assert n[2] + (ns - 1) * every in events[events.index("c"):]
    # the stages after the last issued one, t of them left: each is straight code
    for t in range(ns):
        stage = [n[3] + t * every, "b", "b", t * every, "b", "b", "b", "b"]
        stage += [n[2] + n[3] + (t - 1) * every, "b"] if t else []
        assert any(events[i:i + len(stage)] == stage for i in range(len(events))), (t, stage)


@pytest.mark.parametrize("tile", [t for t, a in ARGS.items() if not a[6]])
def test_ring_projection_tiles_keep_their_counted_wait(proj_asm, tile):
    """The other tiles fill all but one of the ring's NS stages, then a loop
    iteration waits until the copies of at most NS - 2 stages are in flight (or
    for all near the end) and issues one stage's."""
    cw, tw, wmt, wnt, ns, _, _, ks, kd = ARGS[tile]
    copies = kd * 16 * (cw * wmt + tw * wnt) // 8 // (cw * tw)  # a wave's, a stage
    body = _tile_function(proj_asm, ARGS[tile])
    assert not any("scratch_" in ln for ln in body), "the kernel spills"
    loop, blocks = _copy_loop(body)
    inside = [e for k in sorted(loop) for e in _events(blocks[k][0])]
    assert "m" not in inside and inside.count("c") >= copies, inside
    assert {e for e in inside if isinstance(e, int)} == {0, (ns - 2) * copies}, inside
