"""Checks on the compiled gfx950 code (CPU only: hipcc cross-compiles).

The GEMMs issue their LDS DMAs (`buffer_load_dwordx4 ... lds`) from inline asm, which
the compiler's hazard recognizer cannot see into.  A VALU write of an SGPR (for
example a `v_readlane` reloading a spilled resource or offset SGPR) needs 5 wait
states before a vector memory instruction reads that SGPR; the asm supplies them
itself.  Missing wait states made loads use stale offsets (wrong results at
k/q_proj M=512 in an earlier build), so every such pair is checked here, along with
the properties the kernel's manual ordering relies on.
"""

import re

import pytest

from helios_amd import build as hbuild

WAIT_STATES = 5


def _kernels(asm: str, kernel: str = "gemm_kernel"):
    for m in re.finditer(rf"\n(_ZN\S*{kernel}\S*):[^\n]*\n", asm):
        body = asm[m.end():asm.index("s_endpgm", m.end())]
        lines = [l.strip() for l in body.splitlines()
                 if l.strip() and not l.strip().startswith((";", "."))]
        yield m.group(1), lines


def _sgprs(tok: str):
    m = re.match(r"s\[(\d+):(\d+)\]$", tok)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.match(r"s(\d+)$", tok)
    if m:
        return {int(m.group(1))}
    return {"m0"} if tok == "m0" else set()


@pytest.fixture(scope="module")
def gemm_asm():
    return hbuild.device_asm("q4_gemm.hip")


@pytest.fixture(scope="module")
def kpair_asm():
    return hbuild.device_asm("q4_gemm_kpair.hip")


def test_kpair_dma_sgpr_hazards_covered(kpair_asm):
    kernels = list(_kernels(kpair_asm, "kpair_kernel"))
    assert len(kernels) == 6  # tiles of 32, 48, .. 112 rows
    _check_dma_hazards(kernels)


def test_lds_dma_sgpr_hazards_covered(gemm_asm):
    kernels = list(_kernels(gemm_asm))
    # bf16 / fp32 outputs, bf16 / fp32 GeGLU pairs, bf16 / fp32 outputs with a LoRA
    # delta; 256 and 128 x 256 tiles, the 256-row tile's fp16 form and the 128- and
    # 256-row tiles' one-pass 8-bit form
    assert len(kernels) == 30
    assert sum("ELi256ELi256ELi1E" in name for name, _ in kernels) == 6
    assert sum("ELi256ELi2E" in name for name, _ in kernels) == 12
    _check_dma_hazards(kernels)


def _check_dma_hazards(kernels):
    for name, lines in kernels:
        dmas = 0
        for i, line in enumerate(lines):
            if not (line.startswith("buffer_load_dwordx4") and " lds" in line):
                continue
            dmas += 1
            used = set().union(*[_sgprs(t.strip(",")) for t in line.split()[1:]]) | {"m0"}
            waits, j = 0, i - 1
            while j >= 0 and waits < WAIT_STATES:
                op = lines[j].split()[0]
                if op == "s_nop":
                    waits += int(lines[j].split()[1]) + 1
                else:
                    if op.startswith("v_"):
                        dst = lines[j].split()[1].rstrip(",")
                        assert not (_sgprs(dst) & used), f"{name}: {lines[j]!r} feeds {line!r} within {waits} wait states"
                    waits += 1
                j -= 1
        assert dmas > 0, name


@pytest.mark.parametrize("asm", ["gemm_asm", "kpair_asm"])
def test_no_spills_and_lds_budget(asm, request):
    # scratch spills would be VMEM loads counted by the kernel's manual vmcnt waits
    asm = request.getfixturevalue(asm)
    for field in ("vgpr_spill_count", "private_segment_fixed_size"):
        vals = [int(v) for v in re.findall(rf"\.{field}:\s+(\d+)", asm)]
        assert len(vals) >= 6 and max(vals) == 0, (field, vals)
    lds = [int(v) for v in re.findall(r"\.group_segment_fixed_size:\s+(\d+)", asm)]
    assert max(lds) <= 160 * 1024


def test_kpair_register_budget(kpair_asm):
    """Two waves per SIMD (one 512-thread workgroup per CU): at most 256 VGPRs, and all of
    a step's words and accumulators in registers."""
    meta = [(n, v, p) for n, v, p in _kernel_meta(kpair_asm) if "kpair_kernel" in n]
    assert len(meta) == 6
    for name, vgprs, private in meta:
        assert private == 0 and vgprs <= 256, f"{name}: {vgprs} VGPRs"


# --------------------------------------------------------------- LDS DMAs and barriers

_COUNTED = re.compile(r"(buffer|global|flat|scratch)_(load|store|atomic)")


def _blocks(asm: str, kernel: str):
    """The kernel's code as basic blocks: [(instructions, successors)], the entry first."""
    m = re.search(rf"\n(\S*{kernel}\S*):[^\n]*\n", asm)
    body = asm[m.end():asm.index(".section", m.end())]
    blocks, names = [[]], {}
    for line in body.splitlines():
        line = line.split(";")[0].strip()
        label = re.match(r"(\.LBB\w+):$", line)
        if label:
            if blocks[-1]:
                blocks.append([])
            names[label.group(1)] = len(blocks) - 1
        elif line and not line.startswith((".", "#")):
            blocks[-1].append(line)
            if line.startswith(("s_branch", "s_cbranch", "s_endpgm")):
                blocks.append([])
    out = []
    for i, ins in enumerate(blocks):
        last = ins[-1] if ins else ""
        nxt = [names[last.split()[1]]] if last.startswith(("s_branch", "s_cbranch")) else []
        if not last.startswith(("s_branch", "s_endpgm")) and i + 1 < len(blocks):
            nxt.append(i + 1)
        out.append((ins, nxt))
    return out


def _dmas_in_flight_at_barriers(asm: str, kernel: str):
    """Barriers that some path reaches with an LDS DMA of the wave still in flight, as
    (the barrier's text with its block's last instructions, loads issued after the DMA).
    Memory operations return in order, so a DMA followed by n of them has landed at a
    wait for vmcnt <= n; per block the worst path (the fewest operations after a DMA)."""
    blocks = _blocks(asm, kernel)
    state, work, bad, dmas = {0: None}, [0], {}, 0
    while work:
        b = work.pop()
        after = state[b]  # operations after the newest DMA in flight; None: none in flight
        for i, ins in enumerate(blocks[b][0]):
            if _COUNTED.match(ins):
                if re.search(r"\blds\b", ins):
                    after, dmas = 0, dmas + 1
                elif after is not None:
                    after = min(after + 1, 64)
            elif ins.startswith("s_waitcnt"):
                n = re.search(r"vmcnt\((\d+)\)", ins)
                if n and after is not None and int(n.group(1)) <= after:
                    after = None
            elif ins.startswith("s_barrier") and after is not None:
                bad[(b, i)] = after
        for n in blocks[b][1]:
            old = state.get(n, "new")
            new = after if old in ("new", None) else old if after is None else min(old, after)
            if old == "new" or new != old:
                state[n] = new
                work.append(n)
    assert dmas > 0, kernel
    return bad


@pytest.mark.parametrize("kmt", [2, 3, 4, 5, 6, 7])
def test_kpair_x_has_landed_at_every_barrier(kpair_asm, kmt):
    """Waves of the kpair GEMM read x rows that other waves' DMAs bring, so every DMA a
    wave issued has landed when it reaches the next barrier.  The waits count the loads
    issued after the DMAs: eight before the first step, ten in every later one."""
    assert _dmas_in_flight_at_barriers(kpair_asm, f"kpair_kernelILi{kmt}E") == {}


def _kernel_meta(asm: str):
    """(name, vgpr_count, spill bytes) of every kernel in the metadata block."""
    for m in re.finditer(r"- \.agpr_count:.*?\.name:\s+(\S+).*?\.private_segment_fixed_size:\s+(\d+).*?"
                         r"\.vgpr_count:\s+(\d+)", asm, re.S):
        yield m.group(1), int(m.group(3)), int(m.group(2))


def test_decode_register_budgets():
    asm = hbuild.device_asm("q4_decode.hip")
    meta = list(_kernel_meta(asm))
    assert any("decode_stream_kernel" in n for n, _, _ in meta)
    for name, vgprs, private in meta:
        assert private == 0, f"{name} spills to scratch"
        stream = re.search(r"decode_stream_kernelILi\d+ELi\d+ELi(\d+)E", name)
        if stream:
            # two buffers: two 8-wave workgroups per CU (the launcher's occupancy
            # assumption); four buffers are launched only at one workgroup per CU
            limit = 128 if stream.group(1) == "2" else 256
            assert vgprs <= limit, f"{name}: {vgprs} VGPRs"
        if "decode_rows_kernel" in name:
            # two waves per SIMD (two 4-wave workgroups per CU)
            assert vgprs <= 256, f"{name}: {vgprs} VGPRs"


def test_limb_register_budgets():
    """decode_limb_kernel's launch shapes (q4_limbs.hip limb_config) assume its
    occupancy: three 8-wave workgroups per CU for one chunk in flight (6 waves per
    SIMD: at most 85 VGPRs), one 16-wave workgroup per CU (4 per SIMD: 128)."""
    asm = hbuild.device_asm("q4_limbs.hip")
    meta = [(n, v, p) for n, v, p in _kernel_meta(asm) if "decode_limb_kernel" in n]
    assert len(meta) == 3
    for name, vgprs, private in meta:
        assert private == 0, f"{name} spills to scratch"
        nbuf, waves = map(int, re.search(r"decode_limb_kernelILi(\d+)ELi(\d+)E", name).groups())
        limit = 85 if nbuf == 1 else (128 if waves == 16 else 256)
        assert vgprs <= limit, f"{name}: {vgprs} VGPRs"


def test_limb_rows_register_budgets():
    """decode_limb_rows_kernel: no scratch; the 16-wave instance dealt round the grid at
    4 rows runs two workgroups per CU (8 waves per SIMD: at most 64 VGPRs); the rest
    run one 16-wave workgroup per CU (at most 128; the two phased ones, BATCH > 0,
    among them) or 8-wave ones."""
    asm = hbuild.device_asm("q4_limbs.hip")
    meta = [(n, v, p) for n, v, p in _kernel_meta(asm) if "decode_limb_rows_kernel" in n]
    assert len(meta) == 11
    assert sum(bool(re.search(r"ELb1ELi[1-9]\d*E", n)) for n, _, _ in meta) == 2
    for name, vgprs, private in meta:
        assert private == 0, f"{name} spills to scratch"
        mt, nbuf, waves = map(int, re.search(r"decode_limb_rows_kernelILi(\d+)ELi(\d+)ELi(\d+)E", name).groups())
        limit = 64 if (mt == 4 and nbuf == 1 and waves == 16) else 128 if waves == 16 else 256
        assert vgprs <= limit, f"{name}: {vgprs} VGPRs"

