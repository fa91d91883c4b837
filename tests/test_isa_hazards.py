"""The product kernels wait for their inline-assembly loads by hand; this compiles them to
assembly with the library's own flags and checks, over every path of every instantiation,
that no instruction touches a register whose load can still be outstanding."""
import functools
import os
import re
import shutil
import subprocess
import tempfile

import pytest

import isa_check
from rustingbrain_amd import build as rb_build

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "rustingbrain_amd", "csrc")
needs_hipcc = pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="needs hipcc")


@functools.lru_cache(maxsize=None)
def assembly(source: str) -> str:
    with tempfile.TemporaryDirectory() as tmp:
        out = os.path.join(tmp, "kernels.s")
        cmd = [rb_build.HIPCC] + [f for f in rb_build.FLAGS if f != "-fPIC"] + ["-S", "--cuda-device-only", "-o", out,
                                                                              os.path.join(CSRC, source)]
        subprocess.run(cmd, check=True, capture_output=True)
        return open(out).read()


def test_checker_flags_a_use_before_the_wait():
    asm = "\n".join(["_Zk:", "\tglobal_load_dwordx4 v[4:7], v1, s[0:1]", "\tglobal_load_dwordx4 v[8:11], v1, s[2:3]",
                     "\ts_waitcnt vmcnt(1)", "\tv_add_u32_e32 v0, v4, v5", "\tv_mov_b32_e32 v2, v9",
                     "\ts_waitcnt vmcnt(0)", "\tv_mov_b32_e32 v3, v9", "\ts_endpgm", ".Lfunc_end0:"])
    res = isa_check.check_asm(asm)["_Zk"]
    assert len(res) == 1 and "v_mov_b32_e32 v2, v9" in res[0]


def test_checker_follows_loops():
    asm = "\n".join(["_Zk:", ".LBB0_1:", "\tv_mov_b32_e32 v2, v9", "\tglobal_load_dwordx4 v[8:11], v1, s[2:3]",
                     "\ts_cbranch_scc1 .LBB0_1", "\ts_waitcnt vmcnt(0)", "\ts_endpgm", ".Lfunc_end0:"])
    res = isa_check.check_asm(asm)["_Zk"]
    assert any("v_mov_b32_e32 v2, v9" in h for h in res)


@needs_hipcc
def test_streaming_kernel_has_no_use_of_outstanding_loads():
    res = isa_check.check_asm(assembly("grouped_stream.hip"), "grouped_stream_kernel")
    assert len(res) >= 4, "expected every instantiation of the kernel in the assembly"
    bad = {k: v[:5] for k, v in res.items() if v}
    assert not bad, bad


def f32_kernels():
    """The instantiations over f32 rows with loads of their own: the last template argument says that rows and weights travel by
    them (the others leave every load and its wait to the compiler)."""
    return {n: k for n, k in isa_check.split_kernels(assembly("grouped_f32.hip")).items()
            if n.startswith("_ZN") and "grouped_f32_kernel" in n and "Lb1EEEv" in n}


@needs_hipcc
def test_f32_kernels_have_no_use_of_outstanding_loads():
    kernels = f32_kernels()
    assert len(kernels) == 26, "three weight types, gate/up and plain, four tiles (f32 weights: five)"
    bad = {n: h[:5] for n, h in ((n, isa_check.check_kernel(k)) for n, k in kernels.items()) if h}
    assert not bad, bad


@needs_hipcc
def test_a_wait_that_lets_two_more_loads_be_outstanding_is_found():
    """The check sees the f32 kernels' row loads: of the waits that leave some outstanding (the prologue's and the loop's), at
    least two of each kernel are flagged when they let two more be (the others stand for loads straight into the LDS only)."""
    for name, lines in f32_kernels().items():
        found = 0
        for i, line in enumerate(lines):
            m = re.search(r"vmcnt\(([1-9]\d*)\) lgkmcnt\(0\)", line)
            if m:
                looser = line.replace(m.group(0), f"vmcnt({int(m.group(1)) + 2}) lgkmcnt(0)")
                found += bool(isa_check.check_kernel(lines[:i] + [looser] + lines[i + 1:]))
        assert found >= 2, name


@needs_hipcc
@pytest.mark.parametrize("source,kernel", [("grouped_stream.hip", "grouped_stream_kernel"), ("grouped_f32.hip", "grouped_f32_kernel")])
def test_a_dense_tile_starts_when_every_wave_has_the_routed_counts(source, kernel):
    """A gate/up launch that works out its own tiles sums the router's histograms through the LDS that its main loop fills by
    LDS-DMA.  One barrier stands in front of the sums; a workgroup whose tile is a dense one fills the LDS right after, and
    a fast wave of it would overwrite the sums of a slow one without a second."""
    kernels = {n: k for n, k in isa_check.split_kernels(assembly(source)).items() if kernel in n}
    found = {n: isa_check.barriers_before_dma(k) for n, k in kernels.items()}
    found = {n: v for n, v in found.items() if v is not None}
    assert len(found) >= 4, "expected the gate/up instantiations among the kernels"
    assert all(v >= 2 for v in found.values()), found


@needs_hipcc
def test_registers_hold_as_many_routing_workgroups_as_the_plan_counts_on():
    """Two workgroups of eight waves on a compute unit where bf16 rows are routed on the matrix cores without a norm, four waves on
    each of its SIMDs with 512 registers; one over a quantized router."""
    asm = assembly("route_exact.hip")
    registers = {n: (int(r), int(lds)) for n, lds, r in re.findall(
        r"\.amdhsa_kernel (\S+)\n.*?\.amdhsa_private_segment_fixed_size (\d+)\n.*?\.amdhsa_next_free_vgpr (\d+)\n", asm, re.S)}
    assert len(registers) == 12
    for name, (vgprs, scratch) in registers.items():
        assert scratch == 0, name
        assert vgprs <= (128 if "ILi32ELi8ELb0E" in name else 256), name


@needs_hipcc
def test_wide_products_that_read_the_tables_keep_their_scalars_in_registers():
    """The code that works a launch's tiles out takes more scalar registers than there are, and a workgroup's first loads wait for
    every move of one into a vector register and back: only the launches that need that code may carry it."""
    found = dict(re.findall(r"\.name:\s+(_ZN\S*?21grouped_stream_kernel\S+)\n.*?\.sgpr_spill_count:\s+(\d+)\n", assembly("grouped_stream.hip"), re.S))
    wide = {n: re.match(r".*grouped_stream_kernelILb(\d)ELb(\d)ELi(\d)E(.*?)EvPK", n).groups() for n in found}
    for gate_up in "01":
        for int8 in "01":
            for blocks in "45":
                spills = {n: int(found[n]) for n, f in wide.items() if f[:3] == (gate_up, int8, blocks) and not f[3].startswith("Lb1E")}
                assert spills and not any(spills.values()), spills


@needs_hipcc
def test_static_scratch_array_is_a_symbol_the_runtime_can_look_up():
    # rbmoe_forward_static's scratch is a static device array whose address the host asks the runtime for by name
    # (hipGetSymbolAddress).  The runtime searches the code object's global symbols, and a missing one ends the
    # process rather than returning an error - so the array must come out of the device compilation as a global
    # object of the declared size, not as a local one.
    lines = [ln.strip() for ln in assembly("rbmoe_api.hip").splitlines() if "rbmoe_static_scratch" in ln]
    name = next(ln.split()[1].split(",")[0] for ln in lines if ln.startswith(".type"))
    assert f".globl {name}" in [" ".join(ln.split()) for ln in lines], lines
    assert not any(ln.startswith(".local") for ln in lines), lines
    assert any(ln.startswith(".size") and ln.endswith(str(8 << 20)) for ln in lines), lines
