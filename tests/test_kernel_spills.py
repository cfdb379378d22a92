"""Spilled registers of the built kernels (gfx950 code objects inside libmosegpu.so), without a GPU.

Budgets: the chemistry kernels that a mechanism runs, and the stage kernels of four and nine species.

Order: the compiler can place a spill of a live register at the head of a block that several branches join, ahead of the
instruction that gives the masked-off lanes back (s_or_b64 exec, exec, ...).  Those lanes then reload what the slot held
before; a RADAU5 kernel built that way stored stale step counts.  No kernel may hold such a block: a store to a spill
slot (scratch, or an accumulation register) between the head of a block and its exec restore, of a register that the
block did not write itself.

The stage kernels: four species do not spill, nine do in the inviscid LMRoe kernel alone."""
import os
import re
import subprocess

import pytest

import mosegpu
from test_kernel_resources import _tool, kernels  # noqa: F401  (the fixture of the kernels' metadata)


def _chem(kernels, name):  # noqa: F811
    return kernels[f"_ZN4mose{len(name)}{name}ILi9EEEvNS_7ChemDevENS_8ChemArgsE"]


# VGPRs that the occupancy needs (registers per lane: 512 over the waves per SIMD) and spilled ones, as built and measured
@pytest.mark.parametrize("name,vgprs,spills", [("k_chem2", 256, 2), ("k_radau2", 512, 4), ("k_chem", 128, 190),
                                               ("k_radau", 512, 4)])
def test_chemistry_kernels(kernels, name, vgprs, spills):  # noqa: F811
    k = _chem(kernels, name)
    assert int(k["vgpr_count"]) <= vgprs
    assert int(k["vgpr_spill_count"]) <= spills


def _stage_kernels(kernels, ns):  # noqa: F811
    """{(fast, viscous, solver, threads, shape): metadata} of the stage kernels of ns species."""
    out = {}
    for name, kv in kernels.items():
        m = re.match(rf"_ZN4mose\d+k_stage(_fast)?ILi{ns}ELi0ELb([01])ELi(\d+)ELi(\d+)ELi(\d+)EEE", name)
        if m:
            out[(m[1] is not None, m[2] == "1", int(m[3]), int(m[4]), int(m[5]))] = kv
    return out


def test_four_species_stage_kernels(kernels):  # noqa: F811
    ks = _stage_kernels(kernels, 4)
    assert len(ks) == 72      # parity 2 x 5 solvers x 4 shapes, performance 2 x 4 x 4
    for key, k in ks.items():
        assert int(k["vgpr_spill_count"]) == 0 and int(k["private_segment_fixed_size"]) == 0, key
        assert int(k["vgpr_count"]) <= 256, key
    for rs in (1, 2):         # two 512-thread workgroups per CU
        assert int(ks[(False, False, rs, 512, 1)]["vgpr_count"]) <= 128


def test_nine_species_stage_kernels(kernels):  # noqa: F811
    ks = {k: v for k, v in _stage_kernels(kernels, 9).items() if not k[0]}
    # viscous tiles hold 128 cells (256 threads), inviscid ones 128 or 256; no fixed shape fits the LDS
    assert {k[1:] for k in ks} == {(v, rs, bs, 0) for v in (False, True) for rs in (1, 2, 3, 4, 12)
                                   for bs in ((256,) if v else (256, 512))}
    for (_, visc, rs, bs, _), k in ks.items():
        spills = 28 if (rs, bs) == (12, 512) else 0
        assert int(k["vgpr_spill_count"]) <= spills, (visc, rs, bs)
        assert int(k["private_segment_fixed_size"]) <= 4 * spills, (visc, rs, bs)


# ---------------------------------------------------------------------------------------------------------------
# the order of spill stores and exec restores
# ---------------------------------------------------------------------------------------------------------------
LINE = re.compile(r"^\s+(\S+)(.*?)\s*//\s*([0-9A-F]+):.*?(?:<[^>+]*\+0x([0-9a-f]+)>)?\s*$")
NOT_VECTOR_RESULT = ("scratch_store", "global_store", "flat_store", "buffer_store", "ds_write", "s_", "v_cmp")


def _regs(op):
    m = re.match(r"^([va])\[(\d+):(\d+)\]$", op)
    if m:
        return {(m[1], q) for q in range(int(m[2]), int(m[3]) + 1)}
    m = re.match(r"^([va])(\d+)$", op)
    return {(m[1], int(m[2]))} if m else set()


def early_spills(listing):
    """The offsets of the exec restores of one kernel's listing (llvm-objdump -d) that a spill of a register from before
    the block precedes."""
    ins, targets = [], set()
    for line in listing.splitlines():
        m = LINE.match(line)
        if m:
            ins.append((int(m[3], 16), m[1], [o.strip() for o in m[2].split(",")]))
            if m[4]:
                targets.add(int(m[4], 16))
    start = ins[0][0]
    found, head, early, written = [], False, False, set()
    for at, op, args in ins:
        if at - start in targets:
            head, early, written = True, False, set()
        if head:
            if op == "s_or_b64" and args[:2] == ["exec", "exec"]:
                if early:
                    found.append(at - start)
                early = False
            elif op.startswith("v_accvgpr_write"):
                early = early or bool(_regs(args[1]) - written)
            elif op.startswith("scratch_store"):
                early = early or bool(set().union(*map(_regs, args)) - written)
            elif op.startswith(("s_endpgm", "s_and_saveexec", "s_barrier")) or (op == "s_mov_b64" and args[0] == "exec"):
                head = False
            if not op.startswith(NOT_VECTOR_RESULT):
                written |= _regs(args[0])
        if op.startswith(("s_cbranch", "s_branch")):
            head, early, written = True, False, set()
    return found


BLOCK = """
\ts_cbranch_execz 3                                          // 000000001000: BF880003 <k+0x10>
\tv_add_f64 v[24:25], v[24:25], -v[2:3]                      // 000000001004: 00000000 00000000
\ts_or_b64 exec, exec, s[4:5]                                // 000000001010: 87FE047E
{}
\ts_or_b64 exec, exec, s[14:15]                              // 000000001020: 87FE0E7E
"""


@pytest.mark.parametrize("line,hits", [
    ("\tscratch_store_dwordx2 off, v[24:25], off offset:76         // 000000001014: 00000000 00000000", 1),
    ("\tv_accvgpr_write_b32 a4, v24                                // 000000001014: 00000000 00000000", 1),
    ("\tv_accvgpr_write_b32 a4, 0                                  // 000000001014: 00000000 00000000", 0),
    ("\tds_read_b64 v[24:25], v3                                   // 000000001014: 00000000 00000000\n"
     "\tv_accvgpr_write_b32 a4, v24                                // 00000000101C: 00000000 00000000", 0)])
def test_the_check_sees_an_early_spill(line, hits):
    # the block joined at +0x10 gives its own lanes back first, then spills ahead of the outer restore
    assert len(early_spills(BLOCK.format(line))) == hits


def test_no_spill_ahead_of_an_exec_restore(kernels, tmp_path):  # noqa: F811
    tools = [_tool(t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-objdump")]
    if None in tools:
        pytest.skip("LLVM tools missing")
    objcopy, bundler, objdump = tools
    spilling = {n for n, k in kernels.items() if int(k["vgpr_spill_count"]) > 0 or int(k.get("agpr_count", 0)) > 0}
    assert any("k_radau2" in n for n in spilling)
    fat = str(tmp_path / "fat.bin")
    subprocess.run([objcopy, "--dump-section=.hip_fatbin=" + fat, str(mosegpu.LIB_PATH), str(tmp_path / "host.o")],
                   check=True, capture_output=True)
    data = open(fat, "rb").read()
    starts = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)] + [len(data)]
    seen = set()
    for n, (a, b) in enumerate(zip(starts[:-1], starts[1:])):
        part, co = str(tmp_path / f"fat{n}.bin"), str(tmp_path / f"gfx950_{n}.co")
        with open(part, "wb") as f:
            f.write(data[a:b])
        subprocess.run([bundler, "--unbundle", "--type=o", "--input=" + part,
                        "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--output=" + co], check=True, capture_output=True)
        os.remove(part)
        for name in sorted(spilling - seen):
            text = subprocess.run([objdump, "-d", "--disassemble-symbols=" + name, co], capture_output=True,
                                  text=True).stdout
            if "s_endpgm" not in text:
                continue
            seen.add(name)
            assert early_spills(text) == [], name
    assert seen == spilling
