"""Spilled registers of the stage kernels of four and nine species, from the built code objects (no GPU)."""
import re

from test_kernel_resources import kernels  # noqa: F401  (the fixture of the kernels' metadata)


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
