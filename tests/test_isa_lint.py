"""The check of hand-counted waits (glowq_amd/isa_lint.py), which the build runs over the assembly of the GEMM on the tiled weights."""
import pytest

from glowq_amd import build, isa_lint

LDS = "\tbuffer_load_dwordx4 v3, s[4:7], s9 offen sc1 lds\n"
REG = "\tbuffer_load_dwordx4 v[8:11], v2, s[12:15], s1 offen offset:1024\n"


def listing(*loads, count=8, head="gemm_tiled_kernel"):
    return (f"_Z17{head}ILi1E:                ; @k\n; %bb.0:\n" + "".join(loads) + f"\t;;#ASMSTART\n\t; loads to LDS are followed by {count} others\n"
            "\t;;#ASMEND\n\ts_waitcnt vmcnt(4)\n\ts_barrier\n\ts_endpgm\n.Lfunc_end0:\n")


@pytest.mark.parametrize("loads", [[LDS, LDS] + [REG] * 8, [REG, REG, LDS] + ["\tv_mov_b32_e32 v1, 0\n"] + [REG] * 8, [REG] * 8])
def test_the_order_of_the_source_passes(loads):
    assert isa_lint.counted_waits(listing(*loads), "gemm_tiled_kernel") == []


@pytest.mark.parametrize("loads", [[LDS] + [REG] * 4 + [LDS] + [REG] * 4,  # as the loads of the left factor once were, among those of r
                                   [REG] * 8 + [LDS, LDS],
                                   [LDS] + [REG] * 7,
                                   [LDS, REG, REG, REG, ".LBB0_1:\n"] + [REG] * 5])
def test_another_order_is_found(loads):
    (found,) = isa_lint.counted_waits(listing(*loads), "gemm_tiled_kernel")
    assert "8 loads are counted" in found
    assert isa_lint.counted_waits(listing(*loads, head="another_kernel"), "gemm_tiled_kernel") == []


def test_the_build_checks_the_gemm():
    assert build.COUNTED_WAITS["gemm.hip"] == "gemm_tiled_kernel"
