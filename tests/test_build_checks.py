"""CPU tests of the build's checks of device listings: registers that only inline assembly
names must not be the compiler's, and a listing that breaks a rule stops the build."""
import pytest

from simplexprojects_amd import build

BLOCK = """
_Z6kernelv: ; @_Z6kernelv
; %bb.0:
\t;;#ASMSTART
\t; block from v{v}{a}
\t;;#ASMEND
\t.p2align 4
\tv_mov_b32_e32 v{use}, 0 ; comment v255
\t;;#ASMSTART
\tv_mov_b64 v[100:101], v[10:11]
\t;;#ASMEND
\tv_fma_f64 v[{lo}:{hi}], v[0:1], v[2:3], v[4:5]
\tv_accvgpr_write_b32 a{acc}, v1
\ts_endpgm
"""


def block(tmp_path, v="0x50", a="", use=79, lo=78, hi=79, acc=200):
    f = tmp_path / "kernel.s"
    f.write_text(BLOCK.format(v=v, a=a, use=use, lo=lo, hi=hi, acc=acc))
    return f


@pytest.mark.parametrize("over", [{}, {"v": "80"}, {"a": " a0x50", "acc": 79}, {"v": "60", "use": 1, "lo": 58, "hi": 59}])
def test_blocks_above_the_compilers_registers(tmp_path, over):
    assert build._check_blocks(block(tmp_path, **over)) == 1


@pytest.mark.parametrize("over", [{"use": 80}, {"use": 255}, {"lo": 79, "hi": 80}, {"v": "79"},
                                  {"a": " a0x50", "acc": 80}])
def test_compiler_in_the_blocks_registers(tmp_path, over):
    with pytest.raises(RuntimeError, match="registers of the block"):
        build._check_blocks(block(tmp_path, **over))


def test_kernel_that_does_not_name_its_block(tmp_path):
    f = tmp_path / "kernel.s"
    f.write_text(BLOCK.format(v=80, a="", use=1, lo=2, hi=3, acc=0).replace("; block", "; no block"))
    with pytest.raises(RuntimeError, match="does not say"):
        build._check_blocks(f)


WAITS = """
_Z6kernelv: ; @_Z6kernelv
\tv_cndmask_b32_e64 v17, v17, 1.0, s[8:9]
\t;;#ASMSTART
\t{wait}
\t;;#ASMEND
\t;;#ASMSTART
\t{use}
\t;;#ASMEND
\ts_endpgm
"""
MFMA = "v_mfma_f32_16x16x1_4b_f32 a[0:15], {}, {}, a[0:15] cbsz:2 abid:0"


@pytest.mark.parametrize("wait,use,good", [
    ("s_nop 4", MFMA.format("v17", "v24"), True), ("s_nop 1", MFMA.format("v24", "v17"), True),
    ("s_nop 0", MFMA.format("v17", "v24"), False), ("s_nop 0", MFMA.format("v16", "v24"), True),
    ("v_mov_b32 v9, 0", MFMA.format("v24", "v17"), False),
    (".set blpg_a, 3", MFMA.format("v17", "v24"), False),
    ("s_mov_b64 exec, -1\n\ts_branch L", "v_permlane32_swap_b32_e32 v16, v17", True),
    ("s_mov_b64 exec, -1", "v_permlane32_swap_b32_e32 v16, v17", False),
    ("v_accvgpr_write_b32 a17, v3", "v_permlane32_swap_b32_e32 v17, v18", False),
    ("s_nop 0", "v_add_f32_e32 v17, v17, v17", True)])
def test_waits_before_reads_of_a_written_register(tmp_path, wait, use, good):
    f = tmp_path / "kernel.s"
    f.write_text(WAITS.format(wait=wait, use=use))
    if good:
        assert build._check_operand_waits(f) == use.startswith("v_mfma")
    else:
        with pytest.raises(RuntimeError, match="wait states after"):
            build._check_operand_waits(f)
