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
