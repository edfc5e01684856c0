"""CPU test of the check's launch plan: a tier that takes a bin by itself holds every LP of it."""
import ctypes as C

import simplexprojects_amd as sa

LIB = sa.load_library()
COVERS = getattr(LIB, "_ZN4blpg18verify_tier_coversEiiii")  # (tier, m, n, tableau element bytes)
CAP = getattr(LIB, "_ZN4blpg16verify_stage_capEiii")        # (tier, m, n)
COVERS.restype, CAP.restype = C.c_bool, C.c_int64


def stage_bytes(m, k, tsz):
    """m rows of k columns, padded to an odd count, in FP64 and in the tableau's precision."""
    return m * (k | 1) * (8 + tsz)


def test_a_covering_tier_holds_the_widest_blocks():
    """Widest: as many columns as basic structurals, and in FP32 one more when phase I ends
    with every structural and the auxiliary variable basic (at most a column per row)."""
    covered = 0
    for m in range(1, 241):
        for n in range(1, 241):
            for tsz, k in ((4, min(m, n + 1)), (8, min(m, n))):
                for tier in (0, 1):
                    if COVERS(tier, m, n, tsz):
                        covered += 1
                        assert stage_bytes(m, k, tsz) <= CAP(tier, m, n), (tier, m, n, tsz)
    assert covered > 10000


def test_x0s_column_does_not_choose_the_first_tier():
    """The first tier is for LPs that can use a dozen staged columns: by the structurals alone."""
    used = getattr(LIB, "_ZN4blpg16verify_tier_usedEiiii")
    used.restype = C.c_bool
    for tsz, dozen in ((4, 10), (8, 12)):
        for m in (13, 20, 40):
            assert [used(0, m, n, tsz) for n in (dozen - 1, dozen)] == [False, True], (m, tsz)
