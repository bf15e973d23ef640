"""CPU: the kernels of the solve leave one partial sum per workgroup in arrays of 16,384;
on no mesh that set_topology accepts may a grid be larger (the sums of the workgroups
beyond would land in the next array while other workgroups read it)."""
import ctypes as C

import pytest

import eolc

MOST = 16384   # stride of one array of partial sums
LAST = 16384 * 1024   # the largest mesh


def rule(name, *args):
    sig = "".join("b" if isinstance(a, bool) else "i" for a in args)
    f = C.CDLL(eolc.LIB_PATH)[f"_ZN4eolc{len(name)}{name}E" + sig]
    f.argtypes = [C.c_bool if isinstance(a, bool) else C.c_int for a in args]
    return f(*args)


UP, MID, DOWN = [256, 512, 1024], [512, 1024, 256], [1024, 512, 256]


@pytest.mark.parametrize("n,rows", [(1, UP), (294912, UP), (294913, MID), (393216, MID), (393217, DOWN),
                                    (524288, DOWN), (524289, MID), (1310720, MID), (1310721, DOWN),
                                    (4194304, DOWN), (4194305, DOWN[:2]), (8388608, DOWN[:2]),
                                    (8388609, DOWN[:1]), (LAST, DOWN[:1])])
def test_patches_fit_the_partial_sums(n, rows):
    """The row counts tried on both sides of their lines, and the patches that they give;
    a mesh in arbitrary vertex order starts with 512 rows instead of 1,024 while those fit."""
    assert [rule("patch_rows", n, True, k) for k in range(4)] == rows + [0] * (4 - len(rows))
    assert all(rule("patch_grid", n, r) <= MOST for r in rows)
    spread = [rule("patch_rows", n, False, k) for k in range(4)]
    assert spread[0] == (512 if rows[:2] == [1024, 512] else rows[0]) and set(spread) == set(rows) | {0}


def test_every_grid_fits_the_partial_sums():
    sizes = {LAST + 1, LAST + 1024}
    for edge in (64, 256, 90000, 288 * 1024, 393216, 524288, 1310720, 8388608, LAST):
        sizes |= {max(1, edge + d) for d in (-1024, -64, -1, 0, 1, 64, 1024)}
    sizes |= set(range(1, LAST, 65537))
    for n in sorted(sizes):
        most = rule("most_partials", n)
        grids = [rule("pcg_grid", n), rule("vec_grid", n)]
        grids += [rule("patch_grid", n, r) for r in (rule("patch_rows", n, True, k) for k in range(4)) if r]
        assert most >= max(grids)
        assert (most <= MOST) == (n <= LAST), n   # set_topology refuses by this
