"""The many-vector core's wait counts (kq_gx_stages.h, host build): before every
stage, in rows of one column and more, the fragments that the stage reads have
arrived in every wave.  A wave's loads complete in order, so a wait for at most
n outstanding ones covers a load with at least n issued after it.  The code
loads of the last column have no use and may be dropped by the compiler, so
they are left out; 1 / S loads, which only some waves issue, are too.
No GPU needed."""
import ctypes
import os

import pytest

import aspida_amd as aa

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emul", "libkq_emul.so")


@pytest.fixture(scope="module")
def emul():
    if not os.path.exists(LIB):
        pytest.skip("tests/emul/libkq_emul.so not built (run build())")
    return ctypes.CDLL(LIB)


@pytest.mark.parametrize("nv", [1, 2])
@pytest.mark.parametrize("kind", aa.KINDS, ids=lambda k: aa.KIND_NAMES[k])
def test_stage_waits_cover_their_fragments(emul, kind, nv):
    ring = emul.kq_emul_gx_ring(kind, nv)
    for columns in range(1, 12):
        done, issued = set(range(ring - 1)), []  # the prologue waits for all of its loads
        for g in range(4 * columns):
            c, j = divmod(g, 4)
            last = c == columns - 1
            wait = emul.kq_emul_gx_stage_wait(kind, nv, j, last)
            assert 0 <= wait < 64
            done.update(issued[:max(0, len(issued) - wait)])
            late = [i for i, s in enumerate(issued) if s == g and i >= len(issued) - wait]
            assert g in done and not late, (columns, g, wait)
            if not last:
                issued += [None] * emul.kq_emul_gx_body_loads(kind, j)
            issued += [g + ring - 1] * (2 * nv)


@pytest.mark.parametrize("kind", aa.KINDS, ids=lambda k: aa.KIND_NAMES[k])
def test_code_loads_of_a_column(emul, kind):
    """16-byte code chunks per row and column that the four stages load (Q5_K's
    and Q3_K's high bits come with the head)."""
    chunks = {aa.Q4_K: 8, aa.Q5_K: 8, aa.Q6_K: 12, aa.Q3_K: 4, aa.Q2_K: 4, aa.Q8_0: 16}[kind]
    # Two lanes (the halves of a wave) share a row: half of the chunks each.
    assert 2 * sum(emul.kq_emul_gx_body_loads(kind, j) for j in range(4)) == chunks
