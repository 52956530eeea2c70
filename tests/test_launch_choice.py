"""Which kernel the launchers take for a shape, read from the launches themselves (recorder.py): the rules over sizes that
no other test would allocate."""
import pytest

from recorder import ptr, recorder

Q8_0 = 8


def rows_form(launches):
    """(waves, blocks an item) of the one launch, where it is the kernel that reads rows in long runs."""
    (one,) = launches
    assert one.kernel == "gemv_rows_kernel", one
    return int(one.params[2]), int(one.params[3])


@pytest.mark.parametrize("n_out", [98304, 128256, 152064, 256000])
@pytest.mark.parametrize("blocks, item", [(13, 1), (14, 2), (16, 2), (17, 2), (18, 0), (19, 2), (20, 2), (32, 2), (72, 2), (73, 1), (80, 1), (94, 1)])
def test_q8_0_matrices_of_many_turns(blocks, item, n_out):
    """Two-block items where their buffers fit LDS, one-block items where they do not: never out of the kernel while those fit
    it.  Of 18 blocks two-block items where the turns are whole (98304 rows on 256 CUs) or many (256000)."""
    want = item or (2 if n_out in (98304, 256000) else 1)
    assert rows_form(recorder().calls("orin_gemv", Q8_0, ptr(1), ptr(2), ptr(3), blocks * 256, n_out)) == (4, want)
