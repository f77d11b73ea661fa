"""CPU test of the kernels' wait counts: at every meeting of wavefronts in the compiled code, a
wavefront's own copies from memory into LDS have landed on every path. The counts are written by
hand (the compiler does not know of the copies' readers), so loads it leaves out make them too large."""
import pytest

import isa

pytestmark = pytest.mark.skipif(not (isa.OBJDUMP.exists() and isa.LIB.exists()), reason="needs llvm-objdump and the built library")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    return isa.kernels(tmp_path_factory.mktemp("isa"))


@pytest.mark.parametrize("family", ["hq_prefill_kernel", "hq_rows_kernel", "hq_decode_xr_kernel", "hq_w8a8_kernel"])
def test_copies_into_lds_land_before_they_are_published(kernels, family):
    found = {n: c for n, c in kernels.items() if family in n}
    assert any(op.startswith("buffer_load") and " lds" in args for c in found.values() for _, op, args, _ in c)
    late = {n: [hex(a) for a in isa.unlanded_copies(c)] for n, c in found.items()}
    assert not {n: a for n, a in late.items() if a}


def test_the_check_sees_a_count_that_is_too_large():
    # Two copies, three loads behind them, and a wait that leaves four operations in flight.
    code = [(0, "buffer_load_dwordx4", "v1, s[0:3], 0 offen lds", None)] * 2
    code += [(0, "buffer_load_dwordx2", "v[2:3], v1, s[0:3], 0 offen", None)] * 3
    code = [(4 * i, *c[1:]) for i, c in enumerate(code)]
    for n, late in ((3, []), (4, [24])):
        assert isa.unlanded_copies(code + [(20, "s_waitcnt", f"vmcnt({n})", None), (24, "s_barrier", "", None),
                                           (28, "s_endpgm", "", None)]) == late
