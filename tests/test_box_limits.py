"""CPU test of the rule that keeps the kernels on box elements within their 32-bit offsets."""
import pytest

# the records of csrc/box.hpp: 2 dim + 1 doubles and 2 dim int32
RECORD = {dim: 8 * (2 * dim + 1) + 4 * 2 * dim for dim in (1, 2, 3)}
NS = {"advection": lambda dim: 1, "euler": lambda dim: dim + 2}


@pytest.mark.parametrize("N", [1, 2, 3, 4, 7])
@pytest.mark.parametrize("dim", [1, 2, 3])
@pytest.mark.parametrize("law", ["advection", "euler"])
def test_box_kernels_take_what_32_bit_offsets_reach(law, dim, N):
    import atum_hip._lib as L
    ns, node = NS[law](dim), (N + 1) ** dim
    fit = lambda K: L.lib.atm_box_elements_fit(dim, N, ns, K)
    # the offsets of the last element's record and of the last component of its last node
    reach = lambda K: max((K - 1) * RECORD[dim], 8 * (ns * node * K - 1))
    lo, hi = 1, 1 << 31
    assert fit(lo) == 1 and fit(hi) == 0
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (mid, hi) if fit(mid) else (lo, mid)
    assert reach(lo) < 1 << 32
    # and nothing much smaller is turned away: the next element is at an offset's end, or at 4 GB of state
    assert reach(lo + 2) >= (1 << 32) - 8 * ns * node


# the first element whose record's 32-bit offset would wrap
@pytest.mark.parametrize("dim,N,K", [(1, 1, 134217728), (1, 2, 134217728), (2, 1, 76695844), (3, 1, 53687091)])
def test_records_larger_than_states(dim, N, K):
    import atum_hip._lib as L
    assert 8 * (N + 1) ** dim * (K + 1) < 1 << 32  # the state alone would still fit
    assert K * RECORD[dim] <= 1 << 32 < (K + 1) * RECORD[dim]
    assert L.lib.atm_box_elements_fit(dim, N, 1, K) == 1
    assert L.lib.atm_box_elements_fit(dim, N, 1, K + 1) == 0


def test_bad_arguments():
    import atum_hip._lib as L
    for a in ((0, 1, 1, 1), (4, 1, 1, 1), (2, 0, 1, 1), (2, 8, 1, 1), (2, 1, 0, 1), (2, 1, 1, -1)):
        assert L.lib.atm_box_elements_fit(*a) < 0, a
