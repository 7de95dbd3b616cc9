"""Plans of a batch of ansatz circuits whose register groups are too wide."""

import pytest

from qibojit_amd.batch import AnsatzBatch


@pytest.mark.parametrize("n,k", [(12, 6), (13, 7), (20, 20)])
def test_groups_of_more_than_five_bits_are_refused(n, k):
    with pytest.raises(ValueError):
        AnsatzBatch([(n, 1)], device="cpu", plan={n: ("pass", k)})


@pytest.mark.parametrize("n,k", [(12, 5), (14, 6), (20, 5), (22, 3)])
def test_groups_that_fit_are_planned(n, k):
    batch = AnsatzBatch([(n, 1)], device="cpu", plan={n: ("pass", k)})
    assert sorted(b for ps in batch.pass_groups[0].passes for b in ps.bits) == list(range(n))
