"""Which states of a batch graph share launches, and which branch runs them."""
import numpy as np
import pytest

import simulador_quantico_amd as hq
from simulador_quantico_amd import _native as N

H = np.array([[1, 1], [1, -1]]) / np.sqrt(2)


def _plan(n, kernel, phase=0.5, dtype=np.complex64):
    gates = [(b, 0, 0, H) for b in range(n)] + [(0, 1 << (n - 1), 1 << (n - 1), np.diag([1, np.exp(1j * phase)]))]
    t = N.default_tuning(block_size=32, repeat_count=4, gpu_region_bits=8, gpu_coalesced_bits=3, kernel=kernel)
    p = hq.Plan(n, hq.make_ops(*zip(*gates)), t, 1, dtype)
    assert p.kernel == kernel
    return p


def test_states_on_one_lds_plan_have_branches_of_their_own():
    lds = _plan(9, N.HGM_KERNEL_LDS)
    group, branch = hq.Batch.layout([lds] * 5)
    assert sorted(group) == [0, 1, 2, 3, 4]
    assert sorted(branch) == [0, 1, 2, 3, 4]


def test_states_on_equal_register_plans_share_their_launches():
    a, b, other = _plan(9, N.HGM_KERNEL_REG), _plan(9, N.HGM_KERNEL_REG), _plan(9, N.HGM_KERNEL_REG, 0.25)
    lds = _plan(9, N.HGM_KERNEL_LDS)
    group, branch = hq.Batch.layout([a, b, a, other, lds, other, lds])
    assert group[0] == group[1] == group[2] and group[3] == group[5]
    assert len(set(group)) == 4 and group[4] != group[6]
    assert len(set(branch)) == 4


@pytest.mark.parametrize("kernel", [N.HGM_KERNEL_REG, N.HGM_KERNEL_LDS])
def test_beyond_64_groups_branches_are_shared(kernel):
    plans = [_plan(9, kernel, 0.01 * (k + 1)) for k in range(70)]
    group, branch = hq.Batch.layout(plans)
    assert sorted(group) == list(range(70))
    assert sorted(set(branch)) == list(range(64))
    assert max(branch.count(k) for k in set(branch)) == 2


def test_layout_refuses_what_a_batch_refuses():
    with pytest.raises(N.HGMError):
        hq.Batch.layout([])
