"""The packed weight jobs equal the ctypes structure's fields (no GPU needed)."""
from __future__ import annotations

import pytest
import torch

from latent_weight_lab_amd import _native as N
from latent_weight_lab_amd import ops


@pytest.mark.parametrize("seed", [0, 7, -1, 2**63 - 1, -(2**63), 2**63 + 5, 2**64 - 1])
def test_packed_job_fields(seed):
    lat = torch.zeros(5898, dtype=torch.float16)
    arr = (N.WeightJob * 3)()
    ops._pack_job(arr, 1, lat, 768 * 768, 2, seed, 0.25, torch.bfloat16, weight=64, grad_weight=128, grad_latent=192,
                  accumulate=1)
    j = arr[1]
    want = N.WeightJob(lat.data_ptr(), 64, 128, 192, 5898, 768 * 768, 2, seed, 1, 2, 0.25, 1)
    for name, _ in N.WeightJob._fields_:
        assert getattr(j, name) == getattr(want, name), name
    assert bytes(arr[0]) == bytes(arr[2]) == bytes(N.WeightJob())


@pytest.mark.parametrize("ld", list(N.DTYPE_CODES))
@pytest.mark.parametrize("wd", list(N.DTYPE_CODES))
@pytest.mark.parametrize("n", [1, 2, 31, 16384, 16385, 32768, 32769, 1 << 20])
def test_rule_for_grouped_weights_is_the_librarys(n, ld, wd):
    """``weight_job_taken`` decides without the library; both answers, over block sizes, dtypes and
    the largest launches (aligned pointers, where it takes no part in them)."""
    lat, arr = torch.zeros(n, dtype=ld), (N.WeightJob * 1)()
    block = ops.next_power_of_two(n)
    for size in (1, 12345, ((1 << 31) - 1) * block, ((1 << 31) - 1) * block + 1):
        for fwd in (1, 0):
            ops._pack_job(arr, 0, lat, size, 2, 0, 1.0, wd, weight=256, grad_weight=256, grad_latent=1 << 20)
            taken = N.lib().lwl_bfht_check_weight_jobs(arr, 1, fwd) == N.LWL_OK
            if ld == torch.bfloat16 != wd and 16384 < n <= 32768:
                assert not taken  # asked of the library itself, with the pointers of the call
            else:
                assert ops.weight_job_taken(lat, size, wd) == taken, (size, fwd)
