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
