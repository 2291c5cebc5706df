"""GPU parity of the reference-domain fused linears (float32 / float16 / bfloat16, block <=
2^14, ``block % in_features == 0``) in grouped launches and at the tile shapes of their
matrix-core variant.

Grouped jobs run the code of their single calls, so they are compared bit for bit; the
single calls at the new tile shapes against ``x @ W^T`` in float64 with W from the C oracle
(float32 1e-5, float16 2e-3, bfloat16 1e-2 relative L2, as the domain's other tests).
"""
from __future__ import annotations

import pytest
import torch

from conftest import gpu_available
from latent_weight_lab_amd import ops
from oracle import c_oracle
from oracle import oracle as O

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

DTYPES = [torch.float32, torch.float16, torch.bfloat16]
TOL = {torch.float32: 1e-5, torch.float16: 2e-3, torch.bfloat16: 1e-2}


def randn(shape, seed, dtype):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def check_grouped(specs):
    got = ops.linear_forward_grouped(specs)
    for spec, y in zip(specs, got):
        kw = spec[6] if len(spec) > 6 else {}
        assert torch.equal(y, ops.linear_forward(*spec[:6], **kw)), (spec[0].shape, spec[2:6])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tokens", [1, 3, 4, 5, 15])
def test_grouped_shapes(dtype, tokens):
    """Blocks of 2^0 .. 2^14 in one call, partial last blocks, rows of one block and of many;
    a quad whose x needs the wide staging (single calls), and more workgroups than CUs."""
    shapes = [(1, 7, 1), (2, 300, 3), (32, 48, 32), (64, 200, 4096), (256, 1000, 2000), (1024, 40, 16384),
              (1024, 41, 9000), (1024, 4099, 16384), (2048, 24, 16384), (4096, 9, 8000), (8192, 5, 8192)]
    specs = []
    for i, (inf, outf, n) in enumerate(shapes):
        extra = {}
        if i % 3 == 1:
            extra = {"bias": randn(outf, 50 + i, dtype)}
        elif i % 3 == 2:
            extra = {"bias": randn(outf, 50 + i, dtype), "base": randn((tokens, outf), 70 + i, dtype)}
        specs.append((randn((tokens, inf), i, dtype), randn(n, 20 + i, dtype), outf, 1 + i % 3, 9 + i, 0.5, extra))
    check_grouped(specs)


def test_grouped_more_jobs_than_one_table():
    specs = [(randn((1 + i % 3, 64), i, torch.float32), randn(900 + i, 100 + i, torch.float32), 65 + i, 2, i, 1.0)
             for i in range(50)]
    check_grouped(specs)


def test_grouped_with_row_sums_and_matrix_core_jobs():
    """A row-sum term runs as a single call; bfloat16 blocks of 2^15 keep their own launch."""
    dtype = torch.bfloat16
    x, xs = randn((3, 768), 1, dtype), randn((3, 256), 2, dtype)
    coef = torch.tensor(0.25, device="cuda")
    specs = [(x, randn(32768, 3, dtype), 100, 3, 4, 1.0),
             (xs, randn(8000, 5, dtype), 77, 2, 6, 1.0, {"row_sum_coef": coef}),
             (xs, randn(8000, 7, dtype), 77, 2, 8, 1.0),
             (randn((40, 256), 9, dtype), randn(8000, 10, dtype), 64, 2, 11, 1.0)]  # matrix-core variant
    check_grouped(specs)


# one 16-row tile per workgroup (float32: two workgroups per CU from 1024 tokens, a last split
# shorter than the others), four row tiles (16-bit: two token tiles per item), a tile of many small
# blocks, and a column count whose tiles do not divide the CUs
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tokens,in_f,out_f,n,layers", [(1030, 1024, 72, 16384, 2), (1100, 1024, 1000, 9000, 3),
                                                        (300, 256, 520, 16000, 1), (70, 32, 1100, 500, 3)])
def test_matrix_core_tiles(dtype, tokens, in_f, out_f, n, layers):
    x, lat = randn((tokens, in_f), tokens, dtype), randn(n, n, dtype)
    got = ops.linear_forward(x, lat, out_f, layers, 17, 0.5)
    w = c_oracle.forward(lat.double().cpu().numpy(), in_f * out_f, layers, 17, 0, in_f * out_f)
    want = 0.5 * (x.double().cpu().numpy() @ w.reshape(out_f, in_f).T)
    assert O.rel_l2(got.double().cpu().numpy(), want) < TOL[dtype]
