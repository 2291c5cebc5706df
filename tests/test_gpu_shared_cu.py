"""GPU parity of the matrix-core launches of more generated blocks than CUs: those whose
workgroups share a CU (one exchange buffer, at most 128 VGPRs: the generator's forward, the
grouped weight calls, the grouped fused linear) and the backward whose workgroups sum several
blocks, against the C oracle and against smaller launches or single calls.

A block runs the same arithmetic in both forms, so where a smaller launch (one workgroup per
CU) covers the same blocks the results are compared bit for bit.
"""
from __future__ import annotations

import pytest
import torch

from conftest import gpu_available
from latent_weight_lab_amd import ops
from oracle import c_oracle
from oracle import oracle as O

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

BF16 = torch.bfloat16
B = 1 << 15
BLOCKS = 257  # one more than the CUs
SEED = 31


def latent_for(n, seed):
    return torch.randn(n, generator=torch.Generator().manual_seed(seed)).to(BF16)


# (latent size, start, elements past the last whole block dropped): whole blocks on the 16-byte
# grid, and a padded latent with both ends inside a block, off that grid by 1..7 elements
SHAPES = [(32768, 0, 0), (16385, 3, 5), (20001, 8 * 11 + 6, 4097)]


@pytest.mark.parametrize("layers", [1, 2, 3])
@pytest.mark.parametrize("n,start,cut", SHAPES)
def test_forward(n, start, cut, layers):
    lat = latent_for(n, layers)
    size = BLOCKS * B
    stop = size - cut
    got = ops.forward(lat.cuda(), size, layers, SEED, start, stop)
    # the same blocks in two launches of at most one workgroup per CU
    mid = 200 * B
    assert torch.equal(got[: mid - start], ops.forward(lat.cuda(), size, layers, SEED, start, mid))
    assert torch.equal(got[mid - start:], ops.forward(lat.cuda(), size, layers, SEED, mid, stop))
    a, b = size - 2 * B - 7, stop
    want = c_oracle.forward(lat.double().numpy(), size, layers, SEED, a, b)
    assert O.rel_l2(got[a - start:].double().cpu().numpy(), want) < 1e-2


@pytest.mark.parametrize("layers", [1, 2, 3])
@pytest.mark.parametrize("blocks,n,start,cut", [(BLOCKS, *s) for s in SHAPES] + [(515, 20001, 0, 9)])
def test_backward(blocks, n, start, cut, layers):
    """Groups of 2 (the last one block) and 3 (the last two): whole blocks, blocks off the
    16-byte grid, and whole blocks read ahead with a partial one at the end."""
    size = blocks * B
    stop = size - cut
    g = torch.randn(stop - start, generator=torch.Generator().manual_seed(layers + 10)).to(BF16)
    got = ops.backward(g.cuda(), n, BF16, size, layers, SEED, start, stop)
    want = c_oracle.backward(g.double().numpy(), n, size, layers, SEED, start, stop)
    assert O.rel_l2(got.double().cpu().numpy(), want) < 1e-2
    assert torch.equal(got, ops.backward(g.cuda(), n, BF16, size, layers, SEED, start, stop))


@pytest.mark.parametrize("layers", [1, 2, 3])
def test_grouped_weights(layers):
    """More blocks than CUs over two jobs, the last block of each partial, one scaled."""
    sizes = [150 * B + 13, 120 * B - 8]
    lats = [latent_for(n, n).cuda() for n in (32768, 30001)]
    specs = [(lat, s, layers, 5 + i, 0.5 + 0.5 * i, BF16) for i, (lat, s) in enumerate(zip(lats, sizes))]
    got = ops.materialize_weights(specs)
    for spec, w in zip(specs, got):
        assert torch.equal(w, ops.materialize_weights([spec])[0])
    grads = [torch.randn(s, generator=torch.Generator().manual_seed(s)).to(BF16).cuda() for s in sizes]
    flush = [(lat, g, s, layers, 5 + i, 1.0, None) for i, (lat, g, s) in enumerate(zip(lats, grads, sizes))]
    for spec, r in zip(flush, ops.flush_weight_grads(flush)):
        assert torch.equal(r, ops.flush_weight_grads([spec])[0])


# widths by the table's layout: whole 16-row tiles or an exact row count, four row tiles, a width
# off 32 (one row division per chunk), no padding at all, and one whose table needs more than half
# the LDS (its launch stays at one workgroup per CU)
@pytest.mark.parametrize("in_f,out_f", [(768, 3072), (640, 4000), (1000, 3001), (3072, 900), (4096, 700), (5120, 513)])
@pytest.mark.parametrize("tokens,layers", [(1, 3), (17, 2), (130, 1), (255, 3)])
def test_grouped_linear(in_f, out_f, tokens, layers):
    nb = (in_f * out_f + B - 1) // B
    count = 256 // nb + 1
    x = torch.randn(tokens, in_f, generator=torch.Generator().manual_seed(in_f)).to(BF16).cuda()
    bias = torch.randn(out_f, generator=torch.Generator().manual_seed(out_f)).to(BF16).cuda()
    lats = [latent_for(20000 + 7 * i, i).cuda() for i in range(count)]
    specs = [(x, lat, out_f, layers, 40 + i, 0.5, {"bias": bias} if i % 2 else {}) for i, lat in enumerate(lats)]
    for spec, got in zip(specs, ops.linear_forward_grouped(specs)):
        assert torch.equal(got, ops.linear_forward(*spec[:6], **spec[6]))


@pytest.mark.parametrize("in_first", [768, 4096])
def test_grouped_linear_of_mixed_rows(in_first):
    """Jobs of short and long rows and of several batches in one launch, whichever comes first:
    the launch starts the blocks with the most work, each job's outputs are its own call's."""
    shapes = [(768, 3072, 130), (4096, 700, 5), (3072, 768, 130), (768, 768, 1), (4096, 600, 250)]
    shapes.sort(key=lambda s: s[0], reverse=in_first == 4096)
    specs = []
    for i, (in_f, out_f, tokens) in enumerate(shapes):
        x = torch.randn(tokens, in_f, generator=torch.Generator().manual_seed(i)).to(BF16).cuda()
        bias = torch.randn(out_f, generator=torch.Generator().manual_seed(out_f)).to(BF16).cuda()
        specs.append((x, latent_for(20000 + 7 * i, i).cuda(), out_f, 3, 40 + i, 0.5, {"bias": bias} if i % 2 else {}))
    assert sum((x.shape[1] * out_f + B - 1) // B for x, _, out_f, *_ in specs) > 256
    for spec, got in zip(specs, ops.linear_forward_grouped(specs)):
        assert torch.equal(got, ops.linear_forward(*spec[:6], **spec[6]))
