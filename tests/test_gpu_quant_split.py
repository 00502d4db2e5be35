"""The quantiser's workgroup-per-token layout at the edges of its dispatch:
255 and 256 tokens (eight and four waves on rows of one pass), one, three,
four and eight passes, partial passes, and the first row too long for it
(K = 16512: one wavefront per token); short rows of many tokens (one wavefront
per token, the row in registers).  Codes, scales and sums bit-exact against
the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from oracle import reference as ref
from webyiq_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K", [(255, 2048), (256, 2048), (257, 128), (256, 1920), (40, 2176), (33, 6144),
                                 (20, 8192), (18, 16384), (18, 16512)])
@pytest.mark.parametrize("GA,G,norm", [(None, 128, True), (None, 32, False), (32, 128, True)])
def test_quant_layout_edges(M, K, GA, G, norm):
    print(f"[case] quant M={M} K={K} GA={GA} G={G} norm={norm}", flush=True)
    rng = np.random.default_rng(M + K)
    x = ref.make_activations(rng, M, K)
    x[M // 2] = 0.0
    nw = rng.normal(1.0, 0.2, size=K).astype(np.float32) if norm else None
    xq, dx, xs = orc.quant_act(x, GA, G, norm_w=nw, eps=1e-6)
    a = ops.quant(torch.from_numpy(x).cuda(), norm=None if nw is None else torch.from_numpy(nw).cuda(), eps=1e-6,
                  GA=GA, G=G)
    assert np.array_equal(a.xq.cpu().numpy(), xq)
    assert np.array_equal(a.dx.cpu().numpy().view(np.uint32), dx.view(np.uint32))
    assert np.array_equal(a.xs.cpu().numpy(), xs)


# both sides of the line where short rows change to one wavefront per token,
# token counts that leave a workgroup of four tokens unfilled
@pytest.mark.parametrize("M,K", [(2047, 384), (2049, 128), (2050, 1536), (2051, 1664), (4095, 256), (4097, 1024),
                                 (4098, 1152), (8191, 128), (8193, 1024)])
@pytest.mark.parametrize("GA,G,norm", [(None, 128, True), (None, 32, False), (32, 128, True), (32, 32, False)])
def test_quant_short_rows(M, K, GA, G, norm):
    print(f"[case] quant short rows M={M} K={K} GA={GA} G={G} norm={norm}", flush=True)
    rng = np.random.default_rng(M + K)
    x = rng.normal(size=(M, K)).astype(np.float32)
    x[M // 2] = 0.0
    nw = rng.normal(1.0, 0.2, size=K).astype(np.float32) if norm else None
    xq, dx, xs = orc.quant_act(x, GA, G, norm_w=nw, eps=1e-6)
    a = ops.quant(torch.from_numpy(x).cuda(), norm=None if nw is None else torch.from_numpy(nw).cuda(), eps=1e-6,
                  GA=GA, G=G)
    assert np.array_equal(a.xq.cpu().numpy(), xq)
    assert np.array_equal(a.dx.cpu().numpy().view(np.uint32), dx.view(np.uint32))
    assert np.array_equal(a.xs.cpu().numpy(), xs)


def test_quant_beyond_one_grid():
    """More tokens than a grid of 512-thread workgroups holds (2^22): the call
    goes out as two launches."""
    M, K, cut = (1 << 22) + 37, 128, 1 << 22
    print(f"[case] quant in two launches M={M} K={K}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(8)
    x = torch.randn((M, K), generator=g, device="cuda")
    a = ops.quant(x, GA=32, G=32)
    for lo, hi in ((0, 64), (cut - 64, cut), (cut, M)):
        xq, dx, xs = orc.quant_act(x[lo:hi].cpu().numpy(), 32, 32)
        assert np.array_equal(a.xq[lo:hi].cpu().numpy(), xq)
        assert np.array_equal(a.dx[lo:hi].cpu().numpy().view(np.uint32), dx.view(np.uint32))
        assert np.array_equal(a.xs[lo:hi].cpu().numpy(), xs)
    for lo, hi in ((0, cut), (cut // 2 + 1, M)):  # the rest: like calls of one launch on its parts
        b = ops.quant(x[lo:hi], GA=32, G=32)
        assert torch.equal(b.xq, a.xq[lo:hi]) and torch.equal(b.dx, a.dx[lo:hi]) and torch.equal(b.xs, a.xs[lo:hi])
