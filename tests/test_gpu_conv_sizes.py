"""The convolution kernels at the sizes where their tiling changes: fewer and more cells
than one wave tile, a weight-gradient step of 32 cells and a block, grids that take one
and four tiles per wave, channel counts of each load width; against the FP64 oracle on
BF16-rounded operands.

Tolerance: products of BF16 values are exact in FP32, so a sum of N products in FP32 is
within N x 2^-24 of the exact one, relative to the sum of the products' magnitudes.
"""
import numpy
import pytest

from oracle import conv as oc

pytestmark = pytest.mark.gpu


def _pad16(v):
    return (v + 15) // 16 * 16


def _bits(x):
    return (numpy.ascontiguousarray(x, numpy.float32).view(numpy.uint32) >> 16).astype(numpy.uint16).view(numpy.int16)


@pytest.mark.parametrize('dim,shape,cin,cout', [
    (2, (3, 1, 1), 32, 3), (2, (7, 5, 1), 3, 32), (2, (33, 31, 1), 32, 32), (2, (300, 230, 1), 32, 3),
    (3, (2, 3, 2), 32, 32), (3, (9, 7, 5), 4, 32), (3, (11, 10, 13), 32, 4), (3, (5, 6, 7), 8, 16),
    (2, (300, 230, 1), 4, 4)])
def test_conv_layer_at_tile_edges(hip, dim, shape, cin, cout):
    import torch
    from transiflow_amd import _lib
    from transiflow_amd.vector import ptr, stream
    nx, ny, nz = shape
    n = nx * ny * nz
    rng = numpy.random.default_rng(n + cin)
    K = oc.taps(dim) * cin
    kpad, npad, kpt, npt = _pad16(K), _pad16(cout), _pad16(oc.taps(dim) * cout), _pad16(cin)
    x = oc.bf16(rng.standard_normal((n, cin)).astype(numpy.float32))
    W = numpy.zeros((kpad, npad), numpy.float32)
    W[:K, :cout] = oc.bf16((rng.standard_normal((K, cout)) * 0.3).astype(numpy.float32))
    b = rng.standard_normal(cout).astype(numpy.float32)
    g = oc.bf16(rng.standard_normal((n, cout)).astype(numpy.float32))
    d = {k: torch.from_numpy(v).cuda() for k, v in dict(x=_bits(x), W=W, b=b, g16=_bits(g), g=g).items()}
    Wf = torch.zeros(kpad * npad, dtype=torch.int16, device='cuda')
    Wt = torch.zeros(kpt * npt, dtype=torch.int16, device='cuda')
    out = torch.full((n, cout), float('nan'), dtype=torch.float32, device='cuda')
    _lib.call('tf_conv_pack', dim, cin, cout, kpad, npad, kpt, npt, ptr(d['W']), ptr(Wf), ptr(Wt), stream())
    _lib.call('tf_conv_fwd', nx, ny, nz, dim, cin, cout, kpad, npad, ptr(d['x']), ptr(Wf), ptr(d['b']), 0, ptr(out),
              None, stream())
    work = torch.full((_lib.load().tf_conv_wgrad_work_size(n, kpad, npad),), float('nan'), dtype=torch.float32,
                      device='cuda')
    dW = torch.full((kpad, npad), float('nan'), dtype=torch.float32, device='cuda')
    db = torch.full((cout,), float('nan'), dtype=torch.float32, device='cuda')
    _lib.call('tf_conv_wgrad', nx, ny, nz, dim, cin, cout, kpad, npad, ptr(d['x']), ptr(d['g16']), ptr(d['g']),
              ptr(work), ptr(dW), ptr(db), stream())
    P, G, Wd = oc.patches(x.astype(float), shape, dim), g.astype(float), W[:K, :cout].astype(float)
    eps = 2.0 ** -24

    def close(got, ref, size, terms):
        err = numpy.abs(got.cpu().numpy() - ref)
        assert numpy.all(err <= (terms + 2) * eps * size + 1e-30), (err / (eps * size + 1e-30)).max()

    close(out, P @ Wd + b, numpy.abs(P) @ numpy.abs(Wd) + numpy.abs(b), kpad + 1)
    close(dW[:K, :cout], P.T @ G, numpy.abs(P).T @ numpy.abs(G), n)
    close(db, G.sum(axis=0), numpy.abs(G).sum(axis=0), n)
    assert not dW.cpu().numpy()[K:].any() and not dW.cpu().numpy()[:, cout:].any()


@pytest.mark.parametrize('dim,shape,cin,cout', [(2, (7, 5, 1), 3, 32), (3, (9, 7, 5), 4, 32), (3, (9, 7, 5), 32, 4)])
def test_weight_gradient_without_the_bias_gradient(hip, dim, shape, cin, cout):
    """db may be null, and g32 with it: the same dW bit for bit at each load width."""
    import torch
    from transiflow_amd import _lib
    from transiflow_amd.vector import ptr, stream
    nx, ny, nz = shape
    n = nx * ny * nz
    rng = numpy.random.default_rng(n + cin)
    kpad, npad = _pad16(oc.taps(dim) * cin), _pad16(cout)
    x, g = (oc.bf16(rng.standard_normal((n, c)).astype(numpy.float32)) for c in (cin, cout))
    d = {k: torch.from_numpy(v).cuda() for k, v in dict(x=_bits(x), g16=_bits(g), g=g).items()}
    out = []
    for with_bias in (True, False):
        work = torch.full((_lib.load().tf_conv_wgrad_work_size(n, kpad, npad),), float('nan'), dtype=torch.float32,
                          device='cuda')
        dW = torch.full((kpad, npad), float('nan'), dtype=torch.float32, device='cuda')
        db = torch.full((cout,), float('nan'), dtype=torch.float32, device='cuda')
        _lib.call('tf_conv_wgrad', nx, ny, nz, dim, cin, cout, kpad, npad, ptr(d['x']), ptr(d['g16']),
                  ptr(d['g']) if with_bias else None, ptr(work), ptr(dW), ptr(db) if with_bias else None, stream())
        out.append(dW.cpu().numpy())
        assert torch.isfinite(db).all().item() == with_bias
    assert numpy.isfinite(out[0]).all() and numpy.array_equal(out[0], out[1])
