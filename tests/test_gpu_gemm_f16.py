"""The q/k/v projections' GEMMs on expanded weights (cm_linear_f16_fwd / cm_linear_f16_bwd,
csrc/gemm_f16.hip) and the adapters' input gradients in one launch (cm_lora_fused_bwd2_multi) on
the GPU: the GEMMs against fp64 products of the same fp16 operands at the edges of their tiles and of
the rounds that choose a tile, the adapters' launch bit for bit against one call per adapter."""

import ctypes

import pytest
import torch

# rows around the 64-, 128- and 256-row tiles; outputs that end inside a tile, one to three of them;
# contractions from one stage; with the tiles each way takes: 128 x 64 while one round of 256
# workgroups holds the output, 256 x 256 (5400 rows, partial tiles both ways and along the contraction)
# where its rounds are a third of 128 x 128's, else 128 x 128
SHAPES = [
    (1, 64, (64,), "narrow", "narrow"),
    (63, 128, (64, 64), "narrow", "narrow"),
    (127, 192, (192, 64, 128), "narrow", "narrow"),
    (129, 64, (320, 64), "narrow", "narrow"),
    (257, 576, (896, 128, 128), "narrow", "narrow"),
    (1276, 1536, (1536, 256, 256), "small", "narrow"),
    (2000, 320, (1536, 256, 256), "small", "narrow"),
    (8200, 256, (1536, 256, 256), "small", "small"),
    (5400, 1600, (1536, 192, 192), "large", "large"),
    (5377, 1536, (1536, 256, 256), "large", "large"),
    (4097, 1536, (1536, 256, 256), "large", "small"),
]


def _form(m, n):
    """The tiles cm_linear_f16_* takes for m x n outputs (launch_best in csrc/gemm_f16.hip)."""
    def rounds(bm, bn):
        return -(-(-(-m // bm) * -(-n // bn)) // 256)

    if rounds(128, 64) <= 1:
        return "narrow"
    return "large" if rounds(256, 256) * 3 <= rounds(128, 128) else "small"


def _bound(a, b, ref):
    """Rounding of the result to fp16 (2^-11) and of the fp32 sums: the length of the contraction
    times 2^-24 of the sum of magnitudes, plus one subnormal."""
    mags = a.double().abs() @ b.double().abs()
    return ref.abs() * 2.0 ** -11 + mags * (a.shape[1] * 2.0 ** -24) + 2.0 ** -24


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,sizes,fwd,bwd", SHAPES, ids=lambda v: str(v))
def test_linear_rows(dev, m, k, sizes, fwd, bwd):
    from claudemaxing_amd.nf4_linear import linear_rows_bwd, linear_rows_fwd

    assert (_form(m, sum(sizes)), _form(m, k)) == (fwd, bwd)
    g = torch.Generator(device=dev).manual_seed(m)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=dev)

    x = normal(m, k + 8).half()[:, :k]  # a padded row stride
    w = (normal(sum(sizes), k) * 0.05).half()
    biases = [None if i == 1 else normal(s).half() for i, s in enumerate(sizes)]
    outs = linear_rows_fwd(x, w, list(sizes), biases)
    for got, wi, b in zip(outs, w.split(sizes), biases):
        ref = x.double() @ wi.double().t()
        ref = ref if b is None else ref + b.double()
        assert got.shape == ref.shape and got.dtype == torch.float16
        bound = _bound(x, wi.t(), ref) + (0 if b is None else 2.0 ** -24 * b.double().abs())
        assert bool(((got.double() - ref).abs() <= bound).all())

    grads = [normal(m, s + 16).half()[:, 8:s + 8] for s in sizes]
    dx = linear_rows_bwd(grads, w, list(sizes))
    merged = torch.cat(grads, 1)
    ref = merged.double() @ w.double()
    assert dx.shape == (m, k)
    assert bool(((dx.double() - ref).abs() <= _bound(merged, w, ref)).all())


# q, k, v weights as NF4, and token counts on both sides of where the fused GEMM's tiles and the number
# of slices of its input gradient change (8 to 1 slices: 4 at 1276 tokens of the first)
NF4_SHAPES = [(m, 1536, (1536, 256, 256)) for m in (1, 65, 257, 640, 1276, 2049, 2500, 3400, 5400)]
NF4_SHAPES += [(300, 2048, (2048, 256, 256)), (1276, 2048, (2048, 256, 256)),
               (900, 256, (1088, 64, 64)), (1276, 384, (640, 192, 64)), (700, 192, (192, 64, 64))]


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,sizes", NF4_SHAPES)
def test_linear_rows_has_the_fused_gemms_bits(dev, m, k, sizes):
    """Both ways, on expanded weights, the bits of the GEMM that expands them inside: the same fp16
    operands, the sums in the same order (the input gradient's in the same slices)."""
    from claudemaxing_amd.nf4 import quantize_nf4
    from claudemaxing_amd.nf4_linear import (expand_rows, linear_rows_bwd, linear_rows_fwd,
                                             nf4_linear_bwd, nf4_linear_fwd)

    g = torch.Generator(device=dev).manual_seed(m + k)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=dev)

    pairs = []
    for s in sizes:
        packed, state = quantize_nf4((normal(s, k) * 0.02).cpu(), 64, True)
        pairs.append((packed.to(dev), state.to(dev)))
    x, grads = normal(m, k).half(), [normal(m, s).half() for s in sizes]
    w = expand_rows(pairs)
    biases = [normal(s).half() for s in sizes]
    for a, b in zip(linear_rows_fwd(x, w, list(sizes), biases), nf4_linear_fwd(x, pairs, biases)):
        assert torch.equal(a, b)
    assert torch.equal(linear_rows_bwd(grads, w, list(sizes)), nf4_linear_bwd(grads, pairs))


@pytest.mark.gpu
def test_linear_f16_refuses(dev):
    from claudemaxing_amd import _lib

    lib = _lib.load()
    t = torch.zeros(64 * 64, dtype=torch.float16, device=dev)
    p = t.data_ptr()

    def fwd(m=64, k=64, n=64, ldx=64, x=p):
        return lib.cm_linear_f16_fwd(x, ldx, m, k, p, 1, (ctypes.c_int * 1)(n), None,
                                     (ctypes.c_void_p * 1)(p), (ctypes.c_int64 * 1)(n), None)

    assert fwd(m=0) == 0
    for bad in (dict(k=32), dict(n=32), dict(ldx=60), dict(x=p + 2), dict(x=None), dict(m=-1)):
        assert fwd(**bad) != 0


@pytest.mark.gpu
@pytest.mark.parametrize("t", [1, 3, 300, 1276, 5000])
@pytest.mark.parametrize("k", [64, 1536, 2048])
@pytest.mark.parametrize("with_dx", [True, False])
def test_bwd2_multi_matches_one_call_per_adapter(dev, t, k, with_dx):
    from claudemaxing_amd import _lib

    g = torch.Generator(device=dev).manual_seed(t + k)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=dev)

    dxb, x16 = normal(t, k).half(), normal(t, k).half()
    ga = [normal(t, 16).half() for _ in range(2)]
    a = [normal(16, k) for _ in range(2)]
    bits = [torch.randint(0, 256, (t * k // 8,), generator=g, device=dev, dtype=torch.uint8)
            for _ in range(2)]
    stream = _lib.stream(dev)

    def outputs():
        return (torch.zeros(t, k, device=dev) if with_dx else None,
                [torch.empty(t, k, dtype=torch.float16, device=dev) for _ in range(2)])

    dx1, xd1 = outputs()
    for i in range(2):
        _lib.call("cm_lora_fused_bwd2", dxb.data_ptr() if with_dx and i == 0 else None,
                  ga[i].data_ptr(), a[i].data_ptr(), x16.data_ptr(), bits[i].data_ptr(),
                  _lib.ptr(dx1), xd1[i].data_ptr(), t, k, 16, 1 / 0.95, stream)
    dx2, xd2 = outputs()
    P = ctypes.c_void_p * 2
    _lib.call("cm_lora_fused_bwd2_multi", dxb.data_ptr() if with_dx else None, x16.data_ptr(),
              _lib.ptr(dx2), t, k, 16, 1 / 0.95, 2, P(*[v.data_ptr() for v in ga]),
              P(*[v.data_ptr() for v in a]), P(*[v.data_ptr() for v in bits]),
              P(*[v.data_ptr() for v in xd2]), stream)
    if with_dx:
        assert torch.equal(dx1, dx2)
    for one, both in zip(xd1, xd2):
        assert torch.equal(one.view(torch.int16), both.view(torch.int16))
