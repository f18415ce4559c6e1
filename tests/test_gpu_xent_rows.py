"""cm_xent_rows on full logits at the edges of its chunks: rows that start anywhere in a 16-byte
chunk, lengths around one chunk, one round of lanes and the line between its two widths, and logits
of -inf, +inf, NaN and the type's lowest value, against float64."""

import pytest
import torch

from claudemaxing_amd import _lib
from tests.conftest import banner

pytestmark = pytest.mark.gpu


def run(z, t, grad, scale=1.0):
    """z: a 2-D view with any row stride, overwritten by the gradient."""
    n = z.shape[0]
    loss, ent = (torch.empty(n, device=z.device) for _ in range(2))
    corr = torch.empty(n, dtype=torch.int32, device=z.device)
    _lib.call("cm_xent_rows", z.data_ptr(), _lib.dtype_code(z.dtype), z.stride(0), t.data_ptr(),
              loss.data_ptr(), ent.data_ptr(), corr.data_ptr(), n, z.shape[1], int(grad), scale,
              _lib.stream(z.device))
    torch.cuda.synchronize()
    return loss, ent, corr


def reference(z, t):
    zd = z.double()
    lse = zd.logsumexp(1)
    p = (zd - lse[:, None]).exp()
    ent = lse - torch.where(p > 0, p * zd, 0.0).sum(1)
    lab = t >= 0
    tt = t.clamp(min=0)[:, None]
    loss = torch.where(lab, lse - zd.gather(1, tt)[:, 0], 0.0)
    grad = torch.where(lab[:, None], p.scatter_add(1, tt, -torch.ones_like(tt, dtype=p.dtype)), 0.0)
    return loss, ent, grad, (zd.argmax(1) == t) & lab


def check(got, want, rtol, atol, what):
    err = ((got.double() - want).abs() - rtol * want.abs()).max().item()
    assert err <= atol, (what, err, atol)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n_cols,pad", [(1, 0), (7, 2), (8, 8), (9, 3), (2047, 1), (2049, 0), (4101, 7),
                                        (16391, 2), (32767, 1), (32768, 0), (32769, 5)])
def test_lengths_and_row_alignments(n_cols, pad, dtype, dev):
    banner(f"xent rows {n_cols} columns, stride +{pad}, {dtype}")
    g = torch.Generator(device=dev).manual_seed(n_cols)
    n = 9
    wide = (torch.randn(n, n_cols + pad, device=dev, generator=g) * 3).to(dtype)
    wide[1, :n_cols] = 0.5  # equal logits: the first column is the maximum's
    t = torch.randint(0, n_cols, (n,), device=dev, generator=g)
    t[1], t[2], t[4] = 0, int(wide[2, :n_cols].float().argmax()), -100
    keep = wide.clone()
    loss, ent, grad, corr = reference(wide[:, :n_cols], t)
    # A term e^x carries a few ulps and the rounding of its argument, |x| log2 e 2^-24 with the
    # weight e^x (below 2^-22 for every x <= 0); sums of n terms in a tree and chains of a few
    # dozen add less than 2^-19. ln and the final differences are relative to |lse| and |z|.
    tol = 2.0 ** -18 * (1 + float(wide.float().abs().max()))
    for write in (False, True):
        z = wide if write else wide.clone()
        got = run(z[:, :n_cols], t, write)
        check(got[0], loss, 0, tol, "loss")
        check(got[1], ent, 0, tol, "entropy")
        assert torch.equal(got[2].bool(), corr)
    # the stored rounding of the type (its subnormal step 2^-24 in fp16), and p - 1 at the label
    check(wide[:, :n_cols], grad, torch.finfo(dtype).eps + tol, 2.0 ** -22, "grad")
    assert torch.equal(wide[:, n_cols:], keep[:, n_cols:])  # between the rows nothing is written


@pytest.mark.parametrize("n_cols", [200, 5003, 40001])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_special_logits(n_cols, dtype, dev):
    banner(f"xent rows special values {n_cols} {dtype}")
    g = torch.Generator(device=dev).manual_seed(3)
    inf, low = float("inf"), torch.finfo(dtype).min
    z = torch.randn(8, n_cols, device=dev, generator=g).to(dtype)
    z[0, 16:120] = -inf          # whole chunks, alone in some lanes
    z[1, :-1] = -inf             # one logit left
    z[2, 16:120] = low
    z[3, 3:] = low
    z[4, 16:24] = float("nan")   # one chunk
    z[5, 40] = inf
    z[6] = -inf
    z[7, :64] = -inf
    t = torch.tensor([5, n_cols - 1, 5, 1, 5, 5, 5, 100], device=dev)
    loss, ent, grad, _ = reference(z, t)
    got_loss, got_ent, got_corr = run(z, t, True)
    ok = [0, 1, 2, 3, 7]
    tol = 2.0 ** -18 * (1 + 6.0)
    check(got_loss[ok], loss[ok], 0, tol, "loss")
    check(got_ent[ok], ent[ok], 0, tol, "entropy")
    check(z[ok], grad[ok], torch.finfo(dtype).eps + tol, 2.0 ** -22, "grad")
    assert got_corr[1].item() == 1
    assert torch.isnan(got_loss[[4, 5, 6]]).all()
