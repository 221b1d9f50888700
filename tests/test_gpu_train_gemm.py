"""The training block's output projection (attention_op.project: nc_linear_residual_rms) and its weight gradient
(attention_op.add_weight_grad: nc_weight_grad) against float64 on the CPU, at sizes around their tiles, stages and
slices, and the operands that go round the kernels.

Bounds. Products of two bf16 values are exact in fp32, and a sum of n of them in any order is within n 2^-23 of the sum
of magnitudes (fp32 rounding at every step, doubled for the matrix cores' own accumulation); the bf16 result adds half a
bf16 step, 2^-9 of the value (2^-8 allowed)."""
import numpy as np
import pytest
import torch

from nanochat_amd import attention_op as op

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -23


def bf(gen, *shape, scale=1.0):
    return (torch.randn(*shape, generator=gen) * scale).to(torch.bfloat16)


def check_projection(x, w, res, h, rstd):
    x, w, res = (t.double() for t in (x, w, res))
    want, mag = x @ w.t() + res, x.abs() @ w.abs().t() + res.abs()
    depth = x.size(1) + 1
    assert bool(((h.double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + depth * EPS * mag).all())
    ms = want.square().mean(-1) + EPS
    # each squared sum is off by at most 2 |s| depth EPS mag, and their own sum by its length
    slack = (2 * want.abs() * depth * EPS * mag).mean(-1) / ms + (w.size(0) + 4) * EPS
    assert bool(((rstd.double().cpu() * ms.sqrt() - 1).abs() <= slack).all())


@pytest.mark.parametrize("tokens,C,K", [(1, 128, 128), (17, 256, 128), (128, 768, 768), (129, 384, 256), (300, 640, 640),
                                        (2049, 1280, 1280), (515, 36, 128), (30000, 768, 128)])
def test_projection_matches_float64(device, tokens, C, K):
    gen = torch.Generator().manual_seed(tokens + C)
    x, w, res = bf(gen, tokens, K), bf(gen, C, K, scale=K ** -0.5), bf(gen, tokens, C)
    h, rstd = op.project(x.to(device), w.to(device), res.to(device))
    torch.cuda.synchronize()
    check_projection(x, w, res, h, rstd)


def test_projection_rows_do_not_depend_on_the_others(device):
    """A row's result and rstd have the same bits alone and among 100 (quarter tiles), 700 (quarters of both row halves) and
    30,000 (whole tiles and a round of pieces)."""
    gen = torch.Generator().manual_seed(3)
    x, w, res = (t.to(device) for t in (bf(gen, 30000, 256), bf(gen, 768, 256, scale=1 / 16), bf(gen, 30000, 768)))
    h, rstd = op.project(x, w, res)
    for n in (1, 100, 700):
        h2, r2 = op.project(x[:n], w, res[:n])
        assert torch.equal(h[:n].view(torch.int16), h2.view(torch.int16)) and torch.equal(rstd[:n], r2)


@pytest.mark.parametrize("tokens,C,K", [(1, 128, 128), (31, 256, 256), (33, 384, 128), (257, 768, 768), (2400, 640, 384),
                                        (9995, 1280, 1280), (4096, 8, 2048)])
def test_weight_grad_matches_float64(device, tokens, C, K):
    gen = torch.Generator().manual_seed(tokens)
    dh, x, start = bf(gen, tokens, C), bf(gen, tokens, K), torch.randn(C, K, generator=gen)
    grad = start.to(device)
    op.add_weight_grad(grad, dh.to(device), x.to(device))
    again = start.to(device)
    op.add_weight_grad(again, dh.to(device), x.to(device))
    torch.cuda.synchronize()
    assert torch.equal(grad, again)
    a, b = dh.double(), x.double()
    want, mag = a.t() @ b + start, a.abs().t() @ b.abs() + start.abs()
    assert bool(((grad.double().cpu() - want).abs() <= (tokens + 300) * EPS * mag).all())


def test_operands_the_kernels_do_not_take(device):
    """Strided and misaligned operands give the same result through the library path; no tokens leave the gradient."""
    gen = torch.Generator().manual_seed(9)
    x, w, res = bf(gen, 70, 256), bf(gen, 256, 256, scale=1 / 16), bf(gen, 70, 256)
    dh = bf(gen, 70, 256)
    xd, wd, rd, dd = (t.to(device) for t in (x, w, res, dh))

    def moved(t):   # the same values one element into their storage
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=device)
        buf[1:] = t.flatten()
        return buf[1:].view(t.shape)

    for args in ((xd, wd.t().contiguous().t(), rd), (xd, moved(wd), rd), (xd, wd, moved(rd)),
                 (xd, wd, rd.t().contiguous().t())):
        h, rstd = op.project(*args)
        check_projection(x, w, res, h, rstd)
    want = dh.double().t() @ x.double()
    for a, b in ((dd.t().contiguous().t(), xd), (moved(dd), xd), (dd, moved(xd))):
        grad = torch.zeros(256, 256, device=device)
        op.add_weight_grad(grad, a, b)
        assert np.allclose(grad.double().cpu().numpy(), want.numpy(), rtol=0, atol=1e-3)
    grad = torch.ones(256, 256, device=device)
    op.add_weight_grad(grad, dd[:0], xd[:0])
    assert bool((grad == 1).all())
    assert op.project(xd[:0], wd, rd[:0])[0].shape == (0, 256)


def test_projection_sizes_that_do_not_agree(device):
    """x of another width than the weight, a residual of other rows or columns: an error, as from the library's product."""
    x = torch.zeros(70, 256, dtype=torch.bfloat16, device=device)
    w, res = x.new_zeros(128, 256), x.new_zeros(70, 128)
    for args in ((x, w[:, :128].contiguous(), res), (x[:, :128].contiguous(), w, res), (x, w, res[:69]),
                 (x, w, x), (x.view(70, 2, 128), w, res)):
        with pytest.raises(RuntimeError):
            op.project(*args)
    torch.cuda.synchronize()


def test_weight_gradient_sizes_that_do_not_agree(device):
    """Other token counts or another gradient's shape: an error, and the gradient keeps its values."""
    dh = torch.zeros(70, 128, dtype=torch.bfloat16, device=device)
    x, grad = dh.new_zeros(70, 256), torch.ones(128, 256, device=device)
    for args in ((grad, dh, x[:69]), (grad, dh[:69], x), (grad, dh, dh), (grad[:64], dh, x)):
        with pytest.raises(RuntimeError):
            op.add_weight_grad(*args)
    torch.cuda.synchronize()
    assert bool((grad == 1).all())


@pytest.mark.parametrize("tokens,C,K", [(1, 8, 8), (300, 264, 520), (64, 2056, 768), (33, 1288, 2568), (9000, 2952, 2944),
                                        (1500, 1672, 1664)])
def test_weight_grad_of_one_slice_and_of_wide_results(device, tokens, C, K):
    """One slice added straight into the result, at edges of its tiles, and results of more tiles than half the CUs, which
    take several slices (the guard behind the gradient stays as it is)."""
    gen = torch.Generator().manual_seed(tokens + C)
    dh, x, start = bf(gen, tokens, C), bf(gen, tokens, K), torch.randn(C, K, generator=gen)
    buf = torch.full((C * K + 4096,), 7.0, device=device)
    grad = buf[:C * K].view(C, K)
    grad.copy_(start)
    op.add_weight_grad(grad, dh.to(device), x.to(device))
    torch.cuda.synchronize()
    a, b = dh.double(), x.double()
    want, mag = a.t() @ b + start, a.abs().t() @ b.abs() + start.abs()
    assert bool(((grad.double().cpu() - want).abs() <= (tokens + 300) * EPS * mag).all())
    assert bool((buf[C * K:] == 7).all())
