"""Edges of the streaming kernels of the vector / vocabulary groups and of the singular-vector pass."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtypes", ["fp32", "bf16", "mixed"])
@pytest.mark.parametrize("numel", [8, 8192 - 8, 8192 + 16, 3 * 8192 + 1])
def test_adam_direction_against_fp64(gpu_device, numel, dtypes):
    """Plain and hyperball AdamW in each access path (one dtype for all arrays, mixed dtypes, unaligned length).  An fp32
    weight differs from the fp64 step by the roundings of the step: at most a few 2^-24 of the weight and of the step; a bf16
    weight additionally by its own rounding, 2^-9 of the value."""
    from archscale_amd.optim import scalar_opts as H
    f32, bf = torch.float32, torch.bfloat16
    wd, gd, md, vd = {"fp32": (f32,) * 4, "bf16": (bf,) * 4, "mixed": (bf, bf, f32, f32)}[dtypes]
    gen = torch.Generator().manual_seed(numel)
    x0 = torch.randn(numel, generator=gen).to(wd)
    g0 = (torch.randn(numel, generator=gen) * 1e-3).to(gd)
    m0 = (torch.randn(numel, generator=gen) * 1e-3).to(md)
    v0 = (torch.randn(numel, generator=gen).square() * 1e-6).to(vd)
    g0[::7], m0[::7], v0[::7] = 0, 0, 0            # a zero direction
    v0[1::7] = 1e-38                               # sqrt(V) far below eps
    lr, b1, b2, eps, step = 1e-2, 0.9, 0.95, 1e-8, 3
    for hyper in (False, True):
        x, g, m, v = (t.clone().to(gpu_device) for t in (x0, g0, m0, v0))
        fn = H.hyperball_adamw_update_foreach if hyper else H.adamw_update_foreach
        fn([x], [g], [m], [v], lr, b1, b2, 0.0, step, eps)
        # the direction from the moments as they were stored
        m64, v64 = m.cpu().double(), v.cpu().double()
        u = m64 / (v64.sqrt() / math.sqrt(1 - b2 ** step) + eps) / (1 - b1 ** step)
        x64 = x0.double()
        if hyper:
            t = lr * x64.norm() / u.norm()
            want = x64 - t * u
            want = want * (x64.norm() / want.norm())
        else:
            t, want = lr, x64 - lr * u
        err = (x.cpu().double() - want).abs()
        bound = 2.0 ** -21 * (x64.abs() + t * u.abs()) + (want.abs() * 2.0 ** -8 if wd is bf else 0)
        assert bool((err <= bound).all()), (hyper, (err / bound).max().item())


@pytest.mark.parametrize("rows,cols", [(1, 1), (33, 65), (64, 64), (100, 257), (300, 70)])
def test_singular_vectors_against_fp64(gpu_device, rows, cols):
    """u and v of a matrix with one dominant direction (converged after a few rounds): the sums over rows and columns at the
    edges of the column blocks and row groups.  The operand is rounded to bf16 before the first product, hence 2^-8."""
    from archscale_amd.emerging import power_iteration
    gen = torch.Generator().manual_seed(rows * 1000 + cols)
    a, b = torch.rand(rows, 1, generator=gen) + 0.5, torch.rand(cols, 1, generator=gen) + 0.5
    w = torch.stack([(a @ b.T + 0.01 * torch.randn(rows, cols, generator=gen)).to(torch.bfloat16) for _ in range(3)])
    s, u, v = power_iteration(w.to(gpu_device), 20)
    U, S, Vh = torch.linalg.svd(w.double(), full_matrices=False)
    for i in range(3):
        for got, want in ((u[i], U[i, :, :1]), (v[i], Vh[i, :1].T)):
            got = got.cpu().double()
            want = want * torch.sign((got * want).sum())
            assert ((got - want).norm() / want.norm()).item() < 2.0 ** -8
        assert abs(s[i].item() - S[i, 0].item()) < 3e-3 * S[i, 0].item()


@pytest.mark.parametrize("numel", [8192 + 16, 8192 + 3])
def test_adam_direction_with_an_epsilon_at_the_bottom_of_the_range(gpu_device, numel):
    """eps sqrt(bias2) below the smallest normal number: a zero moment over a zero second moment stays a zero direction, a
    tiny one gives the finite quotient.  Bound as above."""
    from archscale_amd.optim import scalar_opts as H
    lr, b1, b2, eps, step = 1e-2, 0.875, 1 - 2.0 ** -10, 1e-37, 1   # (betas that fp32 holds exactly)
    x0 = torch.linspace(-1.0, 1.0, numel)
    g0, m0, v0 = torch.zeros(numel), torch.zeros(numel), torch.zeros(numel)
    m0[1::3] = 1e-37
    v0[2::3], m0[2::3] = 1e-6, 1e-3
    for hyper in (False, True):
        x, g, m, v = (t.clone().to(gpu_device) for t in (x0, g0, m0, v0))
        fn = H.hyperball_adamw_update_foreach if hyper else H.adamw_update_foreach
        fn([x], [g], [m], [v], lr, b1, b2, 0.0, step, eps)
        m64, v64 = m.cpu().double(), v.cpu().double()
        u = m64 / (v64.sqrt() / math.sqrt(1 - b2 ** step) + eps) / (1 - b1 ** step)
        x64 = x0.double()
        if hyper:
            t = lr * x64.norm() / u.norm()
            want = x64 - t * u
            want = want * (x64.norm() / want.norm())
        else:
            t, want = lr, x64 - lr * u
        err = (x.cpu().double() - want).abs()
        bound = 2.0 ** -21 * (x64.abs() + t * u.abs())
        assert bool((err <= bound).all()), (hyper, err.max().item())


@pytest.mark.parametrize("numel", [1 << 18, (1 << 18) + 1])
def test_adam_direction_is_the_quotient_to_the_last_bit(gpu_device, numel):
    """With beta1 = 1/2, beta2 = 3/4, step 1, lr = 1/2 and zero weights every other operation of the plain step is exact and
    the new weight is minus the quotient.  The corrected quotient is off by at most 2^-23 + 2^-22 of an ulp (the error of the
    uncorrected one, about two ulp, times the reciprocal's) before its one rounding: never by more than an ulp after it, and
    another last bit in about one of 2^22 quotients."""
    import numpy as np
    from archscale_amd.optim import scalar_opts as H
    gen = torch.Generator().manual_seed(numel)
    eps = 2.0 ** -27
    m0 = torch.randn(numel, generator=gen) * 10.0 ** (torch.rand(numel, generator=gen) * 8 - 6)
    v0 = torch.rand(numel, generator=gen) * 10.0 ** (torch.rand(numel, generator=gen) * 16 - 14)
    x, g, m, v = (t.clone().to(gpu_device) for t in (torch.zeros(numel), torch.zeros(numel), m0, v0))
    H.adamw_update_foreach([x], [g], [m], [v], 0.5, 0.5, 0.75, 0.0, 1, eps)
    mn, vn = m.cpu().numpy(), v.cpu().numpy()
    want = (mn * np.float32(0.5)) / (np.sqrt(vn) + np.float32(eps * 0.5))
    assert want.dtype == np.float32
    off = np.abs((-x).cpu().numpy().view(np.int32).astype(np.int64) - want.view(np.int32).astype(np.int64))
    assert off.max() <= 1 and (off > 0).mean() <= 1e-4, (off.max(), (off > 0).mean())
