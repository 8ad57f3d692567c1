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
