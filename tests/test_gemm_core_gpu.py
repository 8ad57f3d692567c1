"""The product kernel at the edges of its pipeline: reductions of one to a few k-tiles (fewer than there are LDS stages),
extents around the tile sides, K-contiguous and K-major operands, against fp64 products of the same bf16 inputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bf16(shape, seed, dev, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16).to(dev)


def _check_product(got, want, terms):
    """bf16 result of an fp32 sum: half an ulp of bf16 (2^-9 of the value, doubled for the boundary of a binade) plus the
    sum's own rounding, at most (number of terms) x 2^-24 of the sum of magnitudes."""
    err = (got.double() - want).abs()
    bound = want.abs() * 2.0 ** -8 + terms * 2.0 ** -24 * want.abs().max() * 4 + 1e-30
    assert bool((err <= bound).all()), (err / bound).max().item()


@pytest.mark.parametrize("n", [1, 64, 65, 129, 256, 300])
@pytest.mark.parametrize("k", [1, 64, 65, 128, 192, 257, 384])
def test_symmetric_product_short_reductions(gpu_device, n, k):
    import archscale_amd.optim.newton_schulz_hip as ns
    a = _bf16((n, k), 1000 * n + k, gpu_device)
    a64 = a.double()
    d = ns.ns_line_1(a)
    _check_product(d, a64 @ a64.T, k)
    assert torch.equal(d, d.T)
    # with a symmetric addend
    c = _bf16((n, n), 7, gpu_device)
    c = torch.triu(c) + torch.triu(c, 1).T
    want = 1.5 * (a64 @ a64.T) - 0.75 * c.double()
    got = ns.tsyrk_ex(a, c, alpha=1.5, beta=-0.75)
    err = (got.double() - want).abs()
    mag = 1.5 * (a64.abs() @ a64.abs().T) + 0.75 * c.double().abs()
    assert bool((err <= want.abs() * 2.0 ** -8 + mag * (k + 2) * 2.0 ** -24).all())


@pytest.mark.parametrize("m,n", [(1, 1), (64, 64), (64, 65), (65, 129), (128, 192), (200, 320), (256, 257), (129, 500)])
def test_k_major_product_and_bx_short_reductions(gpu_device, m, n):
    """One iteration (0, 1, 0) is X' = (X X^T) X: the K-major symmetric product over n and the BX product over m, each
    rounded to bf16 once more (A, B = A, X'), so 3 x 2^-9 relative per factor plus the fp32 sums."""
    import archscale_amd.optim.newton_schulz_hip as ns
    x = _bf16((m, n), 31 * m + n, gpu_device, 0.5)
    for t in (x, x.T.contiguous()):
        got = ns.newton_schulz(t, [(0.0, 1.0, 0.0)], 0.0, normalize=False)
        t64 = t.double()
        want = t64 @ t64.T @ t64
        mag = t64.abs() @ t64.abs().T @ t64.abs()
        err = (got.double() - want).abs()
        assert bool((err <= mag * (3 * 2.0 ** -9 + (m + n) * 2.0 ** -24) + 1e-30).all())
