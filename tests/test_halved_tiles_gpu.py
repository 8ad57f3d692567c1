"""Symmetric products of a short round of tiles of 256 in tiles of 128: the bits of the matrix alone, for every product of the iteration, the
Gram matrices of the power iteration and single products."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# short reductions up to a full round (192 and 256 tiles of 256), longer ones (200), launches quartered as a whole with long reductions (144 and
# 150 tiles), one that would end in sixteenths (140), one tile a side in one round of smaller tiles (160), a mix of classes, extents that are padded
HALVED = [[(64, 512, 640)], [(64, 512, 700), (64, 250, 700)], [(20, 1024, 1024)], [(144, 256, 4096)], [(15, 1000, 4096)], [(14, 1024, 4096)],
          [(160, 250, 1000)], [(20, 1020, 1030)], [(8, 1024, 1024), (12, 1024, 2816), (8, 256, 1024)]]


@pytest.mark.parametrize("shapes", HALVED)
@pytest.mark.parametrize("prec", ["bf16", "f16"])
def test_launches_that_are_halved(gpu_device, shapes, prec):
    """They are recorded as tiles of 128, with the matrix-core work of those; and the bits are those of a matrix alone."""
    from archscale_amd import _lib
    import archscale_amd.optim.newton_schulz_hip as ns
    x = [torch.full(s, 1e-3, dtype=torch.bfloat16, device=gpu_device) for s in shapes]
    _lib.profile_begin()
    ns.newton_schulz_grouped(x, ns.QUINTIC_SCHEDULE, 1e-7, prec=prec, gram_tail=False)
    torch.cuda.synchronize()
    recs = [r for r in _lib.profile_collect() if r["kind"] == "gemm" and r["mode"] == 1]
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert recs and all(r["tile"] == 128 for r in recs)
        # per matrix: 2 * 128^2 * K for a tile, a quarter less for one on the diagonal (extents padded to tiles of 256)
        work, t = 0.0, [(s[0], (s[1] + 255) // 256 * 2) for s in shapes]
        for batch, side in t:
            work += batch * 2.0 * 128 * 128 * (side * (side + 1) / 2 - 0.25 * side) * side * 128
        for r in recs:
            assert r["flops_issued"] == pytest.approx(work, rel=1e-9)
    test_bits_of_a_matrix_alone(gpu_device, shapes, prec)


def test_bits_of_a_matrix_alone(gpu_device, shapes=[(3, 640, 700)], prec="bf16"):
    import archscale_amd.optim.newton_schulz_hip as ns
    g = torch.Generator(device=gpu_device).manual_seed(sum(map(sum, shapes)))
    stacks = [(torch.randn(*s, generator=g, device=gpu_device) * 1e-3).to(torch.bfloat16) for s in shapes]
    outs = [torch.empty_like(x) for x in stacks]
    ns.newton_schulz_grouped(stacks, ns.QUINTIC_SCHEDULE, 1e-7, prec=prec, outs=outs)
    for x, o in zip(stacks, outs):
        for i in (0, x.shape[0] - 1):
            assert torch.equal(ns.newton_schulz(x[i], ns.QUINTIC_SCHEDULE, 1e-7, prec=prec), o[i]), (tuple(x.shape), i)


# 108, 120, 126 and 128 tiles of 128: one round of quadrants; 130 and 140 with short and long reductions: not
@pytest.mark.parametrize("shapes", [[(3, 1000, 2000)], [(12, 500, 1100)], [(6, 700, 1300)], [(8, 384, 384), (8, 96, 384), (12, 1032, 384)],
                                    [(13, 512, 1500)], [(13, 512, 700)], [(5, 896, 1000)]])
@pytest.mark.parametrize("prec", ["bf16", "f16"])
def test_quadrants_of_one_round(gpu_device, shapes, prec):
    test_bits_of_a_matrix_alone(gpu_device, shapes, prec)


# 200, 156, 240, 160 and 216 tiles of 256: up to half a second round of smaller tiles, all of it with a short reduction, one round of smaller ones of one
# tile a side, and one that stays in tiles of 256; 128, 90 and 84 tiles: quadrants from a third to half a round, smaller tiles
# below if they are little more than one to a unit
@pytest.mark.parametrize("batch,n,k", [(20, 1024, 1024), (52, 512, 512), (40, 768, 256), (160, 256, 1024), (6, 2048, 768), (128, 256, 1024),
                                       (9, 1000, 700), (28, 512, 256)])
def test_stacks_of_single_products(gpu_device, batch, n, k):
    import archscale_amd.optim.newton_schulz_hip as ns
    g = torch.Generator(device=gpu_device).manual_seed(n + k)
    a = torch.randn(batch, n, k, generator=g, device=gpu_device).to(torch.bfloat16)
    got = ns.ns_line_1(a)
    assert torch.equal(got, got.mT)
    for i in (0, batch // 2, batch - 1):
        assert torch.equal(ns.ns_line_1(a[i]), got[i])
