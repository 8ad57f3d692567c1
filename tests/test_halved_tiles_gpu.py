"""Symmetric products of a short round of tiles of 256 in tiles of 128: the bits of the matrix alone, for every product of the iteration, the
Gram matrices of the power iteration and single products."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# short reductions up to a full round (192 and 256 tiles of 256), the band of longer ones (200), a launch quartered as a whole with
# long reductions, one that would end in sixteenths (140), a mix of classes, extents that are padded
@pytest.mark.parametrize("shapes", [[(64, 512, 640)], [(64, 512, 700), (64, 250, 2048)], [(20, 1024, 1024)], [(12, 1000, 2816)], [(14, 1024, 4096)],
                                    [(20, 1020, 1030)], [(8, 1024, 1024), (12, 1024, 2816), (8, 256, 1024)]])
@pytest.mark.parametrize("prec", ["bf16", "f16"])
def test_bits_of_a_matrix_alone(gpu_device, shapes, prec):
    import archscale_amd.optim.newton_schulz_hip as ns
    g = torch.Generator(device=gpu_device).manual_seed(sum(map(sum, shapes)))
    stacks = [(torch.randn(*s, generator=g, device=gpu_device) * 1e-3).to(torch.bfloat16) for s in shapes]
    outs = [torch.empty_like(x) for x in stacks]
    ns.newton_schulz_grouped(stacks, ns.QUINTIC_SCHEDULE, 1e-7, prec=prec, outs=outs)
    for x, o in zip(stacks, outs):
        for i in (0, x.shape[0] - 1):
            assert torch.equal(ns.newton_schulz(x[i], ns.QUINTIC_SCHEDULE, 1e-7, prec=prec), o[i]), (tuple(x.shape), i)


# 108, 120, 126 and 128 tiles of 128: one round of quadrants; 130: not
@pytest.mark.parametrize("shapes", [[(3, 1000, 2000)], [(12, 500, 1100)], [(6, 700, 1300)], [(8, 384, 384), (8, 96, 384), (12, 1032, 384)],
                                    [(13, 512, 1500)]])
@pytest.mark.parametrize("prec", ["bf16", "f16"])
def test_quadrants_of_one_round(gpu_device, shapes, prec):
    test_bits_of_a_matrix_alone(gpu_device, shapes, prec)


@pytest.mark.parametrize("batch,n,k", [(20, 1024, 1024), (40, 512, 512), (70, 768, 256)])
def test_stacks_of_single_products(gpu_device, batch, n, k):
    import archscale_amd.optim.newton_schulz_hip as ns
    g = torch.Generator(device=gpu_device).manual_seed(n + k)
    a = torch.randn(batch, n, k, generator=g, device=gpu_device).to(torch.bfloat16)
    got = ns.ns_line_1(a)
    assert torch.equal(got, got.mT)
    for i in (0, batch // 2, batch - 1):
        assert torch.equal(ns.ns_line_1(a[i]), got[i])
