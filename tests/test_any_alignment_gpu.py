"""Parameters, gradients, state and results that start anywhere and have odd widths: the bits of the same tensors at aligned places (the
partition of the work is by elements, not by addresses), and nothing beside them is touched."""
import pytest
import torch

pytestmark = pytest.mark.gpu

GUARD = 9.0


class _Flat:
    """Tensors in one buffer, each `shift` elements past a multiple of 16 bytes, with guard values between them."""

    def __init__(self, tensors, shift, device):
        self.spans, total = [], 0
        for t in tensors:
            self.spans.append((total + shift, total + shift + t.numel()))
            total += (t.numel() + shift + 31) // 16 * 16
        self.buf = torch.full((total,), GUARD, dtype=tensors[0].dtype, device=device)
        self.views = [self.buf[a:b].view(t.shape) for (a, b), t in zip(self.spans, tensors)]
        for v, t in zip(self.views, tensors):
            v.copy_(t)

    def check_guards(self):
        beside = torch.ones_like(self.buf, dtype=torch.bool)
        for a, b in self.spans:
            beside[a:b] = False
        assert bool((self.buf[beside] == GUARD).all())


def _tensors(shapes, scale, dtype, seed, positive=False):
    g = torch.Generator().manual_seed(seed)
    out = [(torch.randn(*s, generator=g) * scale) for s in shapes]
    return [(t.square() if positive else t).to(dtype) for t in out]


MATRICES = [(129, 257), (257, 129), (65, 1001), (3, 61, 95), (7, 5), (1, 3), (300, 43), (128, 384), (130, 1)]
VECTORS = [(4099,), (1,), (7,), (501, 129), (8192,), (8193,)]


def _run(kind, dtype, shift, device):
    from archscale_amd.emerging import Muon as EmergingMuon
    from archscale_amd.emerging import MuonBall
    from archscale_amd.optim.muon import Muon
    shapes = {"ball": [s for s in MATRICES if len(s) == 2], "emerging": [s for s in MATRICES if len(s) == 2]}.get(kind, MATRICES)
    if kind in ("adamw", "hyperball", "lion"):
        shapes = VECTORS
    w = _Flat(_tensors(shapes, 0.02, dtype, 1), shift, device)
    g = _Flat(_tensors(shapes, 1e-3, dtype, 2), shift, device)
    m = _Flat(_tensors(shapes, 3e-3, dtype, 3), shift, device)
    params = [torch.nn.Parameter(v) for v in w.views]
    for p, t in zip(params, g.views):
        p.grad = t
    flats = [w, g, m]
    if kind in ("muon", "muonh", "per_matrix"):
        opt = Muon(params, lr=0.02, weight_decay=0.1, nesterov=True, cautious_wd=True, use_muonh=kind != "muon",
                   muonh_per_matrix=kind == "per_matrix")
    elif kind == "emerging":
        opt = EmergingMuon(params, lr=0.02, momentum_beta=0.95, weight_decay=0.01, weight_decay_method="l2")
    elif kind == "ball":
        opt = MuonBall(params, lr=0.02, momentum_beta=0.9, weight_decay=0.01, split_fc1=True, is_fc1_fn=lambda p: p.shape[0] == 300,
                       fc1_split_shapes=(131, 169))
    else:
        opt = Muon([dict(params=params, algorithm="lion" if kind == "lion" else "adamw")], lr=1e-3, weight_decay=0.1, cautious_wd=True,
                   use_muonh=kind == "hyperball")
        if kind != "lion":
            flats.append(_Flat(_tensors(shapes, 1e-3, dtype, 4, positive=True), shift, device))
            for p, t in zip(params, flats[-1].views):
                opt.state[p]["variance"] = t
    for p, t in zip(params, m.views):
        opt.state[p]["momentum_buffer" if kind in ("emerging", "ball") else "momentum"] = t
    opt.step()
    torch.cuda.synchronize()
    for f in flats:
        f.check_guards()
    return [[v.clone() for v in f.views] for f in flats]


@pytest.mark.parametrize("kind", ["muon", "muonh", "per_matrix", "emerging", "ball", "adamw", "hyperball", "lion"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_steps_do_not_depend_on_where_tensors_start(gpu_device, kind, dtype):
    want = _run(kind, dtype, 0, gpu_device)
    for shift in (1, 3):
        got = _run(kind, dtype, shift, gpu_device)
        for a, b in zip(want, got):
            for x, y in zip(a, b):
                assert torch.equal(x, y), (shift, tuple(x.shape))


@pytest.mark.parametrize("shape", [(100, 384), (128, 77), (64, 1151), (513, 520), (1001, 250), (2, 1030, 1101), (40, 511, 1001), (1, 4), (3, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_orthogonalisation_of_views(gpu_device, shape, dtype):
    """Inputs and results that start anywhere, and inputs inside a wider matrix."""
    import archscale_amd.optim.newton_schulz_hip as ns
    x = _tensors([shape], 1e-3, dtype, 5)[0].to(gpu_device)
    want = ns.newton_schulz(x)
    for shift in (1, 2, 5):
        a, o = _Flat([x], shift, gpu_device), _Flat([want * 0], shift, gpu_device)
        ns.newton_schulz_grouped([a.views[0]], ns.QUINTIC_SCHEDULE, 1e-7, outs=[o.views[0]])
        assert torch.equal(o.views[0], want), shift
        a.check_guards()
        o.check_guards()
    # rows inside wider matrices: those of a leading dimension that is a multiple of eight at an aligned place, and odd ones anywhere
    cols = shape[-1]
    aligned = torch.full((*shape[:-1], (cols + 15) // 8 * 8), GUARD, dtype=dtype, device=gpu_device)
    aligned[..., :cols] = x
    want = ns.newton_schulz(aligned[..., :cols])
    for left, right in ((3, 2), (1, 4), (8, 0)):
        wide = torch.full((*shape[:-1], left + cols + right), GUARD, dtype=dtype, device=gpu_device)
        wide[..., left:left + cols] = x
        assert torch.equal(ns.newton_schulz(wide[..., left:left + cols]), want), (left, right)
