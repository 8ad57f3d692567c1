"""Launches too small for the large tiles: the smaller configurations give the bits of the larger ones, and symmetric products that
read and write the caller's tensors directly."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(1, 1), (64, 64), (65, 130), (128, 384), (200, 900), (513, 520), (640, 1700), (1030, 1100), (1024, 3001)])
@pytest.mark.parametrize("prec", ["bf16", "f16"])
def test_matrix_alone_and_in_a_large_batch(gpu_device, m, n, prec):
    """Alone: tiles of 64 or the deep pipeline; in the batch: the tiles of 128 and 256 that fill the chip."""
    import archscale_amd.optim.newton_schulz_hip as ns
    batch = 20 if m > 512 else 48
    g = torch.Generator().manual_seed(m * 10000 + n)
    x = (torch.randn(batch, m, n, generator=g) * 1e-3).to(torch.bfloat16).to(gpu_device)
    for t in (x, x.mT.contiguous()):
        all_ = ns.newton_schulz(t, prec=prec)
        for i in (0, batch - 1):
            assert torch.equal(ns.newton_schulz(t[i], prec=prec), all_[i])


@pytest.mark.parametrize("n,k", [(128, 64), (256, 1024), (384, 320), (1280, 1024)])
@pytest.mark.parametrize("addend", [False, True])
def test_symmetric_product_in_place_and_through_the_workspace(gpu_device, n, k, addend):
    """Aligned operands are used as they lie.  The same product from an unaligned view, into a strided result and over its own
    operand goes through the workspace and gives the same bits."""
    import archscale_amd.optim.newton_schulz_hip as ns
    g = torch.Generator().manual_seed(n + k)
    a = (torch.randn(2, n, k, generator=g)).to(torch.bfloat16).to(gpu_device)
    c = (torch.randn(n, n, generator=g)).to(torch.bfloat16).to(gpu_device)
    c = torch.triu(c) + torch.triu(c, 1).T

    def product(t, cc=c, out=None):
        return ns._syrk(t, cc if addend else None, 1.5, -0.75 if addend else 0.0, out)

    got = product(a[0])
    a64 = a[0].double()
    want = 1.5 * (a64 @ a64.T) - (0.75 * c.double() if addend else 0)
    mag = 1.5 * (a64.abs() @ a64.abs().T) + (0.75 * c.double().abs() if addend else 0)
    assert bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + mag * (k + 2) * 2.0 ** -24).all())
    for pad, shift in ((8, 8), (8, 0), (3, 1)):      # rows and start aligned to 16 bytes, and not
        wide = torch.zeros(n, k + pad, dtype=torch.bfloat16, device=gpu_device)
        wide[:, shift:shift + k] = a[0]
        cw = torch.zeros(n, n + pad, dtype=torch.bfloat16, device=gpu_device)
        cw[:, shift:shift + n] = c
        dw = torch.full((n, n + pad), 7.0, dtype=torch.bfloat16, device=gpu_device)
        assert torch.equal(product(wide[:, shift:shift + k], cw[:, shift:shift + n], dw[:, shift:shift + n]), got)
        rest = torch.cat([dw[:, :shift], dw[:, shift + n:]], 1)
        assert bool((rest == 7.0).all())             # nothing beside the result is touched
    if addend:
        cc = c.clone()
        assert torch.equal(product(a[0], cc, cc), got)          # over its own addend
    else:
        assert torch.equal(ns._syrk(a, None, 1.5, 0.0, None)[0], got)
        if n == k:
            t = a[0].clone()
            assert torch.equal(product(t, out=t), got)
    sq = torch.randn(n, n, generator=g).to(torch.bfloat16).to(gpu_device)
    ref = ns._syrk(sq, None, 1.0, 0.0, None)
    assert torch.equal(ns._syrk(sq, None, 1.0, 0.0, sq), ref)   # over its own operand


def test_leftover_tiles_in_sixteenths(gpu_device):
    """136 triangle tiles of 256 (short side 4096): 128 in quadrants and 8 in sixteenths alone, whole rounds and a quartered or
    sixteenth rest in batches of 2 and 3."""
    import archscale_amd.optim.newton_schulz_hip as ns
    g = torch.Generator(device=gpu_device).manual_seed(11)
    x = (torch.randn(3, 4000, 4100, generator=g, device=gpu_device) * 1e-3).to(torch.bfloat16)
    coeffs = ns.QUINTIC_SCHEDULE[:3]
    three = ns.newton_schulz(x, coeffs)
    assert torch.equal(ns.newton_schulz(x[:2], coeffs), three[:2])
    for i in range(3):
        assert torch.equal(ns.newton_schulz(x[i], coeffs), three[i])


@pytest.mark.parametrize("normalize_by", ["add", "clamp"])
def test_many_classes_in_one_call(gpu_device, normalize_by):
    """More classes than one staging or product launch holds, both element types and orientations, padded extents, views, and a
    matrix with more partial sums than a copy block adds up itself: every matrix as alone."""
    import archscale_amd.optim.newton_schulz_hip as ns
    g = torch.Generator().manual_seed(5)
    shapes = [(64, 64), (65, 100), (100, 65), (1, 7), (7, 1), (3, 128, 200), (2, 200, 128), (300, 64), (64, 300), (129, 129),
              (2, 640, 160), (160, 640), (512, 100), (33, 1000), (1000, 33), (2, 96, 96), (256, 512), (520, 513), (2900, 2900)]
    xs = []
    for i, s in enumerate(shapes):
        t = torch.randn(*s[:-1], s[-1] + (8 if i % 4 == 1 else 0), generator=g) * 10.0 ** (i % 5 - 2)
        t = t.to(torch.float32 if i % 3 == 0 else torch.bfloat16).to(gpu_device)
        xs.append(t[..., 8:] if i % 4 == 1 else t)
    for first in (True, False):
        kw = dict(eps_mode=normalize_by, cast_input_first=first)
        outs = ns.newton_schulz_grouped(xs, **kw)
        for x, o in zip(xs, outs):
            assert torch.equal(o, ns.newton_schulz(x, **kw)), tuple(x.shape)


def test_only_newton_schulz_launches_are_recorded(gpu_device):
    """The launch records serve the accounting of a Newton-Schulz call: single products and the power iteration share its kernels
    but not its records."""
    import archscale_amd.optim.newton_schulz_hip as ns
    from archscale_amd import _lib
    from archscale_amd.emerging import spectral_norm
    a = torch.randn(256, 512, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(gpu_device)
    _lib.profile_begin()
    ns.ns_line_1(a)
    spectral_norm(a[None], 10)
    assert _lib.profile_collect() == []
    _lib.profile_begin()
    ns.newton_schulz(a, gram_tail=False)
    recs = _lib.profile_collect()
    assert len(recs) == 15 and all(r["kind"] == "gemm" and r["flops_algorithmic"] > 0 for r in recs)


@pytest.mark.parametrize("shape", [(1, 128, 128), (3, 128, 192), (2, 192, 128), (2, 256, 320), (1, 1024, 1088), (2, 640, 256), (1, 1152, 1024),
                                   (2, 128, 200), (2, 130, 256), (1, 256, 1028)])
def test_spectral_norms_of_matrices_where_they_lie(gpu_device, shape):
    """bfloat16 matrices whose extents need no padding are read in place, fp32 copies of the same values through the workspace:
    the same norms bit for bit, rows apart and matrices apart included."""
    from archscale_amd.emerging.spectral_ball_utils import power_iteration, spectral_norm
    g = torch.Generator().manual_seed(shape[1] + shape[2])
    b, r, c = shape
    wide = (torch.randn(2 * b, r, c + 24, generator=g) * 0.02).to(torch.bfloat16).to(gpu_device)
    for W in (wide[:b, :, :c].contiguous(), wide[::2, :, 8:8 + c], wide[b:, :, 4:4 + c]):   # dense; strided; not 16-byte aligned
        for steps in (1, 7, 50):
            assert torch.equal(spectral_norm(W, steps), spectral_norm(W.float(), steps)), steps
        for got, want in zip(power_iteration(W, 7), power_iteration(W.float(), 7)):
            # (the long-side vector of a tall matrix in place is summed in another order: an fp32 sum of unit size moves by about
            # 1e-6, a value that is then rounded to bfloat16 by one place, 2^-7 at most)
            assert torch.allclose(got.float(), want.float(), rtol=2.0 ** -7, atol=2e-6)
        u = power_iteration(W, 7)[1].float().squeeze(-1)
        assert torch.allclose(u.norm(dim=-1), torch.ones(b, device=gpu_device), atol=4e-3)


@pytest.mark.parametrize("shape", [(1, 6144, 128), (3, 192, 128), (2, 1088, 1024), (1, 8256, 128), (2, 3008, 384), (1, 9024, 1152)])
@pytest.mark.parametrize("transposed", [False, True])
def test_squares_of_tall_matrices_where_they_lie(gpu_device, shape, transposed):
    """Fewer and more elements than the blocks of the first launch take at once, rows that a wave fills several times and only in part;
    stored long side first, or short side first and meant transposed: the norms of fp32 copies, bit for bit."""
    import ctypes
    from archscale_amd import _lib
    b, rows, cols = shape if not transposed else (shape[0], shape[2], shape[1])
    g = torch.Generator(device=gpu_device).manual_seed(rows)
    wide = (torch.randn(2 * b, rows, cols + 24, generator=g, device=gpu_device) * 0.02).to(torch.bfloat16)
    L = _lib.lib()

    def norms(w, steps):
        n, out = w.shape[0], torch.empty(w.shape[0], device=gpu_device)
        ptrs = (ctypes.c_void_p * n)(*[w[i].data_ptr() for i in range(n)])
        q = (_lib.SnProblem * 1)()
        q[0].w_ptrs, q[0].sigma_out = ctypes.cast(ptrs, ctypes.POINTER(ctypes.c_void_p)), out.data_ptr()
        q[0].dtype, q[0].ld, q[0].batch, q[0].rows, q[0].cols = _lib.dtype_code(w.dtype), w.stride(-2), n, rows, cols
        q[0].flags = _lib.SN_TRANSPOSED if transposed else 0
        ws = _lib.workspace(gpu_device, L.muon_spectral_norm_workspace_bytes(q, 1), tag="sn")
        _lib.check(L.muon_spectral_norm(q, 1, steps, ws.data_ptr(), ws.numel(), _lib.current_stream_ptr(gpu_device)), "muon_spectral_norm")
        return out

    for w in (wide[:b, :, :cols].contiguous(), wide[::2, :, 8:8 + cols]):
        for steps in (1, 7):
            assert torch.equal(norms(w, steps), norms(w.float(), steps))
    w.fill_(0)
    assert not norms(w, 2).any()


@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 1, 257), (2, 255, 256), (2, 130, 4096), (1, 4097, 64), (1, 33, 8200)])
def test_unit_vectors_and_norm_from_one_launch(gpu_device, shape):
    """Around the ends of a thread's run of 16 elements: sigma has the bits of the call for norms alone, the unit vectors are those of
    the call that leaves them unnormalised (an fp32 norm of n elements is off by less than n 2^-24, then one rounding to bfloat16)."""
    import ctypes
    from archscale_amd import _lib
    from archscale_amd.emerging.spectral_ball_utils import power_iteration, spectral_norm
    b, r, c = shape
    g = torch.Generator().manual_seed(r + c)
    W = (torch.randn(b, r, c, generator=g) * 0.02).to(torch.bfloat16).to(gpu_device)
    sigma, u, v = power_iteration(W, 6)
    assert torch.equal(sigma, spectral_norm(W, 6))
    raw = [torch.empty(b, n, device=gpu_device) for n in (r, c)]
    s = torch.empty(b, device=gpu_device)
    ptrs = (ctypes.c_void_p * b)(*[W[i].data_ptr() for i in range(b)])
    pp = ctypes.cast(ptrs, ctypes.POINTER(ctypes.c_void_p))
    prob = (_lib.SnProblem * 1)()
    prob[0].w_ptrs, prob[0].sigma_out, prob[0].dtype, prob[0].ld, prob[0].batch, prob[0].rows, prob[0].cols, prob[0].flags = pp, s.data_ptr(), 0, c, b, r, c, 0
    L = _lib.lib()
    ws = _lib.workspace(W.device, L.muon_spectral_norm_workspace_bytes(prob, 1), tag="sn")
    _lib.check(L.muon_power_iteration(pp, 0, c, b, r, c, 6, s.data_ptr(), raw[0].data_ptr(), raw[1].data_ptr(), ws.data_ptr(),
                                      ws.numel(), _lib.current_stream_ptr(W.device)), "muon_power_iteration")
    assert torch.equal(s, sigma)
    for got, x in zip((u, v), raw):
        want = x.double() / x.double().norm(dim=-1, keepdim=True)
        assert bool(((got.squeeze(-1).double() - want).abs() <= want.abs() * (2.0 ** -8 + x.shape[-1] * 2.0 ** -24)).all())


@pytest.mark.parametrize("shape", [(192, 128), (100, 130), (128, 128), (33, 8200)])
@pytest.mark.parametrize("value", [float("inf"), 3e38, float("nan")])
def test_unit_vectors_of_lengths_that_are_not_numbers(gpu_device, shape, value):
    """A vector with a NaN or an infinity after the last round is what dividing it by its norm makes of it: NaN in every place the
    norm is one, not only where the vector was."""
    import ctypes
    from archscale_amd import _lib
    from archscale_amd.emerging.spectral_ball_utils import power_iteration
    W = (torch.randn(1, *shape, generator=torch.Generator().manual_seed(8)) * 0.02)
    W.view(-1)[W.numel() // 3] = value
    W = W.to(torch.bfloat16).to(gpu_device)
    r, c = shape
    L = _lib.lib()
    for steps in (1, 2, 7):
        _, u, v = power_iteration(W, steps)
        raw = [torch.empty(1, n, device=gpu_device) for n in (r, c)]
        s = torch.empty(1, device=gpu_device)
        pp = ctypes.cast((ctypes.c_void_p * 1)(W.data_ptr()), ctypes.POINTER(ctypes.c_void_p))
        prob = (_lib.SnProblem * 1)()
        prob[0].w_ptrs, prob[0].sigma_out, prob[0].ld, prob[0].batch, prob[0].rows, prob[0].cols = pp, s.data_ptr(), c, 1, r, c
        ws = _lib.workspace(W.device, L.muon_spectral_norm_workspace_bytes(prob, 1), tag="sn")
        _lib.check(L.muon_power_iteration(pp, 0, c, 1, r, c, steps, s.data_ptr(), raw[0].data_ptr(), raw[1].data_ptr(), ws.data_ptr(),
                                          ws.numel(), _lib.current_stream_ptr(W.device)), "muon_power_iteration")
        for got, x in zip((u, v), raw):
            want = x / x.norm(dim=-1, keepdim=True).clamp_min(1e-12)
            assert torch.equal(got.squeeze(-1).isnan(), want.isnan()), steps


@pytest.mark.parametrize("batch,n,k", [(1, 128, 3840), (1, 256, 4096), (2, 300, 4000), (1, 1000, 8200), (1, 640, 16384), (3, 512, 4096)])
@pytest.mark.parametrize("addend", [False, True])
def test_few_tiles_with_a_long_reduction(gpu_device, batch, n, k, addend):
    """Products whose reduction is cut into parts: bf16 rounding of the fp32 result, the same bits every time, symmetric."""
    import archscale_amd.optim.newton_schulz_hip as ns
    from archscale_amd import _lib
    g = torch.Generator().manual_seed(n + k)
    a = (torch.randn(batch, n, k, generator=g) / k ** 0.5).to(torch.bfloat16).to(gpu_device)
    a = a[0] if batch == 1 else a
    c = None
    if addend:
        c = torch.randn(*a.shape[:-2], n, n, generator=g) * 0.1
        c = (c + c.mT).to(torch.bfloat16).to(gpu_device)
    want = a.float() @ a.float().mT.contiguous()
    if addend:
        want = 1.2 * want - 0.7 * c.float()
    first = None
    for fill in (0, 0x7f, 0xff):   # whatever the workspace holds
        for ws in list(_lib._workspaces.values()):
            ws.fill_(fill)
        got = ns.ns_line_1(a) if c is None else (ns.tsyrk_ex(a, c, alpha=1.2, beta=-0.7) if batch == 1 else ns._syrk(a, c, 1.2, -0.7, None))
        assert torch.equal(got, got.mT)
        first = got if first is None else first
        assert torch.equal(got, first)
    # one bf16 rounding (2^-9 of the value) beside sums of k products in fp32 (k 2^-24 of the root mean square at most)
    assert ((first.float() - want).abs() <= want.abs() * 2.0 ** -8 + 2e-3 * want.pow(2).mean().sqrt()).all()


@pytest.mark.parametrize("batch,n,k", [(4, 640, 16384), (2, 1000, 4000), (4, 1000, 4000), (8, 512, 4096), (17, 512, 4090), (16, 1024, 4096),
                                       (90, 100, 6400)])
@pytest.mark.parametrize("addend", [False, True])
def test_parts_of_a_reduction_do_not_depend_on_the_stack(gpu_device, batch, n, k, addend):
    """Products whose reduction is cut, alone (a block to a part) and in stacks (the same up to 85 tiles of 128, then one block to all
    parts, with both pipelines): equal bits, matrix by matrix."""
    import archscale_amd.optim.newton_schulz_hip as ns
    g = torch.Generator(device=gpu_device).manual_seed(n + k)
    a = (torch.randn(batch, n, k, generator=g, device=gpu_device) / k ** 0.5).to(torch.bfloat16)
    c = None
    if addend:
        c = torch.randn(batch, n, n, generator=g, device=gpu_device) * 0.1
        c = (c + c.mT).to(torch.bfloat16)
    stack = ns._syrk(a, c, 1.2, -0.7 if addend else 0.0, None)
    for i in (0, 1, batch - 1):
        assert torch.equal(ns._syrk(a[i], c[i] if addend else None, 1.2, -0.7 if addend else 0.0, None), stack[i])


@pytest.mark.parametrize("m,n", [(130, 1024), (256, 1090), (511, 1500), (512, 2048), (640, 1025), (2100, 300)])
@pytest.mark.parametrize("prec", ["bf16", "f16"])
def test_tiles_of_32_give_the_bits_of_larger_ones(gpu_device, m, n, prec):
    """Alone, X X^T of these matrices runs in tiles of 32 (short side up to 640, long side from 1024 on); sixteen of them, in larger ones."""
    import archscale_amd.optim.newton_schulz_hip as ns
    g = torch.Generator().manual_seed(m + n)
    x = (torch.randn(16, m, n, generator=g) * 1e-3).to(torch.bfloat16).to(gpu_device)
    batch = ns.newton_schulz(x, prec=prec)
    for i in (0, 15):
        assert torch.equal(ns.newton_schulz(x[i], prec=prec), batch[i])


@pytest.mark.parametrize("m,n,fine", [(130, 1024, True), (512, 2048, True), (640, 1025, True), (512, 890, False), (512, 1000, True), (700, 1500, False), (2100, 300, True)])
def test_which_products_take_tiles_of_32(gpu_device, m, n, fine):
    """X X^T of up to 16 tiles of 128 over at least 1024 k-values (padded to tiles: 890 has 896 of them, 1000 has 1024), alone; none of sixteen such matrices together, and no other product."""
    import archscale_amd.optim.newton_schulz_hip as ns
    from archscale_amd import _lib
    x = (torch.randn(16, m, n, generator=torch.Generator().manual_seed(m + n)) * 1e-3).to(torch.bfloat16).to(gpu_device)
    for t, want in ((x[0], fine), (x, False)):
        _lib.profile_begin()
        ns.newton_schulz(t, gram_tail=False)
        recs = _lib.profile_collect()
        grams = [r for r in recs if r["mode"] == 3]
        assert len(grams) == 5 and all((r["tile"] == 32) == want for r in grams)
        assert all(r["tile"] != 32 for r in recs if r["mode"] != 3)


@pytest.mark.parametrize("shape", [(2, 192, 128), (2, 128, 192), (1, 6144, 128)])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), 3e38])
def test_values_out_of_range_in_matrices_where_they_lie(gpu_device, shape, value):
    """One such value: the norms and vectors of its matrix are those of the fp32 copy, NaN in the same places, and the other matrix of the
    stack does not see it."""
    from archscale_amd.emerging.spectral_ball_utils import power_iteration, spectral_norm
    W = torch.randn(*shape, generator=torch.Generator().manual_seed(4)) * 0.02
    clean = spectral_norm(W.to(torch.bfloat16).to(gpu_device), 5)
    W[0].view(-1)[W[0].numel() // 3] = value
    W = W.to(torch.bfloat16).to(gpu_device)
    for steps in (1, 5):
        for got, want in zip((spectral_norm(W, steps), *power_iteration(W, steps)), (spectral_norm(W.float(), steps), *power_iteration(W.float(), steps))):
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(spectral_norm(W, 5)[1:], clean[1:])
