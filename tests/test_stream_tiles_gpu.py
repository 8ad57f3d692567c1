"""X' = B X with the tiles of a block one after the other: a matrix gives the bits that it gives alone (where launches are too small for
that form), whatever the number of tiles per block, the mix of classes, the orientation of the result and the storage."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _streamed(call):
    """(launches of X' = B X between iterations, final ones) of a call that took the form, or None where the lines are those of another device."""
    from archscale_amd import _lib
    _lib.profile_begin()
    call()
    torch.cuda.synchronize()
    recs = [r for r in _lib.profile_collect() if r["kind"] == "gemm" and r["stream"]]
    assert all(r["mode"] == 2 and r["tile"] == 256 for r in recs)
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        return None
    return sum(not r["final"] for r in recs), sum(r["final"] for r in recs)


def _check(ns, stacks, prec, coeffs, final=True):
    outs = [torch.empty_like(x) for x in stacks]
    took = _streamed(lambda: ns.newton_schulz_grouped(stacks, coeffs, 1e-7, prec=prec, outs=outs))
    assert took is None or (took[0] > 0 and (took[1] > 0) == final), took
    for x, o in zip(stacks, outs):
        for i in {0, x.shape[0] // 2, x.shape[0] - 1}:
            alone = torch.empty_like(x[i])
            took = _streamed(lambda: ns.newton_schulz_grouped([x[i]], coeffs, 1e-7, prec=prec, outs=[alone]))
            assert took is None or took == (0, 0)
            assert torch.equal(alone, o[i]), (tuple(x.shape), i)


# tiles of X' on 256 units: 400, 416, 432 and 480 (most units one, some two), 648, 1280 and 1536, 640 of which 128 go in quadrants; reductions
# from the shortest (K = 256) to the longest (2048); more than eight tile rows; extents that are padded, whose final launch needs bounds checks
@pytest.mark.parametrize("batch,m,n", [(160, 256, 2048), (128, 256, 1280), (52, 512, 1024), (48, 512, 1280), (64, 768, 2048), (6, 2048, 2304),
                                       (12, 1536, 2304), (5, 2048, 2560), (160, 250, 2000), (52, 500, 1000)])
@pytest.mark.parametrize("prec", ["bf16", "f16"])
def test_stacks_of_one_shape(gpu_device, batch, m, n, prec):
    import archscale_amd.optim.newton_schulz_hip as ns
    g = torch.Generator(device=gpu_device).manual_seed(batch + m + n)
    x = (torch.randn(batch, m, n, generator=g, device=gpu_device) * 1e-3).to(torch.bfloat16)
    for t in (x, x.mT.contiguous()):
        _check(ns, [t], prec, ns.QUINTIC_SCHEDULE, final=m % 256 == 0 and n % 256 == 0)


@pytest.mark.parametrize("prec", ["bf16", "f16"])
def test_classes_of_different_reductions_and_orientations(gpu_device, prec):
    """Blocks go from tiles of one problem to those of another: other strides, reductions, results in rows and in columns; iterates below
    and above the size from which X' = B X walks forwards."""
    import archscale_amd.optim.newton_schulz_hip as ns
    g = torch.Generator(device=gpu_device).manual_seed(3)
    for scale in (1, 3):
        shapes = [(10 * scale, 512, 2048), (9 * scale, 2048, 256), (5 * scale, 1024, 1024), (4 * scale, 2816, 1024), (7 * scale, 256, 3072)]
        stacks = [(torch.randn(*s, generator=g, device=gpu_device) * 1e-3).to(torch.bfloat16) for s in shapes]
        _check(ns, stacks, prec, ns.QUINTIC_SCHEDULE)


def test_results_that_are_not_aligned(gpu_device):
    """A result that is not 16-byte aligned leaves the form for the final launch: the same bits, nothing beside it is touched."""
    import archscale_amd.optim.newton_schulz_hip as ns
    g = torch.Generator(device=gpu_device).manual_seed(4)
    x = (torch.randn(160, 256, 2048, generator=g, device=gpu_device) * 1e-3).to(torch.bfloat16)
    want = torch.empty_like(x)
    took = _streamed(lambda: ns.newton_schulz_grouped([x], ns.QUINTIC_SCHEDULE, 1e-7, outs=[want]))
    assert took is None or (took[0] > 0 and took[1] == 1)
    flat = torch.full((want.numel() + 8,), 7.0, dtype=torch.bfloat16, device=gpu_device)
    took = _streamed(lambda: ns.newton_schulz_grouped([x], ns.QUINTIC_SCHEDULE, 1e-7, outs=[flat[1:1 + want.numel()].view(want.shape)]))
    assert took is None or (took[0] > 0 and took[1] == 0)
    assert torch.equal(flat[1:1 + want.numel()].view(want.shape), want)
    assert bool((flat[:1] == 7.0).all()) and bool((flat[1 + want.numel():] == 7.0).all())


# launches that take the form but for their result: extents of whole tiles inside a wider matrix (which they keep), and padded ones; wide and tall
@pytest.mark.parametrize("batch,m,n", [(160, 256, 2048), (52, 512, 1024), (160, 250, 2000), (52, 500, 1000)])
@pytest.mark.parametrize("tall", [False, True])
@pytest.mark.parametrize("left,right", [(8, 24), (3, 0)])
def test_results_inside_wider_matrices(gpu_device, batch, m, n, tall, left, right):
    """Results whose rows lie further apart than they are long: the bits of contiguous ones, nothing beside them is touched."""
    import archscale_amd.optim.newton_schulz_hip as ns
    from archscale_amd import _lib
    rows, cols = (n, m) if tall else (m, n)
    g = torch.Generator(device=gpu_device).manual_seed(batch + m + n)
    x = (torch.randn(batch, rows, cols, generator=g, device=gpu_device) * 1e-3).to(torch.bfloat16)
    want = torch.empty_like(x)
    ns.newton_schulz_grouped([x], ns.QUINTIC_SCHEDULE, 1e-7, outs=[want])
    wide = torch.full((batch, rows, left + cols + right), 7.0, dtype=torch.bfloat16, device=gpu_device)
    view = wide[:, :, left:left + cols]
    q = (_lib.NsProblem * 1)()
    q[0].in_ptr, q[0].out_ptr, q[0].in_dtype, q[0].in_ld, q[0].out_ld = x.data_ptr(), view.data_ptr(), _lib.dtype_code(x.dtype), cols, wide.shape[2]
    q[0].in_batch_stride, q[0].out_batch_stride, q[0].batch, q[0].rows, q[0].cols = rows * cols, rows * wide.shape[2], batch, rows, cols
    L = _lib.lib()
    ws = _lib.workspace(gpu_device, L.muon_ns_grouped_workspace_bytes(q, 1, _lib.PREC_BF16))
    took = _streamed(lambda: _lib.check(L.muon_ns_grouped(
        q, 1, _lib.abc_array(ns.QUINTIC_SCHEDULE), 5, 1e-7, _lib.EPS_ADD, _lib.PREC_BF16, _lib.NS_CAST_INPUT_FIRST, ws.data_ptr(), ws.numel(),
        _lib.current_stream_ptr(gpu_device)), "muon_ns_grouped"))
    assert took is None or (took[0] > 0 and took[1] == (1 if m % 256 == 0 and left == 8 else 0)), took
    assert torch.equal(view, want)
    assert bool((wide[:, :, :left] == 7.0).all()) and bool((wide[:, :, left + cols:] == 7.0).all())
