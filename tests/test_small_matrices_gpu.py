"""GPU: matrices whose whole iteration runs in one block, against the same matrices in the chain of product launches.

A call that holds a larger matrix as well takes the chain for all of its matrices, so a grouped call with a filler matrix is the
general path.  Both do the same products in the same order with the same rounding: the bits have to agree.
"""
import pytest
import torch

from archscale_amd.optim import newton_schulz_hip as H

pytestmark = pytest.mark.gpu

POLAR = [(8.2051, -22.9019, 16.4607), (4.0664, -2.8612, 0.5184), (3.9096, -2.8234, 0.5250), (3.2856, -2.4153, 0.4853),
         (2.2779, -1.6198, 0.3985)]
KINDS = {
    "quintic": dict(coeffs=H.QUINTIC_SCHEDULE),
    "no tail": dict(coeffs=H.QUINTIC_SCHEDULE, gram_tail=False),
    "constant, half": dict(coeffs=[H.SIMPLE_ROW] * 5, prec="f16"),
    "polar, half, fp32 norm": dict(coeffs=POLAR, prec="f16", cast_input_first=False),
    "half with tail": dict(coeffs=H.QUINTIC_SCHEDULE, prec="f16", gram_tail=True),
    "one row": dict(coeffs=[H.SIMPLE_ROW]),
}
# (batch, rows, cols): edges of the fragments, of the two kernels (short side 64 / 128) and of what fits one compute unit
SHAPES = [(1, 1, 1), (2, 1, 9), (1, 15, 17), (3, 64, 64), (2, 65, 64), (1, 128, 128), (2, 127, 129), (1, 128, 384), (1, 384, 127),
          (2, 97, 383), (1, 64, 1152), (1, 1151, 33), (1, 63, 770), (1, 128, 385), (1, 64, 1153)]


def _input(batch, rows, cols, dtype, ld=None):
    g = torch.Generator().manual_seed(1000 * rows + cols)
    x = torch.randn(batch, rows, ld or cols, generator=g) * 1e-3
    return x.to(dtype).cuda()[..., :cols]


def _chain(x, **kw):
    filler = torch.randn(160, 160, generator=torch.Generator().manual_seed(0)).to(x.dtype).cuda()
    return H.newton_schulz_grouped([x, filler], **kw)[0]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_one_block_gives_the_bits_of_the_chain(kind, dtype):
    kw = KINDS[kind]
    for batch, rows, cols in SHAPES:
        x = _input(batch, rows, cols, dtype)
        got, want = H.newton_schulz(x, **kw), _chain(x, **kw)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (batch, rows, cols)


@pytest.mark.parametrize("rows,cols,ld", [(100, 200, 203), (96, 384, 400), (200, 48, 56), (7, 5, 8)])
def test_strided_rows_and_the_input_as_result(rows, cols, ld):
    x = _input(2, rows, cols, torch.bfloat16, ld)
    want = _chain(x)
    assert torch.equal(H.newton_schulz(x).view(torch.int16), want.view(torch.int16))
    y = x.contiguous()
    H.newton_schulz(y, out=y)
    assert torch.equal(y.view(torch.int16), H.newton_schulz(x.contiguous()).view(torch.int16))


def test_results_in_the_place_of_other_inputs():
    """Every input is read before any result is written, also where a result lies over the input of another matrix."""
    # the same stack one matrix further on: more matrices than a round of blocks
    stack = _input(600, 64, 200, torch.bfloat16).contiguous()
    want = H.newton_schulz(stack[:-1].clone())
    H.newton_schulz(stack[:-1], out=stack[1:])
    assert torch.equal(stack[1:].view(torch.int16), want.view(torch.int16))
    # results of one kernel (short side up to 64) over inputs of the other, and each over the other's
    a, b, c = (_input(1, r, k, torch.bfloat16)[0].contiguous() for r, k in ((64, 128), (128, 300), (64, 128)))
    wants = [H.newton_schulz(x.clone()) for x in (a, b, c)]
    over = [b.view(-1)[:64 * 128].view(64, 128), torch.empty_like(b), a]
    outs = H.newton_schulz_grouped([a, b, c], outs=over)
    for got, want in zip(outs, wants):
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    # a result within its own fp32 input
    x = _input(3, 50, 70, torch.float32).contiguous()
    want = H.newton_schulz(x.clone())
    out = x.view(torch.bfloat16).view(-1)[:x.numel()].view(x.shape)
    H.newton_schulz(x, out=out)
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))


def test_many_classes_zeros_and_tiny_norms_in_one_call():
    shapes = [(33 + 3 * i, 40 + 7 * i) for i in range(28)] + [(128, 384), (5, 1000)]
    xs = [_input(1, r, c, torch.bfloat16)[0] for r, c in shapes]
    xs[3].zero_()
    xs[4].mul_(1e-9)
    small = H.newton_schulz_grouped(xs)
    filler = torch.randn(160, 160, generator=torch.Generator().manual_seed(0)).to(torch.bfloat16).cuda()
    chain = H.newton_schulz_grouped(xs + [filler])
    for x, a, b in zip(xs, small, chain):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16)), x.shape
    assert not small[3].any()


def test_calls_of_small_matrices_leave_records():
    """One record per kernel of a call, with the work of the chain's products."""
    from archscale_amd import _lib
    a, b = _input(3, 64, 200, torch.bfloat16), _input(2, 100, 120, torch.bfloat16)
    _lib.profile_begin()
    H.newton_schulz_grouped([a, b])
    recs = _lib.profile_collect()
    assert [(r["kind"], r["side"]) for r in recs] == [("small", 64), ("small", 128)] and all(r["ms"] > 0 for r in recs)
    filler = torch.randn(160, 160, generator=torch.Generator().manual_seed(0)).to(torch.bfloat16).cuda()
    for x, r in zip((a, b), recs):
        work = []
        for xs in ([x, filler], [filler]):
            _lib.profile_begin()
            H.newton_schulz_grouped(xs)
            work.append(sum(q["flops_algorithmic"] for q in _lib.profile_collect()))
        assert r["flops_algorithmic"] == pytest.approx(work[0] - work[1], rel=1e-9) and r["flops_issued"] >= r["flops_algorithmic"]


def test_more_classes_than_one_launch_takes():
    """30 classes with a short side up to 64 and 27 above it: two launches of either kernel."""
    from archscale_amd import _lib
    shapes = [(2 + 2 * i, 64 + 5 * i) for i in range(30)] + [(66 + 2 * i, 129 + 9 * i) for i in range(27)]
    xs = [_input(1 + i % 3, r, c, torch.bfloat16 if i % 2 else torch.float32) for i, (r, c) in enumerate(shapes)]
    _lib.profile_begin()
    small = H.newton_schulz_grouped(xs)
    assert [r["side"] for r in _lib.profile_collect()] == [64, 64, 128, 128]
    filler = torch.randn(160, 160, generator=torch.Generator().manual_seed(0)).to(torch.bfloat16).cuda()
    for x, a, b in zip(xs, small, H.newton_schulz_grouped(xs + [filler])):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16)), x.shape


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -3e38, 1e-38])
def test_values_out_of_range(dtype, value):
    """One such value in the first matrix of a stack: what the chain makes of it, and nothing in the other matrices."""
    for rows, cols in ((64, 64), (40, 300), (128, 384), (97, 30)):
        for kind in ("quintic", "polar, half, fp32 norm"):
            x = _input(3, rows, cols, dtype).contiguous()
            clean = H.newton_schulz(x, **KINDS[kind])
            x[0].view(-1)[rows * cols // 3] = value
            got, want = H.newton_schulz(x, **KINDS[kind]), _chain(x, **KINDS[kind])
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(0.0), want.nan_to_num(0.0)), (rows, cols, kind)
            assert torch.equal(got[1:], clean[1:])
