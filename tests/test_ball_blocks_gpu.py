"""The spherical weight update over blocks inside wider matrices and over dense ones, of any width and start: against fp64, and nothing
beside a block is touched."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("ld_w,ld_phi", [(0, 0), (5, 5), (8, 8), (0, 3), (11, 0)])
@pytest.mark.parametrize("shift", [0, 1])
def test_blocks_of_any_width(gpu_device, dtype, ld_w, ld_phi, shift):
    """Leading dimensions `ld_w` and `ld_phi` beyond the width, starts `shift` elements into the buffers; one to several chunks of 8192, with
    and without a rest of fewer than eight elements, rows shorter than a run of eight and whole runs."""
    from archscale_amd import _lib
    g = torch.Generator().manual_seed(7)
    blocks = [(1, 1), (3, 1), (9000, 1), (9001, 3), (1171, 7), (1025, 8), (2000, 9), (513, 16), (512, 17), (400, 53), (65, 257), (7, 2400), (1, 8193)]
    items, prefix, data = np.zeros(len(blocks), dtype=_lib.BALL_ITEM), [0], []
    lr, decay = 0.02, 0.998
    for it, (rows, cols) in zip(items, blocks):
        w = (torch.randn(shift + rows * (cols + ld_w) + 8, generator=g) * 0.05).to(dtype)
        phi = torch.randn(shift + rows * (cols + ld_phi) + 8, generator=g).to(torch.bfloat16)
        wd, pd = w.to(gpu_device), phi.to(gpu_device)
        it["w"], it["phi"], it["sigma"] = wd.data_ptr() + shift * wd.element_size(), pd.data_ptr() + 2 * shift, 0
        it["ld_w"], it["ld_phi"], it["rows"], it["cols"] = cols + ld_w, cols + ld_phi, rows, cols
        it["radius"], it["lr_ratio"], it["w_dtype"] = 1.0, 0.7, _lib.dtype_code(dtype)
        prefix.append(prefix[-1] + (rows * cols + _lib.CHUNK_ELEMS - 1) // _lib.CHUNK_ELEMS)
        data.append((w, phi, wd, pd))
    tab, pre = torch.from_numpy(items.view(np.uint8).copy()).to(gpu_device), torch.tensor(prefix, dtype=torch.int32, device=gpu_device)
    _lib.check(_lib.lib().muon_ball_apply(tab.data_ptr(), pre.data_ptr(), len(blocks), prefix[-1], lr, decay, _lib.RETRACT_HARD, 0.0, 0,
                                          _lib.current_stream_ptr(gpu_device)), "muon_ball_apply")
    torch.cuda.synchronize()
    fw, fp = float(np.float32(decay)), float(np.float32(np.float32(lr) * np.float32(0.7)))
    for (rows, cols), (w, phi, wd, pd) in zip(blocks, data):
        got, at = wd.cpu(), lambda t, ld: t[shift:shift + rows * (cols + ld)].view(rows, cols + ld)[:, :cols].double()
        a, b = fw * at(w, ld_w), fp * at(phi, ld_phi)
        # three roundings to fp32 of terms of this size (two where the compiler fuses), one to the stored type
        bound = 3 * 2.0 ** -24 * (a.abs() + b.abs()) + (2.0 ** -8 * (a - b).abs() if dtype == torch.bfloat16 else 0)
        assert bool(((at(got, ld_w) - (a - b)).abs() <= bound).all()), (rows, cols)
        inside = torch.zeros(w.numel(), dtype=torch.bool)
        inside[shift:shift + rows * (cols + ld_w)].view(rows, cols + ld_w)[:, :cols] = True
        assert torch.equal(got[~inside], w[~inside]), (rows, cols)
        assert torch.equal(pd.cpu(), phi)
