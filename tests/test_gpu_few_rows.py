"""Calls of few rows: whole-vocabulary bands, no row order for one row tile,
the forward's split counts and the operators' host side, against the oracle."""
import numpy as np
import pytest
import torch

from tests.cce_common import IGNORE
from tests.test_gpu_parity import _rand_case, compare, run_hip, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,d,V,chunk,bias,need_dw,hdtype", [
    (1, 64, 300, 256, False, True, torch.bfloat16),        # one row, one slab of dW
    (64, 448, 9000, 1024, True, True, torch.bfloat16),     # one band; 256 + 192 hidden columns; dH in 17 splits
    (200, 320, 7001, 512, False, True, torch.float32),     # 256 + 64: tail tiles; fp32 gradients
    (256, 136, 70000, 8192, True, True, torch.float16),    # a full row tile, one band of 70144 columns
    (256, 64, 200000, 8192, False, True, torch.bfloat16),  # three bands of equal width
    (255, 192, 5003, 256, True, False, torch.bfloat16),    # frozen weight, ragged band
    (257, 256, 5003, 8192, True, True, torch.bfloat16),    # two row tiles: the row order is back
    (2900, 64, 9000, 1024, False, True, torch.bfloat16),   # 3072 rows in tiles: not widened
])
def test_few_rows(gpu, N, d, V, chunk, bias, need_dw, hdtype):
    print(f"case few rows N={N} d={d} V={V} chunk={chunk} bias={bias} dw={need_dw} {hdtype}", flush=True)
    h, w, lab, b = _rand_case(N, d, V, seed=N + V, ignore_frac=0.3, bias=bias)
    lab[0] = V - 1
    if hdtype == torch.float16:
        h, w = h.half().float(), w.half().float()
    kw = dict(chunk=chunk, z=1e-4)
    got = run_hip(gpu, h, w, lab, b, need_dw=need_dw, hdtype=hdtype, wdtype=hdtype, **kw)
    ref = run_oracle(h, w, lab, b, **kw)
    if not need_dw:
        ref["dw"] = None
    compare(got, ref, f"few rows N{N}d{d}V{V}")
    ignored = (lab == IGNORE).numpy()
    assert not got["dh"][ignored].any()
    again = run_hip(gpu, h, w, lab, b, need_dw=need_dw, hdtype=hdtype, wdtype=hdtype, **kw)
    assert np.array_equal(got["dh"], again["dh"])


@pytest.mark.parametrize("dtype,f32_grad", [(torch.bfloat16, False), (torch.bfloat16, True), (torch.float32, False)])
@pytest.mark.parametrize("V", [1, 37, 5001])
def test_ignored_logits_rows_have_zero_gradient(gpu, dtype, f32_grad, V):
    """Whatever the logits of an ignored row are, its gradient is zero, in the
    autograd backward and in the one-kernel form; the other rows do not change."""
    from chronicals_amd.kernels.logits_cross_entropy import chunked_cross_entropy_loss
    g = torch.Generator().manual_seed(V)
    x = torch.randn(9, V, generator=g).to(dtype)
    lab = torch.randint(0, V, (9,), generator=g)
    lab[::3] = IGNORE
    grads, fused = [], []
    for fill in (None, float("nan")):
        y = x.clone()
        if fill is not None:
            y[::3] = fill
        yd = y.to(gpu).requires_grad_(True)
        chunked_cross_entropy_loss(yd, lab.to(gpu), reduction="sum").backward()
        grads.append(yd.grad.float().cpu())
        fused.append(torch.ops.chronicals_hip.ce_logits_fwd_bwd(y.to(gpu), lab.to(gpu), IGNORE, 0.0, 0.0, 0, 1, True,
                                                                f32_grad)[3].float().cpu())
    for a, c in (grads, fused):
        assert not a[::3].any() and torch.equal(a, c)


def test_operators_host_side(gpu):
    """Views at unaligned offsets and strided labels are taken as they were; a
    backward through an operator, a wrong dtype and operands of two devices raise."""
    from chronicals_amd import _lib
    h, w, lab, _ = _rand_case(40, 64, 500, seed=3)
    hd, wd, ld = h.to(gpu, torch.bfloat16), w.to(gpu, torch.bfloat16), lab.to(gpu)
    args = (None, IGNORE, 0.0, 0.0, 0, _lib.CCE_REDUCTION_MEAN)
    ref = torch.ops.chronicals_hip.cce_fwd(hd, wd, ld, *args)
    buf = torch.zeros(wd.numel() + 1, dtype=torch.bfloat16, device=gpu)
    buf[1:] = wd.reshape(-1)
    strided = torch.stack([ld, ld + 1], 1)[:, 0]
    got = torch.ops.chronicals_hip.cce_fwd(hd, buf[1:].view(500, 64), strided, *args)
    for a, c in zip(ref, got):
        assert torch.equal(a, c)
    with pytest.raises(RuntimeError, match="bf16"):
        torch.ops.chronicals_hip.cce_fwd(hd.float(), wd, ld, *args)
    with pytest.raises(RuntimeError, match="libchronicals_cce error"):
        torch.ops.chronicals_hip.cce_fwd(hd, wd, ld, None, IGNORE, 2.0, 0.0, 0, _lib.CCE_REDUCTION_MEAN)
    with pytest.raises(RuntimeError, match="same device"):
        torch.ops.chronicals_hip.cce_fwd(hd, wd, lab, *args)
    loss = torch.ops.chronicals_hip.cce_fwd(hd.requires_grad_(True), wd, ld, *args)[0]
    with pytest.raises(RuntimeError):
        loss.backward()
