"""Hidden sizes that are no multiple of the 64-wide K slab, against the oracle."""
import numpy as np
import pytest
import torch

from tests.cce_common import IGNORE
from tests.test_gpu_parity import _rand_case, compare, run_hip, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,d,V,chunk,bias,need_dw,hdtype", [
    (70, 8, 300, 256, False, True, torch.bfloat16),      # one slab of 8 columns
    (300, 56, 900, 512, True, True, torch.bfloat16),     # one slab, one column group short
    (257, 72, 2000, 1024, False, False, torch.float32),  # a second slab of 8 columns; frozen weight
    (600, 200, 3000, 2048, True, True, torch.float16),   # one partly filled 256-wide hidden tile
    (1100, 264, 5000, 1024, False, True, torch.bfloat16),  # 256 + 8: a tail tile of 8 columns, dH split
    (513, 1000, 700, 512, True, True, torch.bfloat16),   # 15 slabs and 40 columns
])
def test_hidden_sizes_off_the_slab(gpu, N, d, V, chunk, bias, need_dw, hdtype):
    """The last slab's columns past d belong to the next row (or lie past the
    operand: hidden and weight end inside larger NaN-filled buffers here) and
    have to count as zero."""
    print(f"case off-slab N={N} d={d} V={V} chunk={chunk} bias={bias} dw={need_dw} {hdtype}", flush=True)
    h, w, lab, b = _rand_case(N, d, V, seed=N + d, ignore_frac=0.2, bias=bias)
    lab[0] = 1
    kw = dict(chunk=chunk, eps=0.1, z=1e-4)
    if hdtype == torch.float16:
        h, w = h.half().float(), w.half().float()
    got = run_hip(gpu, h, w, lab, b, need_dw=need_dw, hdtype=hdtype, wdtype=hdtype, **kw)
    ref = run_oracle(h, w, lab, b, **kw)
    if not need_dw:
        ref["dw"] = None
    compare(got, ref, f"off-slab N{N}d{d}")
    # the same operands at the end of NaN-filled buffers: bitwise the same, so nothing past them was read
    from chronicals_amd.kernels.cut_cross_entropy import cut_cross_entropy
    out = []
    for pad in (0, 4096):
        hb = torch.full((N * d + pad,), float("nan"), dtype=torch.bfloat16, device=gpu)
        wb = torch.full((V * d + pad,), float("nan"), dtype=torch.bfloat16, device=gpu)
        hd, wd = hb[:N * d].view(N, d), wb[:V * d].view(V, d)
        hd.copy_(h)
        wd.copy_(w)
        hd.requires_grad_(True)
        wd.requires_grad_(True)
        loss = cut_cross_entropy(hd, wd, lab.to(gpu), None, chunk, IGNORE)
        out.append([loss.detach()] + list(torch.autograd.grad(loss, [hd, wd])))
    for x, y in zip(*out):
        assert torch.isfinite(x.float()).all() and torch.equal(x, y)


def test_infinite_row_stays_in_its_row(gpu):
    """An infinite hidden row makes its own loss NaN or infinite, not its
    neighbour's: the neighbour's last slab does not take the row's values."""
    N, d, V = 40, 72, 500
    h, w, lab, _ = _rand_case(N, d, V, seed=5, ignore_frac=0.0)
    ref = run_hip(gpu, h, w, lab, reduction="none", need_dh=False, need_dw=False)["loss"]
    h[7] = float("inf")
    got = run_hip(gpu, h, w, lab, reduction="none", need_dh=False, need_dw=False)["loss"]
    rows = np.arange(N) != 7
    assert not np.isfinite(got[7]) and np.array_equal(got[rows], ref[rows])
