"""Single values of the GEMM epilogues, where a tolerance over a whole matrix
does not see them, against 64-bit torch."""
import math

import pytest
import torch

from tests.cce_common import IGNORE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [257, 258, 259, 5003, 2 ** 29 + 261])
def test_bias_of_the_last_columns(gpu, V):
    """The bias is added to every column that exists, whatever V is modulo four
    and where a byte offset from the first column no longer fits 31 bits
    (V 2^29 + 261, d 8: 8.6 GB of weight).  With a zero weight the row's
    log-sum-exp is that of the bias: fp32 holds it to about 1e-6."""
    from chronicals_amd import _lib
    print(f"case last bias V={V}", flush=True)
    w = torch.zeros(V, 8, dtype=torch.bfloat16, device=gpu)
    h = torch.ones(2, 8, dtype=torch.bfloat16, device=gpu)
    lab = torch.tensor([V - 1, IGNORE], device=gpu)
    b = torch.zeros(V, device=gpu)
    for at in (0, V // 2, V - 5, V - 1):
        b[at] = 40.0
        _, lse, _, target = torch.ops.chronicals_hip.cce_fwd(h, w, lab, b, IGNORE, 0.0, 0.0, 0,
                                                             _lib.CCE_REDUCTION_MEAN, _lib.CCE_LSE_ALL_ROWS)
        want = math.log(V - 1 + math.exp(40.0))
        assert float(target[0]) == float(b[V - 1])
        for got in lse.tolist():
            assert abs(got - want) <= 2e-6 * want, (at, got, want)
        b[at] = 0.0


@pytest.mark.parametrize("V,chunk,bias,eps,z", [
    (3001, 8192, False, 0.0, 0.0),   # one band; interior and edge tiles
    (3001, 256, False, 0.1, 1e-4),   # two bands, the first of 1465 columns: labels from there on are the next band's
    (3001, 256, True, 0.0, 0.0),
    (512, 8192, True, 0.1, 0.0),
])
def test_gradient_of_confident_targets(gpu, V, chunk, bias, eps, z):
    """Rows whose target has a probability near 1 (0.998 in the median): the target's entry
    of the logits' gradient G, about p - 1, is a small difference and has to be
    taken before G is rounded to bf16.  G then differs from its 64-bit value by
    2^-8 of itself and by what fp32 logits and exponentials leave in p (1e-5);
    dH = G W and dW = G^T H, returned in fp32, by no more than that error
    carried through, plus 1e-5 of the sums' terms."""
    from chronicals_amd.kernels.cut_cross_entropy import cut_cross_entropy
    print(f"case confident V={V} chunk={chunk} bias={bias} eps={eps} z={z}", flush=True)
    N, d = 300, 128
    g = torch.Generator().manual_seed(V + chunk)
    w = (torch.randn(V, d, generator=g) * 0.1).to(torch.bfloat16).float()
    lab = torch.randint(0, V, (N,), generator=g)
    lab[:3] = torch.tensor([V - 1, V // 2, 0])
    a = torch.linspace(11.0, 13.0, N)[torch.randperm(N, generator=g)]
    h = (w[lab] * a[:, None]).to(torch.bfloat16).float()
    b = torch.randn(V, generator=g) * 0.1 if bias else None
    lab[torch.rand(N, generator=g) < 0.1] = IGNORE
    hd, wd = h.to(gpu).requires_grad_(True), w.to(gpu).requires_grad_(True)
    ld, bd = lab.to(gpu), None if b is None else b.to(gpu).requires_grad_(True)
    cut_cross_entropy(hd, wd, ld, bd, chunk, IGNORE, eps, z, reduction="sum").backward()
    h6, w6 = hd.detach().double(), wd.detach().double()
    x = h6 @ w6.t() + (0.0 if b is None else bd.detach().double())
    lse = torch.logsumexp(x, 1, keepdim=True)
    p = (x - lse).exp()
    valid = (ld != IGNORE).double()[:, None]
    hot = torch.zeros_like(x).scatter_(1, ld.clamp(min=0)[:, None], 1.0)
    top = (p * hot).sum(1)[ld != IGNORE]
    assert 0.99 < float(top.median()) < 0.9999
    G = valid * (p * (1 + 2 * z * lse) - (1 - eps) * hot - eps / V)
    err = 2.0 ** -8 * G.abs() + valid * 1e-5 * p
    for got, ref, bound in ((hd.grad, G @ w6, err @ w6.abs() + 1e-5 * (G.abs() @ w6.abs())),
                            (wd.grad, G.t() @ h6, err.t() @ h6.abs() + 1e-5 * (G.abs().t() @ h6.abs()))):
        over = ((got.double() - ref).abs() / (bound + 1e-12)).max()
        assert float(over) <= 1.0, float(over)
    if b is not None:
        assert ((bd.grad.double() - G.sum(0)).abs() <= err.sum(0) + 1e-5 * G.abs().sum(0) + 1e-12).all()
