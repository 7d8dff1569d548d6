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
