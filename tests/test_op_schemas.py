"""What tracing sees of the operators: host only."""
import pytest
import torch

import chronicals_amd.ops  # noqa: F401

OPS = ("cce_fwd", "cce_bwd", "ce_logits_fwd", "ce_logits_bwd", "ce_logits_bwd_", "ce_logits_fwd_bwd",
       "ce_logits_fwd_bwd_")


@pytest.mark.parametrize("name", OPS)
def test_operators_are_traceable(name):
    """Compliant with torch.compile's rules for operators, and integers that may be symbolic."""
    op = getattr(torch.ops.chronicals_hip, name).default
    assert torch.Tag.pt2_compliant_tag in op.tags
    assert "SymInt ignore_index" in str(op._schema) and " int " not in str(op._schema)


def test_a_symbolic_integer_is_not_specialised():
    """A chunk size taken from a dynamic shape stays one in the traced graph."""
    from torch.fx.experimental.proxy_tensor import make_fx

    def f(g, h, w, lab, lse, nv):
        return torch.ops.chronicals_hip.cce_bwd(g, h, w, lab, lse, nv, None, -100, 0.0, 0.0, 1, h.shape[0], True, True,
                                                False, False, False)

    def meta(*shape, dtype=torch.float32):
        return torch.empty(shape, dtype=dtype, device="meta")
    args = (meta(), meta(300, 64, dtype=torch.bfloat16), meta(1000, 64, dtype=torch.bfloat16),
            meta(300, dtype=torch.int64), meta(300), meta(1, dtype=torch.int32))
    graph = make_fx(f, tracing_mode="symbolic")(*args).graph
    call = [n for n in graph.nodes if n.target == torch.ops.chronicals_hip.cce_bwd.default]
    assert len(call) == 1 and isinstance(call[0].args[11], torch.fx.Node), call[0].args
