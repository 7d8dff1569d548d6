"""tests.cce_common.backward_plan against the library's workspace queries: host only."""
import random

import pytest

from chronicals_amd import _lib
from tests.cce_common import backward_plan


@pytest.mark.parametrize("budget_mb", [0, 1, 8])
@pytest.mark.parametrize("gather", ["", "0", "1"])
def test_plan_matches_the_workspace(monkeypatch, budget_mb, gather):
    for name, value in (("CHRONICALS_CCE_G_BUDGET_MB", budget_mb), ("CHRONICALS_CCE_ROW_GATHER", gather)):
        if value:
            monkeypatch.setenv(name, str(value))
        else:
            monkeypatch.delenv(name, raising=False)
    rng = random.Random(budget_mb)
    for _ in range(600):
        N = rng.choice([0, 1, 64, 255, 256, 257, 700, 1088, 2816, 2817, 3072, 4100, 16384, 2 ** 17, rng.randint(1, 9000)])
        d = rng.choice([8, 64, 72, 320, 896, 1000, 3584, 8 * rng.randint(1, 600)])
        V = rng.choice([1, 257, 5003, 50257, 151936, rng.randint(1, 200000)])
        chunk = rng.choice([0, 256, 1000, 4096, 8192, 16384])
        need = [rng.random() < 0.7 for _ in range(4)]
        assert backward_plan(N, d, V, chunk, *need, budget_mb, gather).workspace == \
            _lib.backward_workspace_bytes(N, d, V, chunk, *need), (N, d, V, chunk, need)
