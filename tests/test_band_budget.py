"""The backward's band gradient stays within its budget when few rows widen the bands: host only."""
import pytest

from chronicals_amd import _lib


@pytest.mark.parametrize("budget_mb", [1, 4, 8, 64, 0])
@pytest.mark.parametrize("N,V,chunk", [(1, 151936, 8192), (64, 32000, 8192), (512, 151936, 8192), (700, 20000, 256),
                                       (2100, 7000, 2048), (2816, 151936, 4096), (3072, 151936, 8192)])
def test_widened_bands_stay_within_the_budget(monkeypatch, N, V, chunk, budget_mb):
    """With no gradient of hidden or weight the workspace is the two band
    gradient buffers and 24 bytes a row (the rows are read in place).  The
    buffers take at most the budget, or 256 rows of an unwidened band."""
    monkeypatch.setenv("CHRONICALS_CCE_ROW_GATHER", "1")
    if budget_mb:
        monkeypatch.setenv("CHRONICALS_CCE_G_BUDGET_MB", str(budget_mb))
    else:
        monkeypatch.delenv("CHRONICALS_CCE_G_BUDGET_MB", raising=False)
    band = min(chunk, -(-V // 256) * 256)
    bound = max((budget_mb or 512) << 20, 4 * 256 * band)
    got = _lib.backward_workspace_bytes(N, 64, V, chunk, False, False)
    assert got <= bound + 24 * N + 8 * 256
