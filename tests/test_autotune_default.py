"""The autotuner's choice is never slower than the unbatched default setting (levels 0)."""
import pytest

from test_autotune import sweep_with


@pytest.mark.parametrize("default_ms,chosen", [(0.3, 0), (0.7, 2)])
def test_the_default_is_a_candidate(default_ms, chosen):
    def t(key):
        B, lay, levels, tile, zc = key
        if B == 1:
            return {0: default_ms, 1: 1.0, 2: 0.5, 3: 0.6}[levels]
        return 0.55 * B
    rep, _, _ = sweep_with(t)
    assert [(c["B"], c["zchunk"], c["shape"]) for c in rep["candidates"] if c["levels"] == 0] == [(1, 0, None)]
    assert rep["choice"]["B"] == 1 and rep["choice"]["levels"] == chosen
    assert rep["best"]["1"]["ms_per_step"] == pytest.approx(min(default_ms, 0.5))
