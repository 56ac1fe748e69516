"""The autotuner's report says what an untuned solver takes, and whether that is the faster one."""
import pytest

from test_autotune import sweep_with


@pytest.mark.parametrize("default_ms,faster", [(0.3, True), (0.7, False)])
def test_the_default_is_timed(default_ms, faster):
    def t(key):
        B, lay, levels, tile, zc = key
        if B == 1:
            return {0: default_ms, 1: 1.0, 2: 0.5, 3: 0.6}[levels]
        return 0.55 * B
    rep, _, nodes = sweep_with(t)
    d = rep["default"]
    assert (d["B"], d["levels"], d["faster_than_choice"]) == (1, 0, faster)
    assert d["ms_per_step"] == pytest.approx(default_ms)
    assert d["per_source_gvox"] == pytest.approx(nodes / default_ms / 1e6, rel=1e-5)
    assert rep["choice"]["levels"] == 2
