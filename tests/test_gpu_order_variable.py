"""GIRIH_XCD_ORDER names the workgroup order that a stepper starts with, 0 (plain) too;
without it sweeps go by the rule."""
import pytest

from girih_amd import gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t_block", [1, 4])
@pytest.mark.parametrize("value", ["0", "1", "2", None])
def test_variable_sets_the_order(monkeypatch, value, t_block):
    monkeypatch.delenv("GIRIH_XCD_ORDER", raising=False)
    if value is not None:
        monkeypatch.setenv("GIRIH_XCD_ORDER", value)
    with gpu.Stepper(1, 70, 40, 30, dtype=gpu.GR_F32, coef=[0.4, 0.1], t_block=t_block) as st:
        assert st.stats()["xcd_order"] == (int(value) if value else 2)
