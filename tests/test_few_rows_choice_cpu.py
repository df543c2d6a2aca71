"""When a mixer model's product of a few rows leaves ``F.linear`` for its own kernel: not where anything besides the plain
product is asked for. The shapes and devices the kernel takes count as given here."""
import pytest
import torch

from astrai_amd.extension import _mix
from astrai_amd.model import mixers


@pytest.fixture(autouse=True)
def any_shape(monkeypatch):
    monkeypatch.setattr(_mix, "few_rows_linear_supported", lambda *a, **k: True)


def _operands():
    return torch.randn(4, 16), torch.randn(8, 16), torch.randn(8)


@pytest.mark.parametrize("which", range(3))
def test_gradients_of_every_operand(which):
    ops = _operands()
    assert mixers.few_rows(*ops)
    ops[which].requires_grad_(True)
    assert not mixers.few_rows(*ops)
    with torch.no_grad():
        assert mixers.few_rows(*ops)
    out = mixers.linear(*ops)
    out.sum().backward()
    assert ops[which].grad is not None
