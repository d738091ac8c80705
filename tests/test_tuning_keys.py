"""The FP64 configurations of large work (phpc_set_tuning keys 0, 3, 4, 5): every configuration can
be chosen and the defaults restored, and plans follow keys 0 and 3."""
import pytest

from conftest import phpc

DEFAULTS = {0: 16, 3: 11, 4: 11, 5: 16}


@pytest.fixture
def restore(lib):
    yield
    for key, value in DEFAULTS.items():
        phpc.set_tuning(key, value)


@pytest.mark.parametrize("key", [0, 3])
def test_every_configuration_and_the_default(lib, restore, key):
    n = lib.phpc_num_configs()
    for value in list(range(n)) + [DEFAULTS[key]]:
        assert lib.phpc_set_tuning(key, value) == phpc.PHPC_OK, value
    for value in (-1, n):
        assert lib.phpc_set_tuning(key, value) == phpc.PHPC_ERR_ARG


def planned(panel):
    import torch
    n = 6144
    A = torch.zeros(n, n, dtype=torch.float64, device="cuda")
    C = torch.zeros_like(A)
    plan = phpc.Plan(phpc.F64, [(A, A, C, panel)])
    plan.launch()
    torch.cuda.synchronize()
    config = plan.info()["config"]
    plan.close()
    return config


@pytest.mark.gpu
def test_plans_follow_and_return(restore):
    assert planned(0) == 11 and planned(256) == 16
    phpc.set_tuning(3, 14)
    phpc.set_tuning(0, 12)
    assert planned(0) == 14 and planned(256) == 12
    phpc.set_tuning(0, 4)  # no panel-grouped variants
    assert planned(256) == 16
    phpc.set_tuning(3, 11)
    assert planned(0) == 11
