"""Which steps a rollout takes its RunningNorm partial sums from (GpuDogfightVecEnv.norm_fuse_pays),
asked of the library with stand-in environments: no GPU call."""
from types import SimpleNamespace

import pytest

from conftest import import_pkg


def _pays(nenv, **kw):
    env = SimpleNamespace(nenv=nenv, OBS_SIZE=184, fused_step=True, fused_finite=True, substeps=6,
                          step_roles=4, obr=SimpleNamespace(_lib=import_pkg("_lib").lib()))
    for k, v in kw.items():
        setattr(env, k, v)
    return import_pkg("rl_env").GpuDogfightVecEnv.norm_fuse_pays(env)


@pytest.mark.parametrize("other", [{"step_roles": 2}, {"fused_step": False},
                                   {"fused_finite": False}, {"substeps": 0}])
def test_norm_partials_pay_wherever_the_step_has_128_aircraft_workgroups(other):
    """Only the four-role one-launch step has a 64-aircraft form to keep; the two-role step and the
    two launches form the partials in any batch, as they did before that form existed."""
    for nenv in (1, 200, 8192, 8193, 16384):
        assert _pays(nenv, **other), (nenv, other)


def test_norm_partials_of_the_four_role_step():
    """The four-role step keeps its 64-aircraft workgroups while each has a compute unit (8,192
    engagements on 256)."""
    assert [_pays(n) for n in (1, 777, 8192, 8193, 16384)] == [False, False, False, True, True]
