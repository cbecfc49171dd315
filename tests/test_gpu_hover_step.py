"""The hover environment's one-launch step at the edges of its 64-env tiles,
with short episodes (many resets in one tile at once), and its five-launch
path (articulated contacts on; the hover worlds have no joints, so nothing
else changes), against the oracle bit for bit."""
import numpy as np
import pytest

from b3test import hover_actions, hover_cpu_run, oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,horizon,dt,options", [(1, 256, 1.0 / 60.0, 0), (63, 7, 1.0 / 60.0, 0), (64, 1, 1.0 / 60.0, 0),
                                                  (130, 5, 1.0 / 30.0, 1), (65, 6, 0.0, 0), (130, 5, 1.0 / 60.0, 2)])
def test_step_edges(n, horizon, dt, options):
    from puffysics_amd import _native
    from puffysics_amd.hover import B3HoverConfig, HoverEnvs
    steps = 60
    actions = hover_actions(n, steps, seed=n)
    want = hover_cpu_run(oracle(), "ohover", n, actions, seed=3, config=(2.0, 10.0, dt, 4, horizon))
    envs = HoverEnvs(n, seed=3, config=B3HoverConfig(2.0, 10.0, dt, 4, horizon))
    assert _native.engine_lib().b3_engine_set_options(envs.engine_handle(), options) == 0
    envs.reset()
    got = [[envs.observations.cpu().numpy()], [envs.rewards.cpu().numpy()], [envs.terminals.cpu().numpy()]]
    for t in range(steps):
        envs.actions.copy_(torch.from_numpy(actions[t]))
        envs.step()
        for k, x in enumerate((envs.observations, envs.rewards, envs.terminals)):
            got[k].append(x.cpu().numpy())
    log = envs.log()
    envs.close()
    for k in range(3):
        assert np.array_equal(np.stack(got[k]).view(np.uint32), want[k].view(np.uint32))
    assert np.array_equal(np.array(list(log.values()), np.float32), want[3])
    assert want[2].sum() > 0 or horizon > steps
