"""The sight pass of the summary on every board height up to 24 that the maps
have: where 64 lanes do not hold a whole number of board rows (12 rows, five
times over in 60 lanes), the partial rows of one height's lanes must not leak
into another row.  Hidden-information observations of env.step, its final
observation and of a fused rollout of few games, against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from nanorts_amd.content import map_name_to_scenario
from oracle.oracle import Oracle, batch_initial
from tests.helpers import roots, to_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["basesWorkers8x8", "FourBasesWorkers12x12", "EightBasesWorkers16x12",
                                  "basesWorkers16x16", "basesWorkers24x24A"])
def test_hidden_observations_match_oracle(name, oracle_threads):
    import torch

    import nanorts_amd

    print("sight rows", name, flush=True)
    game = map_name_to_scenario(name, max_cycles=110)
    L = 16
    oracle = Oracle(game)
    st = batch_initial(game, L, roots(L, 3))
    oracle.rollout(st, (1, 2), 0, 90, True, threads=oracle_threads, record=False)
    env = nanorts_amd.make("NanoRTS", scenario=game, partial_observability=True, device="cuda:0")
    dev = to_device(env, st)
    for t in range(24):
        actions = oracle.sample_actions(oracle.avail_rows(st), (3, 4), t)
        acts = {a: torch.as_tensor(np.ascontiguousarray(actions[:, i]), device="cuda:0")
                for i, a in enumerate(env.agents)}
        obs, dev, _, _, infos = env.step(None, dev, acts, donate=True)
        want = oracle.env_step(st, actions, True)
        for i, agent in enumerate(env.agents):
            np.testing.assert_array_equal(obs[agent].feature_maps.cpu().numpy(), want["feature_maps"][:, i],
                                          err_msg=f"{name} cycle {t}")
    got = env.rollout(dev, 40, (5, 9))
    want = oracle.rollout(st, (5, 9), 0, 40, True, threads=oracle_threads)
    np.testing.assert_array_equal(got["feature_maps"][0].cpu().numpy(), want["feature_maps"])
