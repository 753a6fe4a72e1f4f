"""Boards whose width is not a multiple of 4: the summary's observation groups
of four cells span two rows there, or there is no summary where the cells are
no multiple of 4 (15x14).  Every observation, mask, fused rollout and
seat rollout against the oracle, bit for bit, with and without hidden
information; walls, both orders of an observation's rows and units on every
column come with the boards' random play."""
from __future__ import annotations

import numpy as np
import pytest

from nanorts_amd.content import map_name_to_scenario
from nanorts_amd.model import UnitTypeTableVersion
from oracle.oracle import Oracle, batch_initial, empty_carry
from tests.helpers import assert_states_equal, roots, to_device, to_host

pytestmark = pytest.mark.gpu

BOARDS = ("NoWhereToRun9x8", "basesWorkers10x10", "itsNotSafe", "melee14x12Mixed18")


def _env(game, partial, **kw):
    import nanorts_amd

    return nanorts_amd.make("NanoRTS", scenario=game, partial_observability=partial, device="cuda:0", **kw)


@pytest.mark.parametrize("partial", [False, True])
@pytest.mark.parametrize("name", BOARDS)
def test_steps_and_rollouts_match_oracle(name, partial, oracle_threads):
    import torch

    print("odd width", name, partial, flush=True)
    game = map_name_to_scenario(name, utt=UnitTypeTableVersion.ORIGINAL, conflict_strategy="CANCEL_RANDOM",
                                max_cycles=150)
    L = 37
    oracle = Oracle(game)
    st = batch_initial(game, L, roots(L, 3))
    oracle.rollout(st, (1, 2), 0, 110, partial, threads=oracle_threads, record=False)
    env = _env(game, partial)
    dev = to_device(env, st)
    for t in range(60):  # over the horizon: final observations and resets
        rows = oracle.avail_rows(st)
        masks = env.get_avail_actions(dev)
        np.testing.assert_array_equal(torch.stack([masks[a] for a in env.agents], 1).cpu().numpy().astype(np.uint8),
                                      rows.reshape(L, 2, -1, rows.shape[-1]).astype(np.uint8))
        actions = oracle.sample_actions(rows, (3, 4), t)
        acts = {a: torch.as_tensor(np.ascontiguousarray(actions[:, i]), device="cuda:0")
                for i, a in enumerate(env.agents)}
        obs, dev, rewards, dones, infos = env.step(None, dev, acts)
        want = oracle.env_step(st, actions, partial)
        for i, agent in enumerate(env.agents):
            np.testing.assert_array_equal(obs[agent].feature_maps.cpu().numpy(), want["feature_maps"][:, i])
            np.testing.assert_array_equal(obs[agent].scalars.cpu().numpy(), want["scalars"][:, i])
        assert_states_equal(st, to_host(dev), f"{name} cycle {t}")
    got = env.rollout(dev, 200, (5, 9), record_actions=True)
    want = oracle.rollout(st, (5, 9), 0, 200, partial, threads=oracle_threads, record_actions=True)
    for field in ("actions", "rewards", "dones"):
        np.testing.assert_array_equal(got[field].cpu().numpy(), want[field].astype(got[field].cpu().numpy().dtype))
    np.testing.assert_array_equal(got["feature_maps"][0].cpu().numpy(), want["feature_maps"])
    np.testing.assert_array_equal(got["scalars"][0].cpu().numpy(), want["scalars"])
    assert_states_equal(st, to_host(dev), f"{name} rollout")


@pytest.mark.parametrize("partial", [False, True])
@pytest.mark.parametrize("name", BOARDS[:3])
def test_seat_rollouts_match_oracle(name, partial):
    import torch

    from nanorts_amd import bots

    print("odd width seat", name, partial, flush=True)
    game = map_name_to_scenario(name, conflict_strategy="CANCEL_ALTERNATING", max_cycles=250)
    o = Oracle(game)
    L, C, steps, key = 17, game.bucket.per_player_capacity, 300, (41, 43)
    st = batch_initial(game, L, roots(L, 13))
    carry = empty_carry(L, C)
    seat = bots.SeatEnv(bots.lightRushAI, scenario=game, partial_observability=partial)
    device_carry = {k: torch.as_tensor(np.ascontiguousarray(v), device="cuda:0") for k, v in carry.items()}
    device_carry["trained"] = device_carry["trained"].to(torch.bool)
    state = bots.SeatState(to_device(seat.env, st), device_carry, torch.zeros(L, dtype=torch.int32, device="cuda:0"))
    got = seat.rollout(state, steps, key, record_actions=True)
    rewards, dones, actions = (got[k].cpu().numpy() for k in ("rewards", "dones", "actions"))
    for t in range(steps):
        want_actions = np.ascontiguousarray(o.sample_actions(o.avail_rows(st), key, t)[:, 0])
        np.testing.assert_array_equal(actions[t], want_actions, err_msg=f"actions at cycle {t}")
        want = o.seat_step(st, carry, 1, 4, 0, want_actions, partial, observe=t == steps - 1)
        np.testing.assert_array_equal(rewards[t], want["reward"], err_msg=f"cycle {t}")
        np.testing.assert_array_equal(dones[t], want["done"].astype(bool), err_msg=f"cycle {t}")
    assert_states_equal(st, to_host(state.environment_state), f"{name} seat final state")
    np.testing.assert_array_equal(got["feature_maps"][0].cpu().numpy(), want["feature_maps"])
    np.testing.assert_array_equal(got["scalars"][0].cpu().numpy(), want["scalars"])
