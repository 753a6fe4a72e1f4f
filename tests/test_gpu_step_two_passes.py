"""env.step as two launches: a first pass with two games per wave on the slot
window, which says in the caller's work words which games it stepped, and the
full block for the others.  The launches are asked for with games that a test
can play on the oracle, and the work words show that both of them stepped
some."""
from __future__ import annotations

import numpy as np
import pytest

from nanorts_amd.content import map_name_to_scenario
from oracle.oracle import Oracle
from tests.helpers import assert_states_equal, roots, to_device, to_host
from tests.test_gpu_parity import _packed

pytestmark = pytest.mark.gpu

UNTOUCHED = -7  # a work word that no launch has written


def two_pass_step(env, state, actions, reset=True):
    """(state, outputs, work words) of env.step's launch from `state` into
    fresh buffers, with the work words here instead of the facade's own."""
    import torch

    from nanorts_amd import native

    L, b, d = state.num_envs, env.bucket, env.device
    acts = torch.stack([actions[a] for a in env.agents], dim=1).contiguous()
    maps = (L, 2, b.height, b.width, 6)
    shapes = {"reward": ((L, 2), torch.float32), "done": ((L,), torch.bool), "terminated": ((L,), torch.bool),
              "truncated": ((L,), torch.bool), "winner": ((L,), torch.int32), "spawn_overflowed": ((L,), torch.bool),
              "feature_maps": (maps, torch.uint8), "scalars": ((L, 2, 4), torch.int32),
              "final_feature_maps": (maps, torch.uint8), "final_scalars": ((L, 2, 4), torch.int32),
              "reward_components": ((L, 2, 6), torch.float32), "spawn_overflow": ((L, 2), torch.int32)}
    out = {name: torch.full(shape, 0x4D, dtype=torch.uint8, device=d).to(dtype) for name, (shape, dtype) in shapes.items()}
    taken = torch.full((L,), UNTOUCHED, dtype=torch.int32, device=d)
    nxt = state.successor()
    code = env.lib.nanorts_amd_env_step_from(
        torch.cuda.current_stream().cuda_stream, env.dev.ref, state.native(), nxt.native(), L, acts[:, 0].data_ptr(),
        acts[:, 1].data_ptr(), acts.stride(0), env.partial, int(reset),
        native.EnvResults(*[t.data_ptr() for t in out.values()]), taken.data_ptr())
    native.check(code, "nanorts_amd_env_step_from")
    return nxt, out, taken.cpu().numpy()


def crowded_start(game, L, seed=3):
    """Starting states in which every third game has 20 to 40 Workers of
    player 0: inside the first pass's 32 slots and 32 available units, at
    their bound and past it."""
    b = game.bucket
    own = _packed(game, [0])["birth"][0, b.neutral_capacity:b.neutral_capacity + b.per_player_capacity]
    counts = (20, 30, 31, 32, 33, 36, 40)
    extra = [counts[(l // 3) % len(counts)] - int((own != -1).sum()) if l % 3 == 0 else 0 for l in range(L)]
    return _packed(game, extra, seed=seed, alternate=False)


@pytest.mark.parametrize("name,strategy,partial", [
    ("basesWorkers8x8", "CANCEL_ALTERNATING", False), ("basesWorkers16x16", "CANCEL_ALTERNATING", True),
    ("basesWorkers16x16", "CANCEL_BOTH", False), ("letMeOut", "CANCEL_RANDOM", True),
    ("basesWorkers24x24A", "CANCEL_RANDOM", True), ("basesWorkers32x32A", "CANCEL_BOTH", True),
    ("GardenOfWar64x64", "CANCEL_RANDOM", True)])
def test_two_passes_match_oracle(name, strategy, partial, monkeypatch, oracle_threads):
    """Every output and the whole state of each step against the oracle, over
    the horizon (final observations, resets), with an odd number of games."""
    import torch

    import nanorts_amd

    print(f"two-pass env.step {name} {strategy} partial={partial}", flush=True)
    monkeypatch.setenv("NANORTS_AMD_FIRST_PASS", "pair")
    game = map_name_to_scenario(name, max_cycles=44, conflict_strategy=strategy)
    oracle, L = Oracle(game), 41
    st = crowded_start(game, L)
    assert (oracle.violations(st) == 0).all()
    oracle.rollout(st, (5, 6), 0, 20, partial, threads=oracle_threads, record=False)
    env = nanorts_amd.make("NanoRTS", scenario=game, partial_observability=partial, reward_components=True,
                           device="cuda:0")
    dev = to_device(env, st)
    seen, ends = set(), 0
    for t in range(28):
        rows = oracle.sample_actions(oracle.avail_rows(st), (7, 8), t)
        actions = {a: torch.as_tensor(np.ascontiguousarray(rows[:, p]), device="cuda:0") for p, a in enumerate(env.agents)}
        dev, got, taken = two_pass_step(env, dev, actions)
        want = oracle.env_step(st, rows, partial, final=True)
        assert_states_equal(st, to_host(dev), f"{name} cycle {t}")
        for field, w in want.items():
            g = got[field].cpu().numpy()
            np.testing.assert_array_equal(g, w.astype(g.dtype), err_msg=f"{field}, cycle {t}")
        seen |= set(taken.tolist())
        ends += int(want["done"].sum())
    assert seen == {0, 1} and ends > 0


@pytest.mark.parametrize("name", ["basesWorkers8x8", "basesWorkers16x16"])
@pytest.mark.parametrize("surface", ["symbolic", "pixels"])
def test_two_passes_match_one(name, surface, monkeypatch):
    """The facade's step and step_env (which keeps an ended game's state) with
    two launches against the one launch, donated and not, on both surfaces."""
    import torch

    import nanorts_amd
    from nanorts_amd import env as envmod
    from tests.test_gpu_step_buffers import _same

    print(f"two passes against one {name} {surface}", flush=True)
    game = map_name_to_scenario(name, max_cycles=30, conflict_strategy="CANCEL_ALTERNATING")
    env = nanorts_amd.make("NanoRTS", scenario=game, partial_observability=True, reward_components=True,
                           surface=surface, device="cuda:0")
    state = to_device(env, crowded_start(game, 33))
    env.rollout(state, 22, (5, 6), record=False)
    monkeypatch.setattr(envmod, "_FEW_GAMES", 0)
    seen, ends = set(), 0
    for t in range(12):
        actions = env.sample_actions(env.get_avail_actions(state, form="words"), (7, 8), t)
        step = env.step_env if t % 3 == 1 else env.step
        monkeypatch.setenv("NANORTS_AMD_FIRST_PASS", "lean")
        *_, taken = two_pass_step(env, state, actions, step == env.step)
        assert set(taken.tolist()) == {UNTOUCHED}
        want = step(None, state.clone(), actions, donate=True)
        monkeypatch.setenv("NANORTS_AMD_FIRST_PASS", "pair")
        *_, taken = two_pass_step(env, state, actions, step == env.step)
        seen |= set(taken.tolist())
        _same(want, step(None, state, actions))
        _same(want, step(None, state.clone(), actions, donate=True))
        ends += int(want[3]["__all__"].sum())
        state = want[1]
    assert seen == {0, 1} and ends > 0


@pytest.mark.parametrize("donate", [True, False])
def test_restart_replaces_every_slot(donate, monkeypatch):
    """A game that ends takes the whole initial state: also slots outside the
    first pass's window, whose leaves a program may have left other than the
    initial state has them (here five leaves of empty slots); a game that goes
    on keeps them."""
    import nanorts_amd
    from nanorts_amd import env as envmod
    from tests.test_gpu_step_buffers import _same

    print(f"restart of every slot donate={donate}", flush=True)
    game = map_name_to_scenario("basesWorkers16x16", max_cycles=44)
    b = game.bucket
    env = nanorts_amd.make("NanoRTS", scenario=game, device="cuda:0")
    _, state = env.reset(envmod.env_roots(3, 9))
    env.rollout(state, 36, (5, 6), record=False)
    state.core_state.leaves["time"][:4] = 43  # their next step is the horizon's
    for name in ("hit_points", "carried_resources", "unit_type", "cell", "pending_issued_at"):
        for first in (b.neutral_capacity + 40, b.neutral_capacity + b.per_player_capacity + 40):
            state.core_state.leaves[name][:, first:first + 20] = 3
    monkeypatch.setattr(envmod, "_FEW_GAMES", 0)
    actions = env.sample_actions(env.get_avail_actions(state, form="words"), (7, 8), 0)
    monkeypatch.setenv("NANORTS_AMD_FIRST_PASS", "lean")
    want = env.step(None, state.clone(), actions, donate=donate)
    monkeypatch.setenv("NANORTS_AMD_FIRST_PASS", "pair")
    *_, taken = two_pass_step(env, state, actions)
    assert set(taken.tolist()) == {1}
    got = env.step(None, state.clone(), actions, donate=donate)
    assert want[3]["__all__"].tolist() == [True] * 4 + [False] * 5
    hp = want[1].core_state.leaves["hit_points"][:, b.neutral_capacity + 40]
    assert hp.tolist() == [0] * 4 + [3] * 5
    _same(want, got)


# games per compute unit on either side of the line between one launch and two
# (None: one launch however many)
@pytest.mark.parametrize("name,one,two", [
    ("basesWorkers8x8", 46, 50), ("basesWorkers16x16", 30, 34), ("basesWorkers12x12", 13, 15),
    ("basesWorkers32x32A", 8, 11), ("TwoBasesBarracks16x16", 16, 18), ("SixBasesWorkers12x12", 66, None),
    ("FourBasesWorkers12x12", 60, 66),
    ("GardenOfWar64x64", 8, None)])
def test_launches_by_board_and_games(name, one, two, monkeypatch):
    """env.step of few games is one launch and of many two, by the board: the
    work words are left alone in the one and written in the other."""
    import torch

    import nanorts_amd
    from nanorts_amd import env as envmod

    monkeypatch.delenv("NANORTS_AMD_FIRST_PASS", raising=False)
    env = nanorts_amd.make("NanoRTS", scenario=map_name_to_scenario(name), device="cuda:0", final_observation=True)
    units = torch.cuda.get_device_properties(0).multi_processor_count
    for games in (one, two):
        if games is None:
            continue
        print(f"launches {name} {games} games a unit", flush=True)
        _, state = env.reset(envmod.env_roots(3, games * units))
        actions = env.sample_actions(env.get_avail_actions(state, form="words"), (7, 8), 0)
        *_, taken = two_pass_step(env, state, actions)
        assert set(taken.tolist()) == ({UNTOUCHED} if games == one else {1})
