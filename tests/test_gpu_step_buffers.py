"""A step that is not given its input state's buffers: the launch reads one
state and writes another.  Each step surface is compared with itself on a
donated copy (which the other tests compare with the oracle), bit for bit,
and the input state must stay as it was.  The boards cover both row copies
(whole vectors and by granule), the summary's observation and the general one
(15x14) and a state with a strided leaf, which is copied first.  Horizons are short, so games end and
reset inside the steps."""
from __future__ import annotations

import dataclasses
import sys

import pytest

from nanorts_amd.content import map_name_to_scenario

pytestmark = pytest.mark.gpu

# map, games (odd counts leave the last workgroup short)
BOARDS = (("basesWorkers8x8", 65), ("NoWhereToRun9x8", 33), ("itsNotSafe", 33), ("basesWorkers16x16", 66),
          ("basesWorkers24x24A", 5))


def _say(*parts):
    print(*parts, flush=True)
    sys.stdout.flush()


def _tensors(value, path="out"):
    import torch

    if isinstance(value, torch.Tensor):
        yield path, value
    elif dataclasses.is_dataclass(value):
        for f in dataclasses.fields(value):
            yield from _tensors(getattr(value, f.name), f"{path}.{f.name}")
    elif isinstance(value, dict):
        for k, v in value.items():
            yield from _tensors(v, f"{path}.{k}")
    elif isinstance(value, (list, tuple)):
        for i, v in enumerate(value):
            yield from _tensors(v, f"{path}[{i}]")


def _same(want, got):
    import torch

    want, got = dict(_tensors(want)), dict(_tensors(got))
    assert want.keys() == got.keys()
    for path, w in want.items():
        assert torch.equal(w, got[path]), path


def _poison():
    """Freed memory that is not zero, for the next allocations."""
    import torch

    for size in (1 << 12, 1 << 16, 1 << 20, 1 << 22):
        held = [torch.full((size,), 0x5A, dtype=torch.uint8, device="cuda:0") for _ in range(40)]
        del held


def _compare(state, step, donated):
    """step(state) against donated(a clone), with the input kept."""
    before = state.clone()
    _poison()
    got = step(state)
    want = donated(before.clone())
    _same(before, state)
    _same(want, got)
    return want


@pytest.mark.parametrize("name,L", BOARDS)
@pytest.mark.parametrize("strided", [False, True])
def test_env_step_writes_fresh_buffers(name, L, strided):
    import torch

    import nanorts_amd
    from nanorts_amd import env as envmod

    _say(f"env.step into fresh buffers {name} strided={strided}")
    game = map_name_to_scenario(name, max_cycles=36, conflict_strategy="CANCEL_ALTERNATING")
    env = nanorts_amd.make("NanoRTS", scenario=game, partial_observability=True, reward_components=True,
                           device="cuda:0")
    _, state = env.reset(envmod.env_roots(3, L))
    env.rollout(state, 30, (5, 6), record=False)
    ends = 0
    for t in range(8):
        actions = env.sample_actions(env.get_avail_actions(state, form="words"), (7, 8), t)
        if strided:
            wide = torch.stack([state.core_state.leaves["carried_resources"]] * 2, dim=-1)
            state.core_state.leaves["carried_resources"] = wide[..., 0]
        fused = env.step if t % 3 else env.step_env
        want = _compare(state, lambda s: fused(None, s, actions), lambda s: fused(None, s, actions, donate=True))
        state = want[1]
        ends += int(want[3]["__all__"].sum())
    assert ends > 0


@pytest.mark.parametrize("name,L", BOARDS)
def test_env_step_reads_actions_where_they_lie(name, L):
    """One result for every form of the same action rows: views of one tensor,
    a block an agent, rows inside a wider tensor, one row of every game
    (stride 0), rows that are not dense and host arrays."""
    import torch

    import nanorts_amd
    from nanorts_amd import env as envmod

    _say(f"action rows {name}")
    game = map_name_to_scenario(name, max_cycles=40, conflict_strategy="CANCEL_RANDOM")
    env = nanorts_amd.make("NanoRTS", scenario=game, device="cuda:0")
    _, state = env.reset(envmod.env_roots(3, L))
    env.rollout(state, 31, (5, 6), record=False)
    drawn = env.sample_actions(env.get_avail_actions(state, form="words"), (7, 8), 0)
    stacked = torch.stack([drawn[a] for a in env.agents], dim=1)
    want = env.step(None, state, {a: stacked[:, p] for p, a in enumerate(env.agents)})
    blocks = {a: v.clone() for a, v in drawn.items()}
    wide = {a: torch.cat([v, v + 1], dim=1)[:, :v.shape[1]] for a, v in drawn.items()}
    loose = {a: torch.stack([v, v], dim=-1)[..., 0] for a, v in drawn.items()}
    mixed = {env.agents[0]: blocks[env.agents[0]], env.agents[1]: wide[env.agents[1]]}
    host = {a: v.cpu().numpy() for a, v in drawn.items()}
    for actions in (blocks, wide, loose, mixed, host):
        _same(want, env.step(None, state, actions))
    first = {a: v[:1] for a, v in drawn.items()}
    same_everywhere = {a: v.repeat(L, 1, 1) for a, v in first.items()}
    expanded = {a: v.expand(L, -1, -1) for a, v in first.items()}
    _same(env.step(None, state, same_everywhere), env.step(None, state, expanded))


@pytest.mark.parametrize("name,L,partial", [("basesWorkers8x8", 12803, False), ("basesWorkers16x16", 8707, True),
                                            ("basesWorkers32x32A", 4098, True)])
def test_env_step_of_many_games_in_two_passes(name, L, partial, monkeypatch):
    """More games than one pass takes: the launch of two games per wave and the
    one for the games it leaves, against the one-pass launch on the same
    states.  Some games start crowded (more than 32 units of a player, past
    the slot window; one at the bound), the horizon ends games inside the
    steps, odd counts leave half a wave empty, and the input's buffers are
    donated or not."""
    import torch

    import nanorts_amd
    from nanorts_amd import env as envmod
    from tests.helpers import to_device
    from tests.test_gpu_parity import _packed
    from tests.test_gpu_step_two_passes import two_pass_step

    _say(f"two-pass env.step {name}")
    game = map_name_to_scenario(name, max_cycles=44, conflict_strategy="CANCEL_RANDOM")
    env = nanorts_amd.make("NanoRTS", scenario=game, partial_observability=partial, reward_components=True,
                           device="cuda:0")
    base = int((_packed(game, [0])["birth"][0] != -1).sum())
    crowd = to_device(env, _packed(game, [n - base for n in (20, 30, 34, 35, 36, 37, 40)], alternate=False))
    _, state = env.reset(envmod.env_roots(3, L))
    for k, v in crowd.core_state.leaves.items():
        state.core_state.leaves[k][:7] = v
        state.core_state.leaves[k][-3:] = v[-3:]
    env.rollout(state, 36, (5, 6), record=False)
    seen, ends = set(), 0
    for t in range(12):
        actions = env.sample_actions(env.get_avail_actions(state, form="words"), (7, 8), t)
        *_, taken = two_pass_step(env, state, actions)
        seen |= set(taken.tolist())
        with monkeypatch.context() as m:
            m.setattr(envmod, "_FEW_GAMES", 1 << 40)
            want = env.step(None, state.clone(), actions, donate=True)
        before = state.clone()
        _poison()
        _same(want, env.step(None, state, actions))
        _same(before, state)
        _same(want, env.step(None, state, actions, donate=True))
        ends += int(want[3]["__all__"].sum())
    assert seen == {0, 1} and ends > 0  # both launches stepped games


@pytest.mark.parametrize("name,L", BOARDS[:4])
@pytest.mark.parametrize("rule", ["player_1", "drawn"])
def test_seat_step_writes_fresh_buffers(name, L, rule):
    import torch

    from nanorts_amd import bots
    from nanorts_amd import env as envmod

    _say(f"seat step into fresh buffers {name} {rule}")
    game = map_name_to_scenario(name, max_cycles=36)
    seat = bots.SeatEnv(bots.workerRushAI, scenario=game, seat=rule, device="cuda:0")
    _, state = seat.reset(envmod.env_roots(4, L))
    seat.rollout(state, 30, (5, 6), record=False)
    ends = 0
    for t in range(8):
        words = seat.env.get_avail_actions(state.environment_state, form="words")
        drawn = seat.env.sample_actions(words, (9, 9), t)
        acts = {bots.LEARNER: torch.where(state.seat.reshape(-1, 1, 1) == 0, drawn["player_0"], drawn["player_1"])}
        want = _compare(state, lambda s: seat.step(None, s, acts), lambda s: seat.step(None, s, acts, donate=True))
        state = want[1]
        ends += int(want[3]["__all__"].sum())
    assert ends > 0


@pytest.mark.parametrize("name,L", BOARDS)
def test_gridnet_step_writes_fresh_buffers(name, L):
    from nanorts_amd import env as envmod
    from nanorts_amd import gridnet

    _say(f"GridNet step into fresh buffers {name}")
    game = map_name_to_scenario(name, max_cycles=6, conflict_strategy="CANCEL_RANDOM")
    grid = gridnet.GridNet(game, gridnet.prepare(game, mask_form="packed"), device="cuda:0")
    state, obs = grid.reset(envmod.env_roots(5, L))
    mask, ends = obs.action_mask, 0
    for t in range(9):
        actions = grid.sample_actions(mask, (1, 2), t)
        if t % 2:
            commands = grid.decode_actions(actions, state)
            first = actions[:, 0].contiguous()
            want = _compare(state, lambda s: grid.step_against(s, first, commands),
                            lambda s: grid.step_against(s, first, commands, donate=True))
        else:
            want = _compare(state, lambda s: grid.step(s, actions), lambda s: grid.step(s, actions, donate=True))
        state, mask = want.environment_state, want.observation.action_mask
        ends += int(want.done.sum())
    assert ends > 0


def test_step_from_entries_refuse_bad_arguments():
    """Nothing is launched for a missing leaf of either state."""
    import ctypes

    from nanorts_amd import native

    lib = native.load()
    buf = (ctypes.c_uint8 * 64)()
    addr = ctypes.cast(buf, ctypes.c_void_p)
    whole = native.State(*[addr] * len(native.STATE_FIELDS))
    rootless = native.State(*[addr] * (len(native.STATE_FIELDS) - 2), None, None)
    game = map_name_to_scenario("basesWorkers8x8")
    from nanorts_amd.env import DeviceGame
    import torch

    dev = DeviceGame(game, torch.device("cuda:0"))
    for first, second in ((native.State(), whole), (whole, native.State()), (rootless, whole), (whole, rootless)):
        assert lib.nanorts_amd_env_step_from(None, dev.ref, first, second, 1, addr, addr, 1, 0, 1, native.EnvResults(), None) == 1
        assert lib.nanorts_amd_gridnet_step_from(None, dev.ref, first, second, 1, addr, None,
                                                 native.GridNetResults()) == 1
    carry = native.AbstractActions(*[addr] * len(native.ABSTRACT_FIELDS))
    code = lib.nanorts_amd_seat_step_from(None, dev.ref, whole, whole, 1, 0, 4, 0, addr, None, 1, carry, carry, addr, 0,
                                          native.EnvResults())
    assert code == 1 and "seats" in lib.nanorts_amd_last_error().decode()


@pytest.mark.parametrize("name,L", BOARDS[:3])
def test_in_place_entries_match_the_from_entries(name, L):
    """The C entries that step a state in place (the facades call the ones with
    a state of their own to write) on stacked action rows of both agents:
    outputs and state as the facades' steps have them."""
    import torch

    import nanorts_amd
    from nanorts_amd import bots, gridnet, native
    from nanorts_amd import env as envmod

    _say(f"in-place entries {name}")
    lib, stream = native.load(), torch.cuda.current_stream().cuda_stream
    game = map_name_to_scenario(name, max_cycles=34, conflict_strategy="CANCEL_ALTERNATING")
    env = nanorts_amd.make("NanoRTS", scenario=game, partial_observability=True, reward_components=True,
                           device="cuda:0")
    b = env.bucket
    _, state = env.reset(envmod.env_roots(3, L))
    env.rollout(state, 30, (5, 6), record=False)

    def buffers(final):
        _poison()
        maps, flags = (L, 2, b.height, b.width, 6), {"dtype": torch.bool, "device": "cuda:0"}
        out = {"reward": torch.empty((L, 2), device="cuda:0"), "done": torch.empty(L, **flags),
               "terminated": torch.empty(L, **flags), "truncated": torch.empty(L, **flags),
               "winner": torch.empty(L, dtype=torch.int32, device="cuda:0"),
               "spawn_overflowed": torch.empty(L, **flags), "maps": torch.empty(maps, dtype=torch.uint8, device="cuda:0"),
               "scalars": torch.empty((L, 2, 4), dtype=torch.int32, device="cuda:0"), "final_maps": None,
               "final_scalars": None, "components": None, "spawn_overflow": None}
        if final:
            out["final_maps"], out["final_scalars"] = torch.empty_like(out["maps"]), torch.empty_like(out["scalars"])
        return out, native.EnvResults(*[None if t is None else t.data_ptr() for t in out.values()])

    def check(got, nxt, want, agents=None):
        obs, state_, rewards, dones, infos = want
        _same(state_, nxt)
        assert torch.equal(got["done"], dones["__all__"])
        for name_ in ("terminated", "truncated", "winner", "spawn_overflowed"):
            assert torch.equal(got[name_], infos[name_]), name_
        for p, agent in enumerate(agents or ()):
            assert torch.equal(got["reward"][:, p], rewards[agent])
            assert torch.equal(got["maps"][:, p], obs[agent].feature_maps)
            assert torch.equal(got["scalars"][:, p], obs[agent].scalars)
            if got["final_maps"] is not None:
                assert torch.equal(got["final_maps"][:, p], infos["final_observation"][agent].feature_maps)

    seat = bots.SeatEnv(bots.workerRushAI, scenario=game, seat="drawn", device="cuda:0")
    _, sst = seat.reset(envmod.env_roots(4, L))
    seat.rollout(sst, 30, (5, 6), record=False)
    grid = gridnet.GridNet(game, gridnet.prepare(game, mask_form="packed"), device="cuda:0")
    ends = 0
    for t in range(8):
        words = env.get_avail_actions(state, form="words")
        actions = env.sample_actions(words, (7, 8), t)
        rows = torch.stack([actions[a] for a in env.agents], dim=1).contiguous()
        for entry, step, final in ((lib.nanorts_amd_env_transition, env.step_env, False),
                                   (lib.nanorts_amd_env_step, env.step, True)):
            want, nxt = step(None, state, actions), state.clone()
            got, results = buffers(final)
            native.check(entry(stream, env.dev.ref, nxt.native(), L, rows.data_ptr(), env.partial, results), "in place")
            check(got, nxt, want, env.agents)
        ends += int(want[3]["__all__"].sum())
        state = want[1]

        learner = {bots.LEARNER: torch.where(sst.seat.reshape(-1, 1, 1) == 0, *[actions[a] for a in env.agents]).contiguous()}
        want, nxt = seat.step(None, sst, learner), sst.clone()
        got, results = buffers(False)
        es = nxt.environment_state
        native.check(lib.nanorts_amd_seat_step_lanes(
            stream, seat.env.dev.ref, es.native(), L, seat.bot.strategy, seat.bot.trained, nxt.seat.data_ptr(), 1,
            bots._carry_struct(nxt.carry), learner[bots.LEARNER].data_ptr(), seat.env.partial, results), "seat in place")
        check(got, nxt, want)
        nxt = sst.clone()
        nxt.seat[:] = 1
        fixed, results = buffers(False)
        native.check(lib.nanorts_amd_seat_step(
            stream, seat.env.dev.ref, nxt.environment_state.native(), L, seat.bot.strategy, seat.bot.trained, 1,
            bots._carry_struct(nxt.carry), learner[bots.LEARNER].data_ptr(), seat.env.partial, results), "seat in place")
        second = (sst.seat == 1).nonzero().reshape(-1)
        for field in ("reward", "done", "winner", "maps", "scalars"):
            assert torch.equal(fixed[field][second], got[field][second]), field
        sst = want[1]

        cells = grid.sample_actions(grid.observe(state).action_mask, (1, 2), t)
        commands = grid.decode_actions(cells, state)
        first = cells[:, 0].contiguous()
        for entry, step, drawn, extra in (
                (lib.nanorts_amd_gridnet_step, lambda s: grid.step(s, cells), cells, ()),
                (lib.nanorts_amd_gridnet_step_against, lambda s: grid.step_against(s, first, commands), first,
                 (native.Commands(*[commands[f].data_ptr() for f, _ in native.Commands._fields_]),))):
            want, nxt = step(state), state.clone()
            done = torch.empty(L, dtype=torch.bool, device="cuda:0")
            comps = torch.empty_like(want.reward_components)
            results = native.GridNetResults(comps.data_ptr(), None, None, None, done.data_ptr())
            native.check(entry(stream, grid.dev.ref, nxt.native(), L, drawn.data_ptr(), *extra, results), "grid in place")
            _same(want.environment_state, nxt)
            assert torch.equal(done, want.done) and torch.equal(comps, want.reward_components)
    assert ends > 0
