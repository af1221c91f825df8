"""The kernels that pack decal slots and screen flashes against the Torch expressions on the same device (which tensors that are not laid
out as the kernels read them still take): equal bit for bit."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def spread(tensor: torch.Tensor) -> torch.Tensor:
    """The same values, every second place of a wider tensor."""

    return torch.stack((tensor, tensor), dim=-1)[..., 0]


@pytest.mark.parametrize("slots", [1, 63, 64, 65, 130])
def test_decal_slots_are_packed_as_the_torch_expressions_pack_them(slots):
    from gradoom_amd import overlay_inputs

    rng = torch.Generator(device="cuda:0").manual_seed(slots)
    lanes, linedefs = 37, 4096
    whole = lambda low, high: torch.randint(low, high, (lanes, slots), generator=rng, device="cuda:0")  # noqa: E731
    real = lambda *shape: torch.randn(shape, generator=rng, device="cuda:0")  # noqa: E731
    serial = whole(-20, 40)                                    # free slots, and impacts of one number
    serial[0] = -1
    serial[1] = whole(0, 200)[0] + (1 << 31) - 100         # numbers on both sides of a free slot's place in the order
    wall, style = whole(-2, linedefs + 2), whole(-25, 60)
    walls = torch.round(real(linedefs, 4) * 300)
    walls[:64, 2:] = walls[:64, :2]                            # no direction at all
    walls[64:128, 2] = walls[64:128, 0]                        # along the axes
    walls[128:192, 3] = walls[128:192, 1]
    walls[192:1024] = real(832, 4)
    along, impact = real(lanes, slots), real(lanes, slots)
    table = torch.as_tensor(overlay_inputs.fine_sine_fixed(), device="cuda:0")
    state, geometry = overlay_inputs.decal_inputs(serial, wall, along, impact, style, walls, table)
    expected_state, expected_geometry = overlay_inputs.decal_inputs(spread(serial), wall, along, impact, style, walls, table)
    assert state.dtype == torch.int32 and torch.equal(state, expected_state)
    assert geometry.dtype == torch.float32 and torch.equal(geometry.view(torch.int32), expected_geometry.view(torch.int32))


def test_every_direction_takes_the_torch_expressions_place_in_the_fine_table():
    from gradoom_amd import overlay_inputs

    count = 1 << 18
    turn = torch.arange(count, dtype=torch.float64, device="cuda:0") * (2.0 * torch.pi / count)
    walls = torch.zeros((count, 4), dtype=torch.float32, device="cuda:0")
    walls[:, 2], walls[:, 3] = torch.cos(turn).to(torch.float32) * 1000, torch.sin(turn).to(torch.float32) * 1000
    wall = torch.arange(count, device="cuda:0").reshape(-1, 64)
    ones = torch.ones_like(wall, dtype=torch.float32)
    table = torch.as_tensor(overlay_inputs.fine_sine_fixed(), device="cuda:0")
    for style in (torch.zeros_like(wall), torch.full_like(wall, 20)):
        packed = overlay_inputs.decal_inputs(wall, wall, ones, ones, style, walls, table)
        expected = overlay_inputs.decal_inputs(spread(wall), wall, ones, ones, style, walls, table)
        assert torch.equal(packed[0], expected[0]) and torch.equal(packed[1], expected[1])


@pytest.mark.parametrize("lanes", [1, 256, 257])
def test_screen_flashes_are_packed_as_the_torch_expressions_pack_them(lanes):
    from gradoom_amd import overlay_inputs

    rng = torch.Generator(device="cuda:0").manual_seed(lanes)
    bonus = torch.randint(-3, 300, (lanes,), generator=rng, device="cuda:0")
    damage = torch.randint(-3, 200, (lanes,), generator=rng, device="cuda:0")
    alphas = torch.rand((114,), generator=rng, device="cuda:0") * 200
    assert torch.equal(overlay_inputs.screen_blend(bonus, damage, alphas), overlay_inputs.screen_blend(spread(bonus), damage, alphas))


@pytest.mark.parametrize("shape", [(114, 1), (1, 114), (2, 114)])
def test_a_table_of_alphas_with_two_dimensions_is_refused_as_the_torch_expressions_refuse_it(shape):
    from gradoom_amd import overlay_inputs

    bonus = torch.arange(5, device="cuda:0")
    damage = torch.arange(5, device="cuda:0").clamp(max=shape[0] - 1)      # every index the expressions take lies in the table
    alphas = torch.ones(shape, device="cuda:0")
    for counters in ((bonus, damage), (bonus.cpu(), damage.cpu())):
        with pytest.raises(RuntimeError, match="stack expects each tensor to be equal size"):
            overlay_inputs.screen_blend(*counters, alphas.to(counters[0].device))


def test_screen_flashes_of_other_shapes_are_packed_as_on_the_host():
    from gradoom_amd import overlay_inputs

    bonus, damage, alphas = torch.arange(6) * 5, torch.arange(6) * 40 - 20, torch.arange(200, dtype=torch.float32)
    for counters in ((bonus, damage, alphas), (bonus[:, None], damage, alphas[:, None]), (bonus[:, None], damage[:, None], alphas), (bonus[:0], damage[:0], alphas)):
        packed = overlay_inputs.screen_blend(*(t.to("cuda:0") for t in counters))
        expected = overlay_inputs.screen_blend(*counters)
        # the device multiplies with the divisor's reciprocal: two roundings of 2^-24 where the host's division has one
        assert packed.shape == expected.shape and torch.allclose(packed.cpu(), expected, rtol=2.0**-22, atol=0)


@pytest.mark.parametrize("lanes", [1, 33, 257])
@pytest.mark.parametrize("form", ["plain", "wide tables", "two starts"])
def test_actors_face_the_camera_as_the_torch_expressions_have_them(lanes, form):
    """The kernel's own rotations against Torch's, which tensors that are not laid out as it reads them still take: every octant, actors on
    the camera, along the axes, and values that are no numbers."""
    from conftest import load_fixture
    from test_actor_inputs import stored_engine

    from gradoom_amd import actor_inputs

    engine = stored_engine(load_fixture("actors")[1])
    rng = torch.Generator(device="cuda:0").manual_seed(lanes)
    per_map = ("_enemy_walk_frame_tics", "_enemy_idle_frame_tics", "_enemy_attack_recovery", "_player_start_z", "_item_z")
    for field in actor_inputs.ENGINE_FIELDS:
        value = getattr(engine, field)
        if field not in per_map:
            value = value[torch.arange(lanes) % value.shape[0]]
        setattr(engine, field, value.to("cuda:0"))
    m = engine.map
    for field in actor_inputs.MAP_FIELDS:
        setattr(m, field, getattr(m, field).to("cuda:0"))
    for kind, first, second in (("enemy", "x", "y"), ("projectile", "velocity_x", "velocity_y"), ("enemy_projectile", "x", "y"), ("enemy_projectile", "velocity_x", "velocity_y")):
        for name, other in ((first, second), (second, first)):
            values = getattr(engine, f"{kind}_{name}")
            values.copy_(torch.randn(values.shape, generator=rng, device="cuda:0") * 300)
            values[:, 0], getattr(engine, f"{kind}_{other}")[:, 0] = 0.0, -0.0
            values[:, 1] = float("inf")
            values[:, 2] = float("nan")
    engine.enemy_x[:, 3], engine.enemy_y[:, 3] = engine.x, engine.y
    engine.enemy_x[:, 4] = engine.x
    angles = torch.arange(engine.enemy_angle.shape[1], device="cuda:0") * (torch.pi / 8)
    engine.enemy_angle.copy_(torch.where(torch.rand(engine.enemy_angle.shape, generator=rng, device="cuda:0") < 0.5, angles, -7.0 * angles))
    if form == "wide tables":
        m.player_starts, m.item_spawns = (torch.cat((t, t), dim=1)[:, : t.shape[1]] for t in (m.player_starts, m.item_spawns))
    if form == "two starts":
        m.player_starts, engine._player_start_z = m.player_starts[:2], engine._player_start_z[:2]
    assert actor_inputs._faced_in_place(engine, lanes)
    packed = actor_inputs.pack_actors_fused(engine, limit=0)
    engine.enemy_angle = spread(engine.enemy_angle)
    assert not actor_inputs._faced_in_place(engine, lanes)
    expected = actor_inputs.pack_actors_fused(engine, limit=0)
    for key in expected:
        same = packed[key] == expected[key]
        if key in ("sprite_x", "sprite_y"):
            same |= packed[key].isnan() & expected[key].isnan()
        assert packed[key].dtype == expected[key].dtype and bool(same.all()), key


@pytest.mark.parametrize("narrow", range(10))
def test_weapon_words_are_read_as_wide_as_they_are_kept(narrow):
    from gradoom_amd import overlay_inputs

    rng = torch.Generator(device="cuda:0").manual_seed(5)
    lanes = 65
    words = {name: torch.randint(-3, 40, (lanes,), generator=rng, device="cuda:0") for name in overlay_inputs._WEAPON_INPUTS}
    tables = {name: torch.randint(0, 50, (8, 2, 11), generator=rng, device="cuda:0") for name in ("weapon_frame_ids", "weapon_flash_ids", "weapon_flash_lights")}
    tables.update(fine_sine=torch.as_tensor(overlay_inputs.fine_sine_fixed(), device="cuda:0"), player_dead=torch.arange(lanes, device="cuda:0") % 3 == 0)
    expected = overlay_inputs.weapon_state(**words, **tables, want_flash_light=True)
    for k, name in enumerate(words):
        if narrow == 9 or k == narrow:
            words[name] = words[name].to(torch.int32)
    packed = overlay_inputs.weapon_state(**words, **tables, want_flash_light=True)
    assert torch.equal(packed[0], expected[0]) and torch.equal(packed[1], expected[1])


@pytest.mark.parametrize("lanes", [1, 64, 65, 1000])
@pytest.mark.parametrize("narrow", [0, 0b01010, 0b11111])
def test_status_bar_words_are_packed_as_the_torch_expressions_pack_them(lanes, narrow):
    from gradoom_amd import _abi, overlay_inputs

    rng = torch.Generator(device="cuda:0").manual_seed(lanes)
    whole = lambda low, high: torch.randint(low, high, (lanes,), generator=rng, device="cuda:0")  # noqa: E731
    real = lambda *shape: torch.rand((lanes, *shape), generator=rng, device="cuda:0")  # noqa: E731
    counters = {name: whole(-2, 3) for name in _abi.HUD_COUNTERS}
    counters["attack_held_tics"] = whole(66, 74)
    counters["mugshot_pain_direction"] = whole(0, 3)
    for k, name in enumerate(_abi.HUD_COUNTERS):
        if (narrow >> k) & 1:
            counters[name] = counters[name].to(torch.int32)
    reals = dict(hud_ready_ammo=real() * 500 - 50, health=real() * 260 - 40, armor=real() * 1200 - 100, weapons=(real(7) < 0.5).to(torch.float32), hud_ammo_counts=real(5) * 900 - 100)
    for name in ("hud_ready_ammo", "health", "armor"):
        reals[name][: lanes // 8] = torch.tensor([float("nan"), float("inf"), -float("inf"), 3e9, -3e9, 1e19, 999.5, -0.5], device="cuda:0")[torch.arange(lanes // 8) % 8]
    fields = dict(active_weapon=whole(0, 8), weapon_ammo_slot=torch.tensor([-1, -1, 0, 1, 0, 3, 2, 1], device="cuda:0"), mugshot_ouch=real() < 0.5, **reals, **counters)
    words = overlay_inputs.hud_state(**fields)
    fields["health"] = spread(fields["health"])
    assert lanes == 1 or overlay_inputs._hud_words_device(whole(0, 3), dict(reals, health=fields["health"]), counters, fields["mugshot_ouch"]) is None
    expected = overlay_inputs.hud_state(**fields)
    assert words.dtype == torch.int32 and words.is_contiguous() and torch.equal(words, expected)
