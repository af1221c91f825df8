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
