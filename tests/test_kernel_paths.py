"""GPU tests of single kernel variants and branches of their dispatch, at the sizes where each
can go wrong, against the CPU oracle."""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest
import torch

from tests.all_to_all_utils import (
    COMBINE_ATOL,
    COMBINE_RTOL,
    ORACLE_DTYPE,
    DeviceStep,
    WorkloadSpec,
    check_dispatch_against_oracle,
    generate,
    make_world,
    to_oracle_groups,
    torch_bits,
)

pytestmark = pytest.mark.gpu


# ---------------------------------------------------------------------------
# Combine of DP groups: one gather for the members that agree
# ---------------------------------------------------------------------------
@pytest.mark.parametrize(
    "dp,K,E,H,M,y_dtype,out_dtype",
    [
        (2, 8, 32, 7168, 120, torch.bfloat16, torch.bfloat16),  # long pieces of each row
        (4, 5, 32, 1000, 7, torch.float32, torch.float16),  # tail of picks, row no multiple of 512
        (2, 1, 8, 8, 1, torch.float16, torch.float16),  # the smallest row and step
        (4, 16, 64, 520, 9, torch.bfloat16, torch.bfloat16),  # every lane holds a pick
        (4, 17, 64, 520, 9, torch.bfloat16, torch.bfloat16),  # one pick too many for a shared wave
        (8, 8, 64, 264, 5, torch.bfloat16, torch.float16),  # a single group of eight
    ],
)
def test_members_of_a_dp_group_share_or_keep_their_own_sums(dp, K, E, H, M, y_dtype, out_dtype):
    """Member 0 and the last member agree on every token; member 1's weights differ on every
    third token, and it has fewer tokens (so for the rest of them it is absent)."""
    from oracle import a2a_oracle as orc

    spec = WorkloadSpec(
        "dpshare", 71, 8, E, K, H, M, torch.bfloat16, out_dtype=out_dtype, expert_y_dtype=y_dtype, dp_size=dp,
        tokens="uniform",
    )  # fmt: skip
    groups = generate(spec, seed=dp * 100 + K)
    step = DeviceStep(spec, groups)
    own = [dataclasses.replace(groups[r // dp]) for r in range(8)]
    for r in range(1, 8, dp):
        weights = own[r].weights.clone()
        weights[::3] *= 1.5
        own[r] = dataclasses.replace(own[r], weights=weights, n=max(1, own[r].n - 2))
        step.weights[r] = weights.cuda()
    world = make_world(spec, group_name="dpshare")
    step.dispatch_world(world)
    expected = check_dispatch_against_oracle(step)
    gen = torch.Generator(device="cuda").manual_seed(3)
    step.expert_y_all.normal_(generator=gen)
    for r in range(8):
        step.bound_m[r] = torch.tensor([own[r].n], dtype=torch.uint32, device="cuda")
    step.combine_world(world)
    assert world.faults() == 0
    world.destroy()
    y = torch_bits(step.expert_y_all.reshape(E, step.cap, H))
    for member in range(dp):
        mine = to_oracle_groups([own[g * dp + member] for g in range(8 // dp)])
        want = orc.c_combine(mine, M, E, K, H, y, ORACLE_DTYPE[y_dtype], ORACLE_DTYPE[out_dtype], expected.slot_map)
        for g, data in enumerate(mine):
            got = step.out_tokens[g * dp + member].cpu()
            np.testing.assert_allclose(
                got[: data.n].float().numpy(), orc.to_float32(want[g], ORACLE_DTYPE[out_dtype]),
                rtol=COMBINE_RTOL, atol=COMBINE_ATOL, err_msg=f"group {g} member {member}",
            )  # fmt: skip
            assert torch.isnan(got[data.n :]).all()
