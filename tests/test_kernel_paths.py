"""GPU tests of single kernel variants and branches of their dispatch, at the sizes where each
can go wrong, against the CPU oracle."""

from __future__ import annotations

import concurrent.futures
import ctypes
import dataclasses

import numpy as np
import pytest
import torch

from pplx_kernels import ops
from tests.all_to_all_utils import (
    COMBINE_ATOL,
    COMBINE_RTOL,
    FP8,
    ORACLE_DTYPE,
    DeviceStep,
    WorkloadSpec,
    check_combine_against_oracle,
    check_dispatch_against_oracle,
    combine_form,
    generate,
    make_world,
    to_oracle_groups,
    torch_bits,
)
from tests.test_contract import FAULT_BAD_EXPERT, FAULT_DUPLICATE, FAULT_ROW_DROPPED, _check_with_repeats_dropped

pytestmark = pytest.mark.gpu

# pplx_a2a_dispatch_form
ONE_LAUNCH, SLOT_MAP, TABLES, SCANNED_TABLES = range(4)


# ---------------------------------------------------------------------------
# Combine of DP groups: one gather for the members that agree
# ---------------------------------------------------------------------------
@pytest.mark.parametrize(
    "dp,K,E,H,M,y_dtype,out_dtype,shared",
    [
        (2, 8, 32, 7168, 120, torch.bfloat16, torch.bfloat16, True),  # long pieces of each row
        (4, 5, 32, 1000, 7, torch.float32, torch.float16, False),
        (4, 5, 32, 1000, 110, torch.float32, torch.float16, True),  # tail of picks, row no multiple of 512
        (2, 1, 8, 8, 1, torch.float16, torch.float16, False),  # the smallest row and step
        (2, 1, 8, 8, 132000, torch.float16, torch.float16, True),  # the smallest row
        (4, 16, 64, 520, 9, torch.bfloat16, torch.bfloat16, False),
        (4, 16, 64, 520, 140, torch.bfloat16, torch.bfloat16, True),  # every lane holds a pick
        (4, 17, 64, 520, 140, torch.bfloat16, torch.bfloat16, False),  # one pick too many for a shared wave
        (8, 8, 64, 264, 5, torch.bfloat16, torch.float16, False),
        (8, 8, 64, 264, 520, torch.bfloat16, torch.float16, True),  # a single group of eight
    ],
)
def test_members_of_a_dp_group_share_or_keep_their_own_sums(dp, K, E, H, M, y_dtype, out_dtype, shared):
    """Member 0 and the last member agree on every token; member 1's weights differ on every
    third token, and it has fewer tokens (so for the rest of them it is absent)."""
    from oracle import a2a_oracle as orc

    spec = WorkloadSpec(
        "dpshare", 71, 8, E, K, H, M, torch.bfloat16, out_dtype=out_dtype, expert_y_dtype=y_dtype, dp_size=dp,
        tokens="uniform",
    )  # fmt: skip
    assert ops.plan_of(ops.Config(M, E, K, 8, dp, H, 2 * H, 0), y_dtype).combine_per_group == shared
    groups = generate(spec, seed=dp * 100 + K)
    for g in groups:
        g.n = min(g.n, 150)
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


# ---------------------------------------------------------------------------
# Slots from the routing tables: one to sixty-four tiles without a scan, more with one
# ---------------------------------------------------------------------------
@pytest.mark.parametrize(
    "E,K,M,R,hidden_bytes",
    [
        # (the rows of a workgroup of the one-launch form would not fit LDS)
        (16, 1, 401, 8, 16368),  # 51 tiles of one chunk, 64 lanes to a pick, the last tile nearly empty
        (64, 33, 129, 8, 8208),  # 17 tiles, one lane to a pick
        (40, 5, 512, 8, 16368),  # exactly 64 tiles; lanes left over (8 to a pick, 5 picks)
        (8, 3, 513, 8, 48),  # 65 chunks: 33 tiles of two
        (24, 10, 4099, 8, 16),  # 513 chunks: 33 tiles of sixteen
        (1024, 2, 2050, 8, 16),  # LDS limits tiles to four chunks: 65 tiles, scanned
        (144, 4, 60, 72, 512),  # rank tables in HBM
    ],
)
def test_slots_from_the_routing_tables(E, K, M, R, hidden_bytes):
    spec = WorkloadSpec("tables", 72, R, E, K, hidden_bytes // 2, M, torch.bfloat16, tokens="uniform")
    form = ops.plan_of(ops.Config(M, E, K, R, 1, spec.hidden_dim, hidden_bytes, 0)).dispatch_form
    assert form == (SCANNED_TABLES if E == 1024 else TABLES)
    groups = generate(spec, seed=E + K)
    groups[0].n, groups[1].n, groups[-1].n = 0, M, M  # an empty rank; a full last tile
    load = np.bincount(
        np.concatenate([g.indices[: g.n].reshape(-1).numpy() for g in groups]), minlength=E
    ).max()  # fmt: skip
    step = DeviceStep(spec, groups, cap=int(load), alloc_expert_y=False)
    world = make_world(spec, group_name="tables")
    for _ in range(2):  # the tables of the step before must not show through
        step.dispatch_world(world)
        check_dispatch_against_oracle(step)
    assert world.faults() == 0
    world.destroy()


@pytest.mark.parametrize(
    "E,K,M,R,hidden_bytes,form",
    [
        (64, 8, 2100, 8, 7168, TABLES),
        (40, 5, 2100, 8, 8208, TABLES),  # no whole registers
        (24, 3, 2100, 8, 16384, TABLES),  # the longest rows that do
        (256, 8, 8200, 8, 7168, SCANNED_TABLES),
        (144, 7, 240, 72, 7168, TABLES),  # rank tables in HBM
    ],
)
@pytest.mark.parametrize("faults", [False, True], ids=["", "faults"])
def test_scatter_that_fetches_row_slots_and_buffers_in_turn(E, K, M, R, hidden_bytes, form, faults):
    fp8 = hidden_bytes == 7168
    spec = WorkloadSpec(
        "in-turn", 75, R, E, K, hidden_bytes if fp8 else hidden_bytes // 2, M, FP8 if fp8 else torch.bfloat16
    )
    groups = generate(spec, seed=E)
    for i, g in enumerate(groups):  # (the batch need not be full for the form to be the one of full ones)
        g.n = (i * 37 + 5) % 90
    if faults:
        groups[1].indices[3, 1] = E + 7
        groups[2].indices[4, K - 1] = groups[2].indices[4, 0]
    ids = np.concatenate([g.indices[: g.n].reshape(-1).numpy() for g in groups])
    load = int(np.bincount(ids[ids < E], minlength=E).max())
    step = DeviceStep(spec, groups, cap=load - 2 if faults else load, alloc_expert_y=False)
    plan = ops.plan_of(
        ops.Config(M, E, K, R, 1, spec.hidden_dim, spec.hidden_dim_bytes, spec.hidden_dim_scale_bytes)
    )
    assert plan.dispatch_form == form and plan.scatter_in_turn
    world = make_world(spec, group_name="in-turn")
    for _ in range(2):
        step.dispatch_world(world)
        if faults:
            _check_with_repeats_dropped(step, after_combine=False)
            assert world.faults() == FAULT_ROW_DROPPED | FAULT_BAD_EXPERT | FAULT_DUPLICATE
        else:
            check_dispatch_against_oracle(step)
            assert world.faults() == 0
    world.destroy()


@pytest.mark.parametrize(
    "M,topk,hidden,in_dtype,form",
    [
        (1792, 8, 1792, torch.bfloat16, ONE_LAUNCH),
        (1793, 8, 8192, torch.bfloat16, ONE_LAUNCH),  # 512-thread workgroups: no limit of bytes
        (2048, 1, 4096, torch.bfloat16, ONE_LAUNCH),
        (4096, 1, 64, torch.bfloat16, ONE_LAUNCH),  # the last step that a workgroup per CU can own
        (4097, 1, 64, torch.bfloat16, TABLES),
        (2048, 1, 5120, torch.bfloat16, ONE_LAUNCH),  # the last one of 512-thread workgroups
        (2049, 1, 5120, torch.bfloat16, TABLES),
        (2816, 8, 4096, torch.bfloat16, ONE_LAUNCH),  # 176 MiB of whole lines
        (2817, 8, 4096, torch.bfloat16, TABLES),
        (2127, 8, 7168, FP8, ONE_LAUNCH),  # 120 MiB with scales
        (2128, 8, 7168, FP8, TABLES),
        (1792, 8, 4096, torch.bfloat16, ONE_LAUNCH),  # 112 MiB
        (1592, 9, 4096, torch.bfloat16, ONE_LAUNCH),  # 112 MiB of picks that are counted one at a time
        (1593, 9, 4096, torch.bfloat16, TABLES),
    ],
)
def test_both_sides_of_the_one_launch_limit(M, topk, hidden, in_dtype, form):
    spec = WorkloadSpec("limit", 73, 1, 16, topk, hidden, M, in_dtype)
    plan = ops.plan_of(
        ops.Config(M, 16, topk, 1, 1, hidden, spec.hidden_dim_bytes, spec.hidden_dim_scale_bytes)
    )
    assert plan.dispatch_form == form
    groups = generate(spec, seed=M)
    groups[0].n = M - 1
    cap = int(np.bincount(groups[0].indices[: M - 1].reshape(-1).numpy(), minlength=16).max())
    step = DeviceStep(spec, groups, cap=cap, alloc_expert_y=False)
    world = make_world(spec, group_name="limit")
    step.dispatch_world(world)
    check_dispatch_against_oracle(step)
    assert world.faults() == 0
    world.destroy()


# ---------------------------------------------------------------------------
# Expert outputs in fp32: how many picks at a time, in pieces of 2 and 4 KiB of a row
# ---------------------------------------------------------------------------
@pytest.mark.parametrize(
    "M,K,H,dp,out_dtype,form",
    [
        (1024, 5, 2048, 1, torch.bfloat16, (2, 1, False)),  # up to 2048 tokens: two, two and one
        (1025, 3, 2048, 1, torch.bfloat16, (3, 1, False)),
        (1025, 8, 3592, 1, torch.float16, (8, 1, False)),  # one vector in the last of eight pieces
        (1025, 5, 2056, 1, torch.bfloat16, (8, 1, False)),  # five pieces: four picks, then one
        (1025, 10, 520, 1, torch.bfloat16, (3, 2, False)),  # one vector beyond a piece; three times three picks, then one
        (1025, 10, 8, 1, torch.bfloat16, (5, 1, False)),  # one piece, of one vector: twice five picks
        (1025, 5, 512, 1, torch.float16, (5, 1, False)),  # a full piece
        (1025, 4, 512, 1, torch.bfloat16, (4, 1, False)),
        (1025, 7, 1536, 2, torch.float16, (3, 1, True)),  # DP groups
        (1025, 3, 2880, 4, torch.float16, (3, 1, True)),
    ],
)
def test_pieces_of_fp32_rows(M, K, H, dp, out_dtype, form):
    spec = WorkloadSpec(
        "pieces", 74, 2 * dp, 8 * dp if dp > 1 else 16, K, H, M, torch.bfloat16, out_dtype=out_dtype,
        expert_y_dtype=torch.float32, dp_size=dp,
    )  # fmt: skip
    assert combine_form(spec) == form
    groups = generate(spec, seed=H + K)
    groups[0].n, groups[1].n = M, M - 3
    experts = np.concatenate([g.indices[: g.n].reshape(-1).numpy() for g in groups])
    step = DeviceStep(spec, groups, cap=int(np.bincount(experts, minlength=spec.num_experts).max()))
    world = make_world(spec, group_name="pieces")
    step.dispatch_world(world)
    expected = check_dispatch_against_oracle(step)
    gen = torch.Generator(device="cuda").manual_seed(5)
    step.expert_y_all.normal_(generator=gen)
    step.combine_world(world)
    check_combine_against_oracle(step, expected.slot_map)
    assert world.faults() == 0
    world.destroy()


@pytest.mark.parametrize("H", [248, 256, 264, 768, 776])
@pytest.mark.parametrize("K,dp", [(3, 1), (8, 2)])
def test_halves_of_an_fp32_piece(H, K, dp):
    """A lane holds two vectors of four columns, 256 columns apart: rows that end in, at and behind a piece's first half."""
    M = 70
    spec = WorkloadSpec(
        "halves", 80, 4, 16, K, H, M, torch.bfloat16, expert_y_dtype=torch.float32, dp_size=dp, tokens="uniform"
    )  # fmt: skip
    groups = generate(spec, seed=H + K)
    groups[0].n, groups[-1].n = M, 1
    step = DeviceStep(spec, groups)
    world = make_world(spec, group_name="halves")
    step.dispatch_world(world)
    expected = check_dispatch_against_oracle(step)
    step.expert_y_all.normal_(generator=torch.Generator(device="cuda").manual_seed(9))
    step.combine_world(world)
    check_combine_against_oracle(step, expected.slot_map)
    assert world.faults() == 0
    world.destroy()


# ---------------------------------------------------------------------------
# Rows that cut 64-byte half lines, and rows without a register variant: through LDS
# ---------------------------------------------------------------------------
@pytest.mark.parametrize(
    "E,K,M,R,row_bytes,form",
    [
        (16, 3, 2, 8, 8208, ONE_LAUNCH),  # no register variant, one vector more than a line
        (16, 2, 3, 8, 16368, ONE_LAUNCH),  # the longest that cuts half lines
        (8, 1, 1, 8, 8304, ONE_LAUNCH),  # one vector less than a line
        (16, 4, 33, 8, 9344, ONE_LAUNCH),  # whole lines without a register variant
        (64, 16, 261, 8, 2064, ONE_LAUNCH),  # 65.8 MiB of short rows
        (64, 8, 129, 8, 3088, ONE_LAUNCH),  # two waves to a token
        (64, 6, 512, 8, 5136, ONE_LAUNCH),  # sixteen rows to a workgroup
        (64, 9, 258, 8, 1392, TABLES),  # picks that are counted one by one
        (64, 1, 512, 8, 10128, ONE_LAUNCH),  # sixteen rows and the tables fill a CU's LDS
        (64, 1, 512, 8, 10144, TABLES),  # ... and no longer fit it; 64 tiles of one chunk, 64 lanes to a pick
        (40, 5, 512, 8, 10240, TABLES),  # whole lines; 64 tiles of one chunk, lanes left over
        (16, 1, 401, 8, 10240, TABLES),  # 51 tiles of one chunk, the last nearly empty
        (40, 5, 520, 8, 1040, TABLES),
        (24, 4, 521, 8, 4208, TABLES),
        (16, 1, 523, 8, 8080, TABLES),
        (8, 8, 530, 8, 16, TABLES),  # eight rows to a line
        (24, 3, 8200, 8, 112, SCANNED_TABLES),
        (16, 2, 5, 8, 16400, SLOT_MAP),
        (16, 2, 5, 8, 32752, SLOT_MAP),  # the longest that goes through LDS
        (144, 3, 3, 72, 8208, ONE_LAUNCH),  # rank tables in HBM
        (144, 3, 60, 72, 1040, TABLES),
        (16, 3, 2, 8, -8592, ONE_LAUNCH),  # (fp8 with 68 scales)
        (32, 6, 520, 8, -2000, TABLES),
    ],
)
@pytest.mark.parametrize("strided", [False, True], ids=["", "strided"])
def test_rows_through_lds(E, K, M, R, row_bytes, form, strided):
    fp8, row_bytes = row_bytes < 0, abs(row_bytes)
    spec = WorkloadSpec(
        "lds-rows", 76, R, E, K, row_bytes if fp8 else row_bytes // 2, M, FP8 if fp8 else torch.bfloat16
    )
    if K * M * R > 20000:
        spec = dataclasses.replace(spec, tokens="uniform")
    plan, in_lds = ops.plan_on(
        ops.Config(M, E, K, R, 1, spec.hidden_dim, spec.hidden_dim_bytes, spec.hidden_dim_scale_bytes)
    )
    assert plan.dispatch_form == form
    assert in_lds == (row_bytes not in (16, 10240))  # (those stay in registers)
    groups = generate(spec, seed=E + K + row_bytes)
    groups[R // 2].n = min(1, groups[R // 2].n)
    ids = np.concatenate([g.indices[: g.n].reshape(-1).numpy() for g in groups])
    step = DeviceStep(spec, groups, cap=int(np.bincount(ids, minlength=E).max()), alloc_expert_y=False)
    if not strided:
        world = make_world(spec, group_name="lds-rows")
        for _ in range(2):
            step.dispatch_world(world)
            check_dispatch_against_oracle(step)
        assert world.faults() == 0
        world.destroy()
        return
    # Through the C ABI, which takes rows at any multiple of 16 bytes: copies 48 bytes apart from 16 bytes behind
    # a line on, sources 16 bytes apart.
    lib = ops.load_library()
    args = (ops.DispatchArgs * R)()
    pitch, rows = row_bytes + 48, E * step.cap
    guard = torch.full((16 + rows * pitch,), 0xA5, dtype=torch.uint8, device="cuda")
    sources = []
    for r in range(R):
        ops.pack_dispatch_args(
            K, step.expert_num_tokens[r], step.expert_x[r], step.expert_x_scale[r], step.dp_x[r], step.dp_x_scale[r],
            step.indices[r], step.bound_m[r], out=args[r],
        )  # fmt: skip
        wide = torch.zeros(step.dp_x[r].shape[0], row_bytes + 16, dtype=torch.uint8, device="cuda")
        wide[:, :row_bytes] = step.dp_x[r].view(torch.uint8)
        sources.append(wide)
        args[r].dp_x, args[r].dp_x_stride_row = wide.data_ptr(), row_bytes + 16
        args[r].out_expert_x = guard.data_ptr() + 16 + r * (E // R) * step.cap * pitch
        args[r].out_expert_x_stride_row, args[r].out_expert_x_stride_expert = pitch, step.cap * pitch
    config = ops.Config(M, E, K, R, 1, spec.hidden_dim, spec.hidden_dim_bytes, spec.hidden_dim_scale_bytes)
    handle = ctypes.c_void_p()
    ops.check_status(lib.pplx_a2a_world_create(ctypes.byref(config), 0, ctypes.byref(handle)))
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    ops.check_status(lib.pplx_a2a_world_dispatch(handle, args, stream))
    torch.cuda.synchronize()
    ops.check_status(lib.pplx_a2a_world_destroy(handle))
    copies = guard[16:].view(rows, pitch)
    step.expert_x_all.view(torch.uint8).view(rows, row_bytes).copy_(copies[:, :row_bytes])
    check_dispatch_against_oracle(step)
    assert (copies[:, row_bytes:] == 0xA5).all() and (guard[:16] == 0xA5).all()


@pytest.mark.parametrize(
    "E,K,M,dp,row_bytes,faults",
    [
        (16, 4, 21, 2, 8208, False),
        (16, 4, 21, 4, 9344, True),  # whole lines without a register variant; a group's rows from four ranks
        (64, 8, 128, 2, 5136, True),  # 20 MiB of rows that a register variant would fit; two waves to a token
        (64, 7, 200, 1, 12304, True),  # seven tokens to a workgroup, picks that the shares of a token do not divide
    ],
)
def test_one_launch_rows_in_lds_of_groups_and_of_faults(E, K, M, dp, row_bytes, faults):
    """Rows in LDS of the one-launch form: eager, dropped rows and bad and repeated picks among them, and replayed from a
    graph."""
    spec = WorkloadSpec("lds-one", 80, 8, E, K, row_bytes // 2, M, torch.bfloat16, dp_size=dp, tokens="uniform")
    plan, in_lds = ops.plan_on(ops.Config(M, E, K, 8, dp, spec.hidden_dim, row_bytes, 0))
    assert plan.dispatch_form == ONE_LAUNCH and in_lds
    groups = generate(spec, seed=row_bytes)
    groups[0].n = M
    if faults:
        groups[0].indices[3, 1] = E + 9
        groups[0].indices[M - 1, K - 1] = groups[0].indices[M - 1, 0]
    ids = np.concatenate([g.indices[: g.n].reshape(-1).numpy() for g in groups])
    load = int(np.bincount(ids[ids < E], minlength=E).max())
    step = DeviceStep(spec, groups, cap=load - 2 if faults else load, alloc_expert_y=False)
    world = make_world(spec, group_name="lds-one")

    def check():
        if faults:
            _check_with_repeats_dropped(step, after_combine=False)
            assert world.faults() == FAULT_ROW_DROPPED | FAULT_BAD_EXPERT | FAULT_DUPLICATE
        else:
            check_dispatch_against_oracle(step)
            assert world.faults() == 0

    step.dispatch_world(world)
    check()
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        with world.capture() as cap:
            step.dispatch_world(world)
        for _ in range(3):
            step.expert_x_all.zero_()
            step.expert_num_tokens_all.zero_()
            stream.synchronize()
            cap.graph.replay(stream)
            stream.synchronize()
            check()
        cap.graph.destroy()
    world.destroy()


@pytest.mark.parametrize("K", [8, 9, 10, 12, 16, 17, 24, 33, 64])
@pytest.mark.parametrize("aligned", [True, False], ids=["", "misaligned-picks"])
def test_one_launch_with_many_picks(K, aligned):
    """Picks beyond eight are held sixteen at a time; repeats are found across those pieces."""
    spec = WorkloadSpec("many-picks", 77, 8, 64, K, 512, 90, torch.bfloat16, tokens="uniform")
    assert ops.plan_of(ops.Config(90, 64, K, 8, 1, 512, 1024, 0)).dispatch_form == ONE_LAUNCH
    groups = generate(spec, seed=K)
    groups[1].n = groups[3].n = 90
    groups[1].indices[3, K - 1] = groups[1].indices[3, 0]
    groups[1].indices[4, K // 2] = groups[1].indices[4, 1]
    groups[3].indices[0, 0] = 64
    groups[3].indices[7] = groups[3].indices[7, 0].item()
    step = DeviceStep(spec, groups, alloc_expert_y=False)
    if not aligned:
        for r, idx in enumerate(step.indices):
            flat = torch.zeros(idx.numel() + 1, dtype=torch.int32, device="cuda").view(torch.uint32)
            flat[1:] = idx.reshape(-1)
            step.indices[r] = flat[1:].view(idx.shape)
    world = make_world(spec, group_name="many-picks")
    step.dispatch_world(world)
    _check_with_repeats_dropped(step, after_combine=False)
    assert world.faults() == FAULT_BAD_EXPERT | FAULT_DUPLICATE
    world.destroy()


@pytest.mark.parametrize("row_bytes", [1024, 1040, 8208])
def test_one_launch_with_many_picks_and_rank_tables_in_hbm(row_bytes):
    spec = WorkloadSpec("many-ranks", 81, 72, 144, 10, row_bytes // 2, 8, torch.bfloat16, tokens="uniform")
    assert ops.plan_of(ops.Config(8, 144, 10, 72, 1, row_bytes // 2, row_bytes, 0)).dispatch_form == ONE_LAUNCH
    step = DeviceStep(spec, generate(spec, seed=row_bytes), alloc_expert_y=False)
    world = make_world(spec, group_name="many-ranks")
    step.dispatch_world(world)
    check_dispatch_against_oracle(step)
    assert world.faults() == 0
    world.destroy()


# ---------------------------------------------------------------------------
# Combine of few picks: pieces that are no longer than the row
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize(
    "H,dp,y_dtype,out_dtype,forms",  # picks and pieces of one to six picks
    [
        (8, 1, torch.bfloat16, torch.bfloat16, "11 21 31 41 51 31"),  # one vector
        (512, 1, torch.float16, torch.float16, "11 21 31 41 51 31"),  # a full segment
        (520, 1, torch.bfloat16, torch.bfloat16, "12 22 31 42 51 31"),  # one vector in the second
        (1032, 1, torch.bfloat16, torch.float16, "13 22 31 41 51 31"),  # one vector in the third
        (1536, 2, torch.float16, torch.bfloat16, "13 22 31 41 51g 81g"),  # three segments; g: once per group
        (1544, 1, torch.bfloat16, torch.bfloat16, "14 22 31 41 51 31"),  # one vector in the fourth
        (4096, 2, torch.bfloat16, torch.bfloat16, "13 24g 31g 42g 51g 81g"),
        (1032, 1, torch.float32, torch.bfloat16, "12 21 31 41 21 21"),
        (504, 4, torch.float32, torch.float16, "11 21 31 41 51 31"),
    ],
)
def test_pieces_of_few_picks(K, H, dp, y_dtype, out_dtype, forms):
    M = 90
    spec = WorkloadSpec(
        "few-picks", 78, 8, 16, K, H, M, torch.bfloat16, out_dtype=out_dtype, expert_y_dtype=y_dtype, dp_size=dp,
        tokens="uniform",
    )  # fmt: skip
    picks, pieces, per_group = combine_form(spec)
    assert f"{picks}{pieces}{'g' if per_group else ''}" == forms.split()[K - 1]
    groups = generate(spec, seed=H + K)
    groups[0].n, groups[-1].n = M, 1
    step = DeviceStep(spec, groups)
    world = make_world(spec, group_name="few-picks")
    step.dispatch_world(world)
    expected = check_dispatch_against_oracle(step)
    step.expert_y_all.normal_(generator=torch.Generator(device="cuda").manual_seed(7))
    step.combine_world(world)
    check_combine_against_oracle(step, expected.slot_map)
    assert world.faults() == 0
    world.destroy()


@pytest.mark.parametrize(
    "K,H,M,y_dtype,dp,form",
    [
        (5, 3592, 48, torch.bfloat16, 1, (5, 1, False)),  # 384 tokens, rows of 8 KiB
        (5, 3592, 49, torch.bfloat16, 1, (3, 1, False)),  # 392: long pieces would leave most CUs without one
        (8, 4096, 256, torch.float16, 1, (1, 8, False)),  # 2048: long pieces, two workgroups to a CU
        (8, 4096, 257, torch.float16, 1, (8, 1, False)),  # 2056
        (7, 3080, 140, torch.bfloat16, 1, (3, 1, False)),  # seven KiB, the last a single vector; 1120 tokens
        (8, 3592, 100, torch.bfloat16, 2, (2, 2, True)),  # DP groups: up to a workgroup of long pieces to a CU
        (8, 3592, 300, torch.bfloat16, 2, (1, 3, True)),  # ... beyond
        (8, 520, 600, torch.float16, 2, (3, 2, True)),  # ... large steps
        (4, 1032, 160, torch.bfloat16, 2, (2, 2, True)),  # ... four picks
        (9, 1032, 60, torch.bfloat16, 1, (5, 1, False)),  # five picks, then four
        (10, 3080, 257, torch.bfloat16, 1, (8, 1, False)),  # eight, then two
        (5, 1032, 60, torch.float32, 1, (2, 1, False)),
        (4, 3080, 257, torch.float32, 1, (8, 1, False)),  # four picks in the form that takes up to eight
        (7, 1032, 520, torch.float32, 2, (3, 1, True)),
    ],
)
def test_pieces_of_many_picks(K, H, M, y_dtype, dp, form):
    spec = WorkloadSpec(
        "many-picks", 81, 8, 16, K, H, M, torch.bfloat16, expert_y_dtype=y_dtype, dp_size=dp, tokens="uniform"
    )  # fmt: skip
    assert combine_form(spec) == form
    groups = generate(spec, seed=H + K)
    groups[0].n, groups[-1].n = M, 1
    step = DeviceStep(spec, groups)
    world = make_world(spec, group_name="many-picks")
    step.dispatch_world(world)
    expected = check_dispatch_against_oracle(step)
    step.expert_y_all.normal_(generator=torch.Generator(device="cuda").manual_seed(10))
    step.combine_world(world)
    check_combine_against_oracle(step, expected.slot_map)
    assert world.faults() == 0
    world.destroy()


@pytest.mark.parametrize(
    "K,H,M,y_dtype,dp,form",
    [
        (1, 3584, 256, torch.bfloat16, 1, (1, 8, False)),  # two workgroups to a CU
        (1, 3208, 250, torch.float16, 1, (1, 8, False)),  # ... a few less, the last of seven KiB a single vector
        (1, 7680, 256, torch.bfloat16, 1, (1, 8, False)),  # ... four workgroups, two pieces to a row
        (2, 1544, 512, torch.float32, 1, (2, 1, False)),  # pieces of 2 KiB, the last a single vector
        (2, 2560, 300, torch.bfloat16, 2, (2, 4, True)),  # five KiB of a DP group's rows
        (2, 1032, 320, torch.float16, 4, (2, 4, True)),  # a single vector in the third
        (1, 2568, 150, torch.float32, 2, (1, 3, True)),  # a single vector in the sixth piece of 2 KiB
    ],
)
def test_long_pieces_of_few_picks(K, H, M, y_dtype, dp, form):
    spec = WorkloadSpec(
        "long-pieces", 79, 8, 16, K, H, M, torch.bfloat16, expert_y_dtype=y_dtype, dp_size=dp, tokens="uniform"
    )  # fmt: skip
    assert combine_form(spec) == form
    groups = generate(spec, seed=H + K)
    groups[0].n, groups[-1].n = M, 1
    step = DeviceStep(spec, groups)
    world = make_world(spec, group_name="long-pieces")
    step.dispatch_world(world)
    expected = check_dispatch_against_oracle(step)
    step.expert_y_all.normal_(generator=torch.Generator(device="cuda").manual_seed(8))
    step.combine_world(world)
    check_combine_against_oracle(step, expected.slot_map)
    assert world.faults() == 0
    world.destroy()


# ---------------------------------------------------------------------------
# Bound steps: rank tables in device memory on the stream that bound them, with the launch elsewhere
# ---------------------------------------------------------------------------
@pytest.mark.parametrize(
    "R,L,M,row_bytes,K",
    [
        (1, 8, 5, 1024, 2),  # one launch
        (8, 4, 90, 5264, 4),  # ... rows in LDS
        (64, 1, 3, 2048, 8),  # the most ranks whose tables fit the arguments
        (72, 1, 3, 1040, 3),  # ... and beyond
        (8, 1, 900, 2064, 3),  # routing and scatter
        (2, 8, 300, 16400, 2),  # ... with the slots in a launch of their own
    ],
)
def test_bound_step_on_its_stream_on_another_and_in_a_graph(R, L, M, row_bytes, K):
    spec = WorkloadSpec("bound", 82, R, R * L, K, row_bytes // 2, M, torch.bfloat16, tokens="uniform")
    step = DeviceStep(spec, generate(spec, seed=1), cap=R * M)
    world = make_world(spec, group_name="bound")
    step.expert_y_all.normal_(generator=torch.Generator(device="cuda").manual_seed(11))
    stream, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        bound = step.bind_world(world)
        bound.dispatch()
        bound.combine()
        stream.synchronize()
        with world.capture() as cap:
            bound.dispatch()
            bound.combine()

    def check(seed, launch):
        new = generate(spec, seed=seed)
        new[-1].n = 0
        for r, g in enumerate(new):
            step.dp_x[r].copy_(g.x)
            step.indices[r].copy_(g.indices.to(torch.uint32))
            step.weights[r].copy_(g.weights)
            step.bound_m[r].copy_(torch.tensor([g.n], dtype=torch.uint32))
            step.out_tokens[r].fill_(float("nan"))
        step.groups = new
        torch.cuda.synchronize()
        launch()
        torch.cuda.synchronize()
        expected = check_dispatch_against_oracle(step)
        check_combine_against_oracle(step, expected.slot_map)

    def launch_on(s):
        bound.dispatch(stream=s)
        bound.combine(stream=s)

    for seed in (2, 3):
        check(seed, lambda: launch_on(stream))
        check(seed + 10, lambda: launch_on(other))
        check(seed + 20, lambda: cap.graph.replay(stream))
    # the graph outlives the bound step, and what its tables were in
    del bound, launch_on
    with torch.cuda.stream(stream):
        reused = [torch.full((1 << 14,), 0x5A, dtype=torch.uint8, device="cuda") for _ in range(8)]
    check(30, lambda: cap.graph.replay(stream))
    assert all((t == 0x5A).all() for t in reused)
    with torch.cuda.stream(stream):
        again = step.bind_world(world)
    check(31, lambda: (again.dispatch(stream), again.combine(stream)))
    assert world.faults() == 0
    cap.graph.destroy()
    world.destroy()


def test_bound_step_on_the_stream_per_thread_takes_its_tables_along():
    spec = WorkloadSpec("bound", 84, 4, 16, 2, 512, 20, torch.bfloat16, tokens="uniform")
    groups = generate(spec, seed=1)
    mine, others = DeviceStep(spec, groups), DeviceStep(spec, groups)
    world = make_world(spec, group_name="bound-per-thread")
    bound, other = mine.bind_world(world), others.bind_world(world)
    packed = [ctypes.addressof(args) for args in bound._keep[:2]]
    tables = torch.empty_like(bound._tables)
    torch.cuda.synchronize()
    per_thread = 2  # hipStreamPerThread: one handle, another stream in every thread
    plan = ops._C.bind_step(world._world_id, *packed, tables.data_ptr(), per_thread)
    torch.cuda.synchronize()
    tables.copy_(other._tables)  # what an unordered launch might see: here the tables of a step on other buffers
    torch.cuda.synchronize()
    for op in (0, 1):
        ops._C.launch_plan(op, world._world_id, plan, 0, per_thread)
    torch.cuda.synchronize()
    expected = check_dispatch_against_oracle(mine)
    check_combine_against_oracle(mine, expected.slot_map)
    assert world.faults() == 0
    del plan
    world.destroy()


@pytest.mark.parametrize("which", ["another thread, global", "this thread", "a blocking stream"])
def test_binding_leaves_captures_alone(which):
    """Where the memory for the tables has to come from the device, and on a stream that a capture keeps launches from."""
    spec = WorkloadSpec("bound", 86, 4, 16, 2, 512, 6, torch.bfloat16, tokens="uniform")
    step = DeviceStep(spec, generate(spec, seed=1))
    step.expert_y_all.normal_(generator=torch.Generator(device="cuda").manual_seed(13))
    world = make_world(spec, group_name="bound-capture")
    captured, fresh = torch.cuda.Stream(), torch.cuda.Stream()
    counter = torch.zeros(1, device="cuda")
    torch.cuda.synchronize()
    torch.cuda.empty_cache()  # nothing is left that the new stream could take memory from

    def bind_on(stream):
        with torch.cuda.stream(stream):
            return step.bind_world(world)

    if which == "another thread, global":
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=captured, capture_error_mode="global"):
            counter.add_(1)
            with concurrent.futures.ThreadPoolExecutor(1) as other:
                bound = other.submit(bind_on, fresh).result(timeout=60)
        replay = graph.replay
    else:
        lib = ops.load_library()
        handle = ctypes.c_void_p(captured.cuda_stream)
        if which == "a blocking stream":  # (torch's are not): the default stream takes no launches meanwhile
            assert lib.hipStreamCreate(ctypes.byref(handle)) == 0
        recorded = torch.cuda.ExternalStream(handle.value)
        with torch.cuda.stream(recorded), world.capture() as cap:
            counter.add_(1)
            bound = bind_on(fresh if which == "this thread" else torch.cuda.default_stream())
        replay = lambda: cap.graph.replay(recorded)  # noqa: E731
    for launches in range(1, 4):
        replay()
        torch.cuda.synchronize()
        assert counter.item() == launches
        bound.dispatch(fresh)
        bound.combine(fresh)
        torch.cuda.synchronize()
        expected = check_dispatch_against_oracle(step)
        check_combine_against_oracle(step, expected.slot_map)
    assert world.faults() == 0
    if which != "another thread, global":
        cap.graph.destroy()
    world.destroy()


def test_an_error_of_hip_at_the_binding_is_raised():
    """Here the one that the default stream reports while a blocking stream is captured."""
    spec = WorkloadSpec("bound", 88, 2, 8, 2, 512, 6, torch.bfloat16, tokens="uniform")
    step = DeviceStep(spec, generate(spec, seed=1))
    world = make_world(spec, group_name="bound-error")
    bound = step.bind_world(world)
    packed = [ctypes.addressof(args) for args in bound._keep[:2]]
    tables = torch.zeros_like(bound._tables)
    torch.cuda.synchronize()
    handle = ctypes.c_void_p()
    assert ops.load_library().hipStreamCreate(ctypes.byref(handle)) == 0
    recorded = torch.cuda.ExternalStream(handle.value)
    with torch.cuda.stream(recorded), world.capture() as cap:
        bound.dispatch()
        with pytest.raises(RuntimeError, match="HIP error"):
            ops._C.bind_step(world._world_id, *packed, tables.data_ptr(), 0)
    cap.graph.replay(recorded)
    torch.cuda.synchronize()
    check_dispatch_against_oracle(step)
    assert world.faults() == 0 and not tables.any()
    cap.graph.destroy()
    world.destroy()


def test_bound_step_that_cannot_be_launched_says_so_at_its_launch():
    spec = WorkloadSpec("bound", 83, 4, 8, 2, 512, 6, torch.bfloat16, dp_size=2, tokens="uniform")
    step = DeviceStep(spec, generate(spec, seed=1))
    world = make_world(spec, group_name="bound-bad")
    step.bound_m[1] = None  # (its group's first rank has one)
    bound = step.bind_world(world)
    with pytest.raises(RuntimeError, match="share a DP group"):
        bound.dispatch()
    world.destroy()


def test_binding_for_a_destroyed_world_fails_at_the_launch():
    spec = WorkloadSpec("bound", 87, 2, 8, 2, 512, 6, torch.bfloat16, tokens="uniform")
    step = DeviceStep(spec, generate(spec, seed=1))
    world = make_world(spec, group_name="bound-gone")
    world.destroy()
    bound = step.bind_world(world)
    for launch in (bound.dispatch, bound.combine):
        with pytest.raises(RuntimeError, match="the world has been destroyed"):
            launch()


# ---------------------------------------------------------------------------
# Rank tables among the arguments: up to eight ranks in a short one
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("ranks,dp", [(1, 1), (7, 1), (8, 1), (8, 4), (9, 1), (10, 2), (63, 1), (64, 2)])
@pytest.mark.parametrize("tokens,H,form", [(40, 1024, ONE_LAUNCH), (4160, 64, TABLES)])
def test_tables_of_few_and_of_many_ranks(ranks, dp, tokens, H, form):
    E = 2 * ranks if ranks > 1 else 8
    M = tokens * dp // ranks + 1
    spec = WorkloadSpec("tables", 17, ranks, E, min(3, E), H, M, torch.bfloat16, dp_size=dp, tokens="uniform")
    assert ops.plan_of(ops.Config(M, E, spec.experts_per_token, ranks, dp, H, 2 * H, 0)).dispatch_form == form
    step = DeviceStep(spec, generate(spec, seed=ranks))
    world = make_world(spec, group_name="tables")
    step.dispatch_world(world)
    expected = check_dispatch_against_oracle(step)
    step.expert_y_all.normal_(generator=torch.Generator(device="cuda").manual_seed(ranks))
    step.combine_world(world)
    check_combine_against_oracle(step, expected.slot_map)
    for t in (step.expert_num_tokens_all, step.expert_x_all):
        t.zero_()
    for t in step.out_tokens:
        t.fill_(float("nan"))
    for do_send in (True, False):
        for r, ata in enumerate(world.ranks):
            ata.dispatch(
                out_expert_num_tokens=step.expert_num_tokens[r], out_expert_x=step.expert_x[r], out_expert_x_scale=None,
                dp_x=step.dp_x[r], dp_x_scale=None, indices=step.indices[r], bound_m=step.bound_m[r],
                do_send=do_send, do_recv=not do_send,
            )  # fmt: skip
    check_dispatch_against_oracle(step, expected)
    for do_send in (True, False):
        for r, ata in enumerate(world.ranks):
            ata.combine(
                out_tokens=step.out_tokens[r], indices=step.indices[r], weights=step.weights[r],
                expert_y=step.expert_y[r], bound_m=step.bound_m[r], do_send=do_send, do_recv=not do_send,
            )  # fmt: skip
    check_combine_against_oracle(step, expected.slot_map)
    assert world.faults() == 0
    world.destroy()


# ---------------------------------------------------------------------------
# Combined rows that cut half lines: plain stores up to 6 MiB of them
# ---------------------------------------------------------------------------
@pytest.mark.parametrize(
    "M,H,K,dp,y_dtype",
    [
        (1, 8, 1, 1, torch.bfloat16),  # the smallest
        (3, 40, 2, 1, torch.float16),
        (9, 992, 6, 1, torch.bfloat16),  # whole half lines: streaming
        (9, 1000, 6, 1, torch.bfloat16),
        (70, 2008, 1, 1, torch.bfloat16),  # pieces of several KiB
        (33, 520, 4, 1, torch.float32),
        (33, 520, 5, 2, torch.float32),
        (100, 2968, 3, 4, torch.float16),  # rows shared by a group's members, each stored by itself
        (392, 1000, 2, 1, torch.bfloat16),  # 5.98 MiB
        (394, 1000, 2, 1, torch.bfloat16),  # 6.01 MiB
    ],
)
def test_combined_rows_that_cut_half_lines(M, H, K, dp, y_dtype):
    spec = WorkloadSpec(
        "cutrows", 23, 8, 16, K, H, M, torch.bfloat16, out_dtype=torch.bfloat16, expert_y_dtype=y_dtype, dp_size=dp,
        tokens="uniform" if M > 1 else "full",
    )  # fmt: skip
    step = DeviceStep(spec, generate(spec, seed=M + H))
    world = make_world(spec, group_name="cutrows")
    for replay in range(2):
        for t in step.out_tokens:
            t.fill_(float("nan"))
        step.dispatch_world(world)
        expected = check_dispatch_against_oracle(step)
        step.expert_y_all.normal_(generator=torch.Generator(device="cuda").manual_seed(replay))
        step.combine_world(world)
        check_combine_against_oracle(step, expected.slot_map)
    assert world.faults() == 0
    world.destroy()
