"""Which kernels a step runs as, on both sides of every line of the rules (no GPU needed)."""

from __future__ import annotations

import pytest
import torch

from pplx_kernels import ops

ONE_LAUNCH, SLOT_MAP, TABLES, SCANNED_TABLES = range(4)


def plan(tokens, row, topk, experts=64, scales=0, ranks=8, dp=1):
    """`tokens` of all groups, rows of `row` bytes with `scales` floats."""
    assert tokens * dp % ranks == 0
    return ops.plan_of(
        ops.Config(tokens * dp // ranks, experts, topk, ranks, dp, row // 2, row, 4 * scales)
    )


@pytest.mark.parametrize(
    "tokens,row,scales,topk,waves,in_turn",
    [
        # 48 KiB and more per wave: three waves, one fetch behind the other, beyond 16384 tokens
        (16384, 7168, 56, 8, 4, False),
        (16392, 7168, 56, 8, 3, True),
        (65536, 7168, 56, 8, 3, True),
        (80000, 7168, 56, 8, 3, True),
        (32768, 14336, 0, 8, 3, True),
        (65536, 16384, 0, 3, 3, True),
        # from 32 KiB on: the same up to 32768 tokens, or for rows of 8 KiB and more
        (16384, 4096, 0, 8, 4, False),
        (16392, 4096, 0, 8, 3, True),
        (32768, 4096, 0, 8, 3, True),
        (32776, 4096, 0, 8, 4, False),
        (32776, 8192, 0, 4, 3, True),
        (65536, 10240, 0, 4, 3, True),
        # from 24 KiB on
        (16392, 4096, 0, 6, 4, False),
        (32768, 8192, 0, 3, 4, False),
        (32776, 8192, 0, 3, 9, False),
        # less
        (32768, 8192, 0, 2, 4, False),
        (32768, 2048, 16, 8, 9, False),
        (32768, 1024, 8, 8, 12, False),
        (32768, 2048, 16, 2, 0, False),
        # rows that cut half lines, through LDS: from 32 KiB on six waves, or eight beyond 32768 tokens; ...
        (16384, 8208, 0, 4, 6, False),
        (16392, 8208, 0, 4, 6, True),  # ... in turn from 8 KiB rows and 16384 tokens on
        (32776, 8208, 0, 4, 6, True),
        (32768, 8176, 0, 6, 6, False),
        (32776, 8176, 0, 6, 8, False),
        (32776, 8176, 0, 3, 8, False),  # from 20 KiB on
        (32776, 8176, 0, 2, 12, False),  # from 12 KiB on
        (32776, 8176, 0, 1, 0, False),
        (32776, 2064, 0, 5, 0, False),
        (32776, 2064, 0, 6, 12, False),
    ],
)
def test_scatter(tokens, row, scales, topk, waves, in_turn):
    p = plan(tokens, row, topk, scales=scales)
    assert p.dispatch_form == (TABLES if tokens <= 65536 else SCANNED_TABLES)
    assert (p.scatter_waves_per_cu, bool(p.scatter_in_turn)) == (waves, in_turn)


@pytest.mark.parametrize(
    "tokens,row,scales,topk,waves",
    [
        (8192, 7168, 56, 2, 4),
        (8200, 7168, 56, 2, 9),
        (8200, 7168, 0, 2, 4),
        (8200, 3584, 28, 4, 9),  # shorter rows: nine with and without
        (8200, 3584, 0, 4, 9),
        (8200, 7168, 56, 4, 4),  # beyond 24 KiB
    ],
)
def test_scatter_of_rows_with_scales(tokens, row, scales, topk, waves):
    p = plan(tokens, row, topk, scales=scales)
    assert (p.dispatch_form, p.scatter_waves_per_cu, bool(p.scatter_in_turn)) == (TABLES, waves, False)


@pytest.mark.parametrize(
    "tokens,row,scales,topk,one_launch",
    [
        # a wave per token in a workgroup per CU
        (4096, 1024, 0, 2, True),
        (4104, 1024, 0, 2, False),
        (2048, 10240, 0, 8, True),
        (2056, 10240, 0, 1, False),
        # bytes of rows: 112 MiB for any number of picks
        (1792, 8192, 0, 8, True),
        (1400, 8192, 0, 10, True),  # 109 MiB
        (1440, 8192, 0, 10, False),  # 112.5
        (2864, 8192, 0, 5, True),  # 111.9
        (2872, 8192, 0, 5, False),  # 112.2
        (1792, 8192, 0, 9, False),  # 126
        # 120 MiB for picks that are counted four at a time, and up to 1024 tokens
        (2120, 7168, 56, 8, True),  # 119.6
        (2128, 7168, 56, 8, False),  # 120.0, 8 KiB beyond
        (3840, 4096, 0, 8, True),  # 120 MiB
        (3848, 4096, 0, 8, False),
        (960, 8192, 0, 16, True),  # 120 MiB
        (968, 8192, 0, 16, False),
        (960, 8192, 0, 17, False),
        # 176 MiB for rows of whole lines, or of 8 KiB, up to 3072 tokens
        (2816, 8192, 0, 8, True),  # 176 MiB
        (2824, 8192, 0, 8, False),
        (2728, 8192, 64, 8, True),  # 175.8
        (2736, 8192, 64, 8, False),  # 176.3
        (3072, 7168, 0, 8, True),  # 168
        (3080, 7168, 0, 8, False),
        # more than sixteen picks, and more than eight that can only be fetched one by one
        (1024, 2048, 0, 17, True),
        (1032, 2048, 0, 17, False),
        (4096, 1024, 0, 16, True),
        (1024, 2048, 0, 9, True),
        (1032, 2048, 0, 9, False),
        (1032, 4096, 0, 9, True),
        (2048, 4096, 0, 9, True),
        (2056, 4096, 0, 9, False),
        (4096, 1024, 0, 10, True),
        # rows in LDS: 180 MiB where they cut half lines, 128 MiB where they do not
        (2880, 8176, 0, 8, True),  # 179.6
        (2888, 8176, 0, 8, False),  # 180.1
        (1816, 9216, 0, 8, True),  # 127.7
        (1824, 9216, 0, 8, False),  # 128.3
        (1824, 9280, 0, 8, False),  # half a line over
        (4096, 9216, 0, 1, True),
        (16, 16368, 0, 2, True),  # the longest that cut half lines
        (16, 16400, 0, 2, False),
    ],
)
def test_one_launch(tokens, row, scales, topk, one_launch):
    assert (plan(tokens, row, topk, scales=scales).dispatch_form == ONE_LAUNCH) == one_launch


@pytest.mark.parametrize(
    "ranks,dp,max_tokens,topk,hidden,dtype,per_group",
    [
        # 10 MiB gathered by all ranks
        (8, 2, 80, 8, 1024, torch.bfloat16, False),
        (8, 2, 81, 8, 1024, torch.bfloat16, True),
        (8, 2, 40, 8, 1024, torch.float32, False),
        (8, 4, 41, 8, 1024, torch.float32, True),
        (64, 4, 1, 8, 7168, torch.bfloat16, False),
        (64, 4, 4, 8, 7168, torch.bfloat16, True),
        # a lane for every member's pick
        (8, 8, 1024, 8, 1024, torch.bfloat16, True),
        (8, 8, 1024, 9, 1024, torch.bfloat16, False),
        (8, 1, 1024, 8, 1024, torch.bfloat16, False),
    ],
)
def test_combine_per_group(ranks, dp, max_tokens, topk, hidden, dtype, per_group):
    p = ops.plan_of(ops.Config(max_tokens, 64, topk, ranks, dp, hidden, 2 * hidden, 0), dtype)
    assert bool(p.combine_per_group) == per_group


@pytest.mark.parametrize(
    "tokens,topk,hidden,dtype,dp,picks,pieces",  # tokens of all groups
    [
        # one and two picks
        (4096, 1, 512, torch.bfloat16, 1, 1, 1),
        (4096, 1, 1024, torch.bfloat16, 1, 1, 2),
        (4096, 1, 2048, torch.bfloat16, 1, 1, 4),
        (4096, 1, 2560, torch.bfloat16, 1, 1, 3),
        (2048, 1, 4096, torch.bfloat16, 1, 1, 8),  # 512 workgroups of 8 KiB pieces
        (1976, 1, 4096, torch.bfloat16, 1, 1, 3),  # 494
        (384, 1, 4096, torch.float32, 1, 1, 1),
        (392, 1, 4096, torch.float32, 1, 1, 2),
        (4096, 1, 4608, torch.bfloat16, 2, 1, 3),
        (4096, 1, 5120, torch.bfloat16, 2, 1, 8),
        (4096, 1, 5120, torch.float32, 2, 1, 3),
        (4096, 2, 512, torch.bfloat16, 1, 2, 1),
        (4096, 2, 4096, torch.bfloat16, 1, 2, 2),
        (4096, 2, 4096, torch.float32, 1, 2, 1),
        (4096, 2, 4096, torch.bfloat16, 2, 2, 4),
        (4096, 2, 4096, torch.float32, 2, 2, 2),
        # three and four
        (4096, 3, 4096, torch.bfloat16, 1, 3, 1),
        (600, 3, 4096, torch.bfloat16, 2, 3, 1),
        (608, 3, 4096, torch.bfloat16, 2, 2, 2),
        (4096, 3, 1024, torch.bfloat16, 2, 3, 1),
        (600, 4, 1024, torch.bfloat16, 1, 4, 1),
        (608, 4, 1024, torch.bfloat16, 1, 4, 2),
        (4096, 4, 4096, torch.bfloat16, 1, 4, 1),
        (600, 4, 4096, torch.bfloat16, 2, 4, 2),
        (608, 4, 4096, torch.bfloat16, 2, 2, 2),
        (2048, 4, 3584, torch.float32, 1, 4, 1),
        (2056, 4, 3584, torch.float32, 1, 8, 1),
        (2056, 4, 3072, torch.float32, 1, 4, 1),
        # more, steps of a few hundred to two thousand tokens
        (384, 8, 7168, torch.bfloat16, 1, 8, 1),
        (392, 8, 7168, torch.bfloat16, 1, 3, 1),  # 196 workgroups of 7 KiB pieces
        (760, 8, 7168, torch.bfloat16, 1, 3, 1),  # 380
        (768, 8, 7168, torch.bfloat16, 1, 1, 7),  # 384, three quarters of two to a CU
        (1024, 8, 4096, torch.bfloat16, 1, 3, 1),  # one to a CU
        (1528, 8, 4096, torch.bfloat16, 1, 3, 1),  # 382
        (1536, 8, 4096, torch.bfloat16, 1, 1, 8),
        (2048, 8, 4608, torch.bfloat16, 1, 3, 1),  # the second piece one KiB
        (2056, 8, 4096, torch.bfloat16, 1, 8, 1),
        (2048, 8, 3072, torch.bfloat16, 1, 8, 1),
        (512, 8, 4096, torch.bfloat16, 2, 2, 2),
        (1024, 8, 4096, torch.bfloat16, 2, 1, 8),  # one to a CU
        (1152, 8, 4096, torch.bfloat16, 2, 1, 3),
        (392, 8, 2048, torch.float32, 1, 2, 1),
        (384, 8, 2048, torch.float32, 1, 8, 1),
        (2048, 8, 1024, torch.float32, 1, 8, 1),
        # ... large ones
        (2056, 8, 1024, torch.float32, 1, 3, 2),
        (2056, 8, 1536, torch.float32, 1, 8, 1),
        (2056, 8, 1536, torch.float32, 2, 3, 1),
        (2056, 8, 512, torch.float32, 1, 8, 1),
        (2056, 5, 4096, torch.bfloat16, 2, 3, 2),
        (2056, 8, 512, torch.bfloat16, 2, 8, 1),
        (2056, 5, 4096, torch.bfloat16, 1, 5, 1),
        (2056, 6, 3072, torch.bfloat16, 1, 3, 1),
        (2056, 6, 3584, torch.bfloat16, 1, 8, 1),
        (384, 6, 3584, torch.bfloat16, 1, 3, 1),
        (2056, 10, 3072, torch.bfloat16, 1, 5, 1),
        (2056, 10, 3584, torch.bfloat16, 1, 8, 1),
        (2056, 9, 512, torch.float32, 1, 5, 1),
        (2056, 7, 3072, torch.bfloat16, 1, 8, 1),
        # ... of more than 512 MiB, or 1 GiB of DP groups
        (43688, 6, 1024, torch.bfloat16, 1, 3, 1),
        (43696, 6, 1024, torch.bfloat16, 1, 8, 1),
        (26208, 10, 1024, torch.bfloat16, 1, 5, 1),
        (26216, 10, 1024, torch.bfloat16, 1, 8, 1),
        (43696, 6, 1032, torch.bfloat16, 1, 3, 1),  # ... and a partial KiB
        (26216, 10, 1032, torch.bfloat16, 1, 8, 1),
        (16392, 8, 4104, torch.bfloat16, 2, 3, 2),
        (43696, 6, 1024, torch.float32, 1, 3, 2),
        (16384, 8, 4096, torch.bfloat16, 2, 3, 2),
        (16392, 8, 4096, torch.bfloat16, 2, 8, 1),
        (13104, 10, 4096, torch.bfloat16, 2, 3, 2),
        (13112, 10, 4096, torch.bfloat16, 2, 8, 1),
        (32768, 7, 4096, torch.bfloat16, 2, 3, 2),
    ],
)
def test_pieces_of_combine(tokens, topk, hidden, dtype, dp, picks, pieces):
    assert tokens % 8 == 0
    p = ops.combine_plan_of(ops.Config(tokens * dp // 8, 64, topk, 8, dp, hidden, 2 * hidden, 0), dtype)
    assert p == (picks, pieces, dp > 1)


@pytest.mark.parametrize(
    "M,H,K,dp,plain",
    [
        (1, 8, 1, 1, True),
        (9, 992, 6, 1, False),  # whole half lines
        (9, 984, 6, 1, True),
        (9, 1000, 6, 1, True),
        (393, 1000, 2, 1, True),  # 8 x 393 x 2000 bytes, 3456 below 6 MiB
        (394, 1000, 2, 1, False),
        (393, 1000, 2, 2, True),  # each rank of a group stores rows of its own
        (394, 1000, 2, 2, False),
        (393, 1000, 2, 4, True),
        (394, 1000, 2, 4, False),
        (4096, 96, 8, 1, False),  # 6 MiB of whole half lines
        (16384, 24, 8, 1, True),  # 6 MiB of rows of 48 bytes
        (16385, 24, 8, 1, False),
    ],
)
def test_stores_of_combine(M, H, K, dp, plain):
    assert ops.combine_stores_plainly(ops.Config(M, 32, K, 8, dp, H, 2 * H, 0)) == plain


@pytest.mark.parametrize(
    "lds,tokens,row,topk,one_launch",
    [
        # 8 x 2 rows of 12 KiB and the tables beside them fit any device's LDS, sixteen rows of 10128 bytes only
        # one of 160 KiB (163712 of its 163840 bytes)
        (160 << 10, 16, 12016, 2, True),
        (64 << 10, 16, 12016, 2, True),
        (0, 16, 12016, 2, True),
        (160 << 10, 4096, 10128, 1, True),
        (163711, 4096, 10128, 1, False),
        (64 << 10, 4096, 10128, 1, False),
        (0, 4096, 10128, 1, False),
        (64 << 10, 4096, 8192, 1, True),  # rows in registers need none
    ],
)
def test_rows_in_lds_need_a_device_that_holds_them(lds, tokens, row, topk, one_launch):
    p, _ = ops.plan_on(ops.Config(tokens // 8, 64, topk, 8, 1, row // 2, row, 0), lds)
    assert (p.dispatch_form == ONE_LAUNCH) == one_launch


@pytest.mark.parametrize(
    "tokens,row,topk,in_lds",
    [
        (8, 8208, 1, True),  # no register variant
        (8, 9216, 1, True),
        (8, 10240, 1, False),
        (672, 3088, 8, False),  # 15.8 MiB of rows that cut half lines
        (680, 3088, 8, True),  # 16.02
        (2744, 3056, 8, False),  # 63.98 MiB of shorter ones
        (2752, 3056, 8, True),  # 64.2
        (4096, 2032, 14, False),  # shorter still
        (2752, 3072, 8, False),  # whole lines
        (2752, 3136, 8, False),  # half a line over
        (8, 8256, 1, True),  # ... and no register variant
    ],
)
def test_rows_of_one_launch_in_lds(tokens, row, topk, in_lds):
    p, rows_in_lds = ops.plan_on(ops.Config(tokens // 8, 64, topk, 8, 1, row // 2, row, 0))
    assert p.dispatch_form == ONE_LAUNCH
    assert rows_in_lds == in_lds


@pytest.mark.parametrize("row,waves", [(26864, 6), (26896, 5), (32752, 4)])
def test_long_rows_in_lds_leave_room_for_fewer_waves(row, waves):
    """LDS is handed out in 128 blocks of 1280 bytes: six rows of 21 blocks, five of 22, four of 26."""
    p = plan(16384, row, 2)
    assert p.dispatch_form == SLOT_MAP and p.scatter_waves_per_cu == waves


@pytest.mark.parametrize(
    "tokens,row,topk,in_lds",
    [
        (40000, 96, 10, False),
        (18728, 112, 3, True),  # rows of 2 MiB together
        (18720, 112, 3, False),
        (5248, 400, 2, True),
        (5240, 400, 2, False),
        (4104, 112, 55, True),  # copies of 24 MiB together
        (4104, 112, 54, False),
        (4104, 512, 8, False),  # whole lines
        (4104, 1088, 8, False),  # half a line over
        (16384, 8256, 4, False),
        (4104, 1008, 1, True),
        (4104, 1040, 8, True),
        (1024, 8192 + 16, 32, True),  # rows from 1 KiB on
        (4104, 10240, 8, False),
        (4104, 32752, 2, True),
        (4104, 32784, 2, False),  # beyond the kernels of one wave per token
    ],
)
def test_rows_of_the_scatter_in_lds(tokens, row, topk, in_lds):
    p, rows_in_lds = ops.plan_on(ops.Config(tokens // 8, 64, topk, 8, 1, row // 2, row, 0))
    assert p.dispatch_form != ONE_LAUNCH
    assert rows_in_lds == in_lds


def test_forms_of_the_routing():
    assert plan(4104, 1024, 2).dispatch_form == TABLES  # 65 chunks
    assert plan(65536, 1024, 2).routing_tiles == 64
    assert plan(65544, 1024, 2).dispatch_form == SCANNED_TABLES
    assert plan(4104, 16384 + 16, 2).dispatch_form == SLOT_MAP  # beyond the register variants
    assert plan(8, 1024, 2).dispatch_form == ONE_LAUNCH
    with pytest.raises(RuntimeError, match="experts_per_token"):
        plan(8, 1024, 0)
