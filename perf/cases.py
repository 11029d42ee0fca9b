"""The measured workloads of the MoE dispatch / combine path.

A case is one step of an MoE layer's communication: dispatch of every simulated rank's tokens into
the experts' buffers, then combine of the experts' outputs into the tokens.  The cases cover what
callers do with the path: the three ways to call it (and the split form of the first), decode
steps of a few tokens up to ragged prefills of tens of thousands, fp8 rows with block scales and
16-bit rows, 16- and 32-bit expert outputs, DP groups of one, two and four ranks, uniform and
skewed routing, token counts that fill the batch or do not.

Fields of a case:
  form      "ranks"  AllToAll.dispatch / .combine once per rank (the operator API)
            "split"  the same in two phases each: every rank sends, then every rank receives
            "world"  LoopbackWorld.dispatch / .combine, all ranks' tensors in one call
            "bound"  a LoopbackWorld.bind of buffers that stay where they are
  ranks, dp, experts, topk, hidden, max_tokens   geometry (max_tokens is per DP group)
  x         dispatched rows: "fp8" (with one fp32 scale per 128 columns), "bf16", "f16"
  y, out    expert outputs ("bf16", "f16", "f32") and combined tokens ("bf16", "f16")
  tokens    "full": every group has max_tokens; "ragged": the groups' counts run from a small
            share of it to nearly all of it; "unbounded": full, without bound_m
  routing   "uniform", "zipf" (s = 1.2) or "mix" (half uniform, half Zipf with s = 1.0)
"""

from __future__ import annotations

import os
import sys

import torch

# The package lives in a folder of the repository that is the working directory.
_PACKAGE_DIR = os.path.join(os.getcwd(), "pplx-kernels_amd")
if _PACKAGE_DIR not in sys.path:
    sys.path.insert(0, _PACKAGE_DIR)

from pplx_kernels import AllToAll, LoopbackWorld  # noqa: E402

_DTYPES = {
    "fp8": torch.float8_e4m3fn,
    "bf16": torch.bfloat16,
    "f16": torch.float16,
    "f32": torch.float32,
}
_BLOCK = 128  # columns per fp32 scale of an fp8 row


def _case(name, form, ranks, dp, experts, topk, hidden, max_tokens, x, y, out, tokens, routing) -> dict:
    case = dict(
        form=form, ranks=ranks, dp=dp, experts=experts, topk=topk, hidden=hidden, max_tokens=max_tokens,
        x=x, y=y, out=out, tokens=tokens, routing=routing,
    )  # fmt: skip
    return {"name": name, **case} if name else case


def listed() -> list[dict]:
    return [
        # The smallest round trip: one rank that holds all experts, 32 tokens of bf16.
        _case("one-rank-32", "bound", 1, 1, 16, 2, 1024, 32, "bf16", "bf16", "bf16", "full", "uniform"),
        # A decode step of a wide expert-parallel deployment: one token on each of 64 ranks.
        _case("decode-64x1", "bound", 64, 1, 256, 8, 7168, 1, "fp8", "bf16", "bf16", "full", "uniform"),
        # A decode step through the operator API, in the smaller of the two shapes of the per-rank
        # latency table (64 experts, top-6, 2048 wide).
        _case("decode-8x4-ranks", "ranks", 8, 1, 64, 6, 2048, 4, "fp8", "bf16", "bf16", "full", "uniform"),
        # The geometry of the operator tests: four ranks in DP groups of two, top-4 of 64, half
        # precision, fewer tokens than the batch holds; all ranks' tensors in one call.
        _case("small-dp2-f16", "world", 4, 2, 64, 4, 1024, 20, "f16", "f16", "f16", "ragged", "uniform"),
        # The headline batch: 128 tokens on each of 8 ranks, 256 experts, top-8, fp8 rows.
        _case("batch-8x128", "bound", 8, 1, 256, 8, 7168, 128, "fp8", "bf16", "bf16", "full", "uniform"),
        # The same batch with unquantised rows and two ranks per DP group, through the operator API.
        _case("batch-dp2-ranks", "ranks", 8, 2, 256, 8, 7168, 128, "bf16", "bf16", "bf16", "unbounded", "uniform"),
        # Send, (expert work elsewhere), receive: the split form, ragged batch.
        _case("batch-8x128-split", "split", 8, 1, 256, 8, 7168, 128, "fp8", "bf16", "bf16", "ragged", "uniform"),
        # A chunk of a chunked prefill, of no round size, tensors handed over as they come.
        _case("chunk-8x509", "world", 8, 1, 256, 8, 7168, 509, "fp8", "bf16", "bf16", "full", "mix"),
        # Prefill in the smaller shape of the latency table, through the operator API.
        _case("prefill-8x1024-ranks", "ranks", 8, 1, 64, 6, 2048, 1024, "fp8", "bf16", "bf16", "full", "uniform"),
        # DP groups of four, rows of no round size, expert outputs accumulated in fp32.
        _case("prefill-dp4-f32", "world", 8, 4, 32, 5, 2880, 3001, "bf16", "f32", "f16", "ragged", "uniform"),
        # Mixtral-shaped prefill: 8 experts, top-2, skewed routing, bf16.
        _case("prefill-8x4096-zipf", "bound", 8, 1, 8, 2, 4096, 4096, "bf16", "bf16", "bf16", "full", "zipf"),
        # The large ragged prefill: up to 8192 tokens per rank, 256 experts, top-8, fp8 rows.
        _case("prefill-8x8192", "world", 8, 1, 256, 8, 7168, 8192, "fp8", "bf16", "bf16", "ragged", "mix"),
    ]


def _log_uniform(rng, low: int, high: int) -> int:
    return min(high, max(low, round(low * (high / low) ** rng.random())))


def draw(rng) -> dict:
    """One more case: forms, types, group sizes and routing at random, sizes spread over their
    logarithm between the smallest and the largest listed case."""
    limit = _bytes_moved(next(c for c in listed() if c["name"] == "prefill-8x8192"))
    while True:
        form = rng.choice(["ranks", "split", "world", "bound"])
        ranks = rng.choice([1, 2, 4, 4, 8, 8, 8, 16, 64])
        dp = rng.choice([d for d in (1, 1, 1, 2, 4) if d == 1 or ranks >= 2 * d])
        experts = ranks * rng.choice([l for l in (1, 2, 3, 4, 8, 16, 32) if 4 <= ranks * l <= 256])
        topk = min(rng.choice([1, 2, 3, 4, 4, 5, 6, 8, 8, 8, 10]), experts)
        x = rng.choice(["fp8", "fp8", "bf16", "f16"])
        y = rng.choice(["bf16", "bf16", "f16", "f32"])
        out = rng.choice(["bf16", "f16"]) if y == "f32" else y
        # (the rows of scales are whole multiples of 16 bytes: four blocks of an fp8 row)
        hidden = 4 * _BLOCK * rng.randint(1, 16) if x == "fp8" else 8 * _log_uniform(rng, 64, 1024)
        groups = ranks // dp
        max_tokens = max(1, _log_uniform(rng, max(groups, 16), 8 * 8192) // groups)
        tokens = rng.choice(["full", "full", "ragged", "unbounded"])
        routing = rng.choice(["uniform", "zipf"] if experts <= 16 else ["uniform", "uniform", "mix"])
        case = _case("", form, ranks, dp, experts, topk, hidden, max_tokens, x, y, out, tokens, routing)
        if _bytes_moved(case) <= limit and _expert_buffer_bytes(case) <= 32e9:
            return case


# ---------------------------------------------------------------------------
# Sizes
# ---------------------------------------------------------------------------
def _token_counts(case: dict) -> list[int]:
    """Tokens present in each DP group (in what order the groups have them follows the seed)."""
    groups = case["ranks"] // case["dp"]
    m = case["max_tokens"]
    if case["tokens"] != "ragged":
        return [m] * groups
    return [max(1, m * (2 * g + 1) // (2 * groups)) for g in range(groups)]


def _capacity(case: dict) -> int:
    """Rows of an expert's buffer: what the busiest expert gets, with room for chance."""
    counts = _token_counts(case)
    total, even = sum(counts), sum(counts) * case["topk"] / case["experts"]
    if case["routing"] == "uniform":
        rows = even + 6 * even**0.5 + 8
    elif case["routing"] == "zipf":
        rows = total
    else:  # the most popular expert of the largest group is picked by most of its skewed half
        rows = even + 6 * even**0.5 + 8 + 0.45 * max(counts) + 0.03 * total
    return (min(int(rows), total) + 15) // 16 * 16


def _expert_buffer_bytes(case: dict) -> int:
    row = case["hidden"] * (_DTYPES[case["x"]].itemsize + _DTYPES[case["y"]].itemsize) + 4 * _scales(case)
    return case["experts"] * _capacity(case) * row


def _scales(case: dict) -> int:
    return (case["hidden"] + _BLOCK - 1) // _BLOCK if case["x"] == "fp8" else 0


def work(case: dict) -> dict:
    """Bytes: a token's row, scales and picks are read once, K copies written; K rows of expert
    outputs with their picks and weights read once per DP group, a row written for each of the
    group's ranks.  Flops: one multiply-add per element of the gathered rows."""
    return {"bytes": _bytes_moved(case), "flops": 2 * sum(_token_counts(case)) * case["topk"] * case["hidden"]}


def _bytes_moved(case: dict) -> int:
    t = sum(_token_counts(case))
    pairs = t * case["topk"]
    row = case["hidden"] * _DTYPES[case["x"]].itemsize + 4 * _scales(case)
    dispatch = t * row + pairs * 4 + pairs * row + case["experts"] * 4
    gathered = pairs * (case["hidden"] * _DTYPES[case["y"]].itemsize + 8)
    combined = t * case["dp"] * case["hidden"] * _DTYPES[case["out"]].itemsize
    return dispatch + gathered + combined


def tolerance(case: dict) -> dict:
    """Dispatch moves bytes, which are compared as such.  Combine accumulates in fp32 and rounds
    once: against the same sums in 64 bits, unrounded, bf16 results differ by 1.7e-3 (2-norm) and
    3.9e-3 of a value at most, f16 results by an eighth of that; four times as much is allowed."""
    return {"rel": 7e-3, "max": 1.6e-2} if case["out"] == "bf16" else {"rel": 9e-4, "max": 2e-3}


# ---------------------------------------------------------------------------
# State of a step
# ---------------------------------------------------------------------------
def _routing(case: dict, n: int, gen: torch.Generator) -> torch.Tensor:
    """[n, K] expert ids, distinct in each row, in no order."""
    experts, k = case["experts"], case["topk"]

    def top(log_pmf) -> torch.Tensor:
        # Gumbel top-k: sampling without replacement
        u = torch.rand(n, experts, generator=gen, device="cuda").clamp_min(1e-20)
        return (log_pmf - torch.log((-torch.log(u)).clamp_min(1e-20))).topk(k, dim=1).indices

    def zipf(s: float) -> torch.Tensor:
        # (which experts are the popular ones differs from group to group)
        order = torch.randperm(experts, generator=gen, device="cuda")
        return -s * torch.log(1.0 + order.float())

    if case["routing"] == "uniform":
        ids = top(0.0)
    elif case["routing"] == "zipf":
        ids = top(zipf(1.2))
    else:
        skewed = torch.rand(n, 1, generator=gen, device="cuda") < 0.5
        ids = torch.where(skewed, top(zipf(1.0)), top(0.0))
    return ids.to(torch.int32).view(torch.uint32)


def _rows(case: dict, n: int, gen: torch.Generator) -> tuple[torch.Tensor, torch.Tensor | None]:
    """N(0, 1) activations; fp8 rows are quantised with an absmax scale per block."""
    h = case["hidden"]
    x = torch.randn(n, h, generator=gen, device="cuda", dtype=torch.float32)
    if case["x"] != "fp8":
        return x.to(_DTYPES[case["x"]]), None
    blocks = x.view(n, h // _BLOCK, _BLOCK)
    scale = blocks.abs().amax(dim=2).clamp_min(1e-12) / 448.0
    return (blocks / scale[:, :, None]).view(n, h).to(_DTYPES["fp8"]), scale


def prepare(case: dict, seed: int) -> dict:
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ranks, dp, experts, topk, hidden = (case[k] for k in ("ranks", "dp", "experts", "topk", "hidden"))
    m, groups, local = case["max_tokens"], case["ranks"] // case["dp"], case["experts"] // case["ranks"]
    counts = _token_counts(case)
    counts = [counts[(g + seed) % groups] for g in range(groups)]

    s: dict = {k: [] for k in ("dp_x", "dp_x_scale", "indices", "weights", "bound_m")}
    s["out_tokens"] = torch.zeros(ranks, m, hidden, dtype=_DTYPES[case["out"]], device="cuda")
    for g in range(groups):
        x, scale = _rows(case, m, gen)
        indices = _routing(case, m, gen)
        weights = torch.softmax(torch.randn(m, topk, generator=gen, device="cuda"), dim=1)
        for member in range(dp):
            # the ranks of a DP group hold copies of the same tokens
            s["dp_x"].append(x if member == 0 else x.clone())
            s["dp_x_scale"].append(scale if scale is None or member == 0 else scale.clone())
            s["indices"].append(indices if member == 0 else indices.clone())
            s["weights"].append(weights if member == 0 else weights.clone())
            s["bound_m"].append(
                None if case["tokens"] == "unbounded"
                else torch.full((1,), counts[g], dtype=torch.int32, device="cuda").view(torch.uint32)
            )  # fmt: skip
    cap, scales = _capacity(case), _scales(case)
    s["counts"] = torch.zeros(ranks, local, dtype=torch.int32, device="cuda")
    s["expert_x"] = torch.zeros(ranks, local, cap, hidden * _DTYPES[case["x"]].itemsize, dtype=torch.uint8,
                                device="cuda").view(_DTYPES[case["x"]])  # fmt: skip
    s["expert_x_scale"] = torch.zeros(ranks, local, cap, scales, device="cuda") if scales else None
    s["expert_y"] = torch.empty(ranks, local, cap, hidden, dtype=_DTYPES[case["y"]], device="cuda")
    for r in range(ranks):
        s["expert_y"][r].normal_(generator=gen)

    geometry = (m, experts, topk, ranks, dp, hidden, hidden * _DTYPES[case["x"]].itemsize, 4 * scales)
    group_name = "-".join(str(v) for v in geometry)
    by_rank = [
        list(s["counts"]), list(s["expert_x"]), list(s["expert_x_scale"]) if scales else [None] * ranks,
        s["dp_x"], s["dp_x_scale"], s["indices"], s["bound_m"],
    ]  # fmt: skip
    s["form"] = case["form"]
    s["dispatch_args"] = by_rank
    s["combine_args"] = [list(s["out_tokens"]), s["indices"], s["weights"], list(s["expert_y"]), s["bound_m"]]
    if case["form"] in ("ranks", "split"):
        m_, e_, k_, r_, dp_, h_, hb_, sb_ = geometry
        s["all_to_all"] = [AllToAll.intranode(m_, e_, k_, r, r_, dp_, h_, hb_, sb_, group_name) for r in range(ranks)]
    else:
        s["world"] = LoopbackWorld(*geometry, group_name=group_name)
        if case["form"] == "bound":
            s["step"] = s["world"].bind(*by_rank, list(s["out_tokens"]), s["weights"], list(s["expert_y"]))
    if case["form"] in ("ranks", "split"):
        # what each rank's program has in hand
        s["dispatch_by_rank"] = [
            dict(out_expert_num_tokens=a, out_expert_x=b, out_expert_x_scale=c, dp_x=d, dp_x_scale=e,
                 indices=f, bound_m=g)
            for a, b, c, d, e, f, g in zip(*by_rank)
        ]  # fmt: skip
        s["combine_by_rank"] = [
            dict(out_tokens=a, indices=b, weights=c, expert_y=d, bound_m=e) for a, b, c, d, e in zip(*s["combine_args"])
        ]
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s: dict) -> dict:
    form = s["form"]
    if form == "bound":
        s["step"].dispatch()
        s["step"].combine()
    elif form == "world":
        s["world"].dispatch(*s["dispatch_args"])
        s["world"].combine(*s["combine_args"])
    elif form == "ranks":
        for ata, kwargs in zip(s["all_to_all"], s["dispatch_by_rank"]):
            ata.dispatch(**kwargs)
        for ata, kwargs in zip(s["all_to_all"], s["combine_by_rank"]):
            ata.combine(**kwargs)
    else:
        for call, by_rank in (("dispatch", s["dispatch_by_rank"]), ("combine", s["combine_by_rank"])):
            for ata, kwargs in zip(s["all_to_all"], by_rank):
                getattr(ata, call)(**kwargs, do_recv=False)
            for ata, kwargs in zip(s["all_to_all"], by_rank):
                getattr(ata, call)(**kwargs, do_send=False)
    outputs = {
        "counts": s["counts"],
        "expert_x": s["expert_x"].view(torch.int64),  # dispatch moves bytes
        "out_tokens": s["out_tokens"],
    }
    if s["expert_x_scale"] is not None:
        outputs["expert_x_scale"] = s["expert_x_scale"].view(torch.int32)
    return outputs
