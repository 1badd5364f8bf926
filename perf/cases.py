"""The work whose speed is watched: dispatch / expert / combine cycles as callers of this package run them.

A pass is one complete cycle of the expert-parallel path, through one of its two public interfaces -

  "world"    whole-world calls (`WorldHarness` over `ep.World`): every logical rank in one call;
  "buffer"   the per-rank Python `Buffer`: one dispatch and one combine call per logical rank, outputs allocated
             inside the calls -

and with one of four things between dispatch and combine:

  "expert"   the rows an expert's GEMMs left (given): combine reads bf16 rows that dispatch did not write;
  "identity" dispatch's own bf16 payload is what combine reads (no expert);
  "cast"     the mock expert of the benchmark programs: packed rows back to bf16 times a factor per expert;
  "packed"   the same mock expert fused into combine.

The world of logical ranks is the process's own, one per number of ranks (`ep.default_world`), as a communicator is:
a program hands it tensors at other addresses from layer to layer and from step to step.  Passes run on the current
stream and do not wait.

Outputs come whole.  Rows of the packed layout at and beyond packed_recv_count are never written; where a payload is
an output it therefore starts from zeros.  A payload that the cycle itself consumes reaches the caller through the
combined tokens.
"""
import math

import torch

from mooncake_amd import Buffer, LogicalGroup, ep
from mooncake_amd.harness import WorldHarness
from mooncake_amd.workloads import EPConfig


def listed():
    base = {"routing": "uniform", "outliers": 0.0, "masked": 0.0, "ragged": False, "batches": 1}

    def case(name, api, chain, ranks, tokens, hidden, experts, topk, fp8, **more):
        return dict(base, name=name, api=api, chain=chain, ranks=ranks, tokens=tokens, hidden=hidden,
                    experts=experts, topk=topk, fp8=fp8, **more)

    return [
        # the smallest calls: one deployed rank with a handful of tokens left in its decode batch
        case("one_rank_8_tokens", "buffer", "cast", 1, 8, 7168, 256, 8, True),
        # one deployed rank's share of a DeepSeek-V3-style decode step
        case("one_rank_decode", "buffer", "cast", 1, 128, 7168, 256, 8, True),
        # the configuration the CPU statement of the contract is checked on
        case("cpu_check", "world", "expert", 4, 128, 2048, 16, 4, False),
        # nothing even: ranks with different token counts, odd hidden, expert and top-k sizes, masked tokens
        case("odd_ragged", "world", "expert", 12, 70, 1152, 108, 5, True, ragged=True, masked=0.15),
        # a decode step of a small expert-parallel group
        case("group_decode", "world", "expert", 8, 64, 4096, 64, 6, True),
        # DeepSeek-V3-style decode step of the whole group, the configuration the headline figure is quoted on
        case("dsv3_decode", "world", "expert", 32, 128, 7168, 256, 8, True),
        # the same step as two micro-batches in flight: both are dispatched before the first is combined
        case("dsv3_two_batches", "world", "expert", 32, 64, 7168, 256, 8, True, batches=2),
        # Qwen3-MoE-style decode, a call per rank
        case("qwen3_decode", "buffer", "identity", 16, 256, 4096, 128, 8, False),
        # DeepSeek-V3-style prefill burst, skewed routing and outlier rows, combine fused with the mock expert
        case("dsv3_prefill", "world", "packed", 32, 128, 7168, 256, 8, True, routing="zipf", outliers=0.01),
        # Mixtral-style, a tenth of the tokens masked, mock expert in between
        case("mixtral", "world", "cast", 8, 1024, 4096, 8, 2, False, masked=0.10),
        # the EP benchmark's shape with an fp8 payload and incast routing: dispatch, mock expert, combine
        case("ep_benchmark_k_hot", "world", "cast", 8, 1024, 7168, 256, 8, True, routing="k_hot"),
        # the largest: prefill-sized calls, more selections than the benchmark's configurations reach
        case("large_prefill", "world", "identity", 8, 4096, 4096, 64, 8, False),
    ]


# A drawn case moves no more than the largest listed one and holds its tensors in this much memory.
_MOST_BYTES = 4.8e9
_MOST_STATE = 40e9


def draw(rng):
    while True:
        ranks = rng.choice([1, 1, 2, 3, 4, 6, 8, 8, 12, 16, 32])
        local = rng.choice([1, 2, 3, 4, 8, 9, 16, 32]) if ranks > 1 else rng.choice([8, 16, 60, 64, 128, 256])
        experts = ranks * local
        topk = min(experts, rng.choice([1, 2, 2, 4, 5, 6, 8, 8, 8, 9, 11]))
        tokens = int(round(math.exp(rng.uniform(math.log(2), math.log(4096)))))
        hidden = 128 * int(round(math.exp(rng.uniform(math.log(6), math.log(64)))))
        fp8 = rng.random() < 0.6
        if fp8:                                        # the scale layout wants ranks * tokens in fours
            while ranks * tokens % 4:
                tokens += 1
        api = "buffer" if rng.random() < 0.3 and ranks <= 16 else "world"
        if api == "buffer":
            chain = "cast" if fp8 else "identity"
        else:
            chain = rng.choice(["expert", "expert", "cast", "packed"] if fp8 else
                               ["expert", "identity", "cast", "packed"])
        case = {"api": api, "chain": chain, "ranks": ranks, "tokens": tokens, "hidden": hidden, "experts": experts,
                "topk": topk, "fp8": fp8, "routing": rng.choice(["uniform", "uniform", "zipf", "k_hot"]),
                "outliers": rng.choice([0.0, 0.01]), "masked": rng.choice([0.0, 0.0, 0.1, 0.3]),
                "ragged": rng.random() < 0.25, "batches": 2 if api == "world" and rng.random() < 0.2 else 1}
        layout = float(experts) * ranks * tokens * hidden * case["batches"]
        state = layout * ((1 if fp8 else 2) + (2 if chain in ("expert", "cast") else 0))
        if work(case)["bytes"] <= _MOST_BYTES and state <= _MOST_STATE:
            return case


# ---------------------------------------------------------------------------


def _token_counts(case):
    R, T = case["ranks"], case["tokens"]
    if not case["ragged"]:
        return [T] * R
    # every rank between a third of the limit and the limit, one of them at it
    return [T - (r * 7 % (T - T // 3 or 1)) for r in range(R)]


def _config(case):
    return EPConfig("case", case["ranks"], case["tokens"], case["hidden"], case["experts"], case["topk"], case["fp8"],
                    routing=case["routing"], outlier_fraction=case["outliers"], masked_fraction=case["masked"])


def _route(case, rows, gen):
    """[rows, topk] distinct experts by Gumbel / Gaussian top-k: uniform, Zipf(1.2), or nine tokens in ten on an
    eighth of the experts."""
    E, K = case["experts"], case["topk"]
    u = torch.rand(rows, E, device="cuda", generator=gen).clamp_(min=1e-20)
    score = -torch.log(-torch.log(u))
    if case["routing"] == "zipf":
        score -= 1.2 * torch.log(torch.arange(1, E + 1, device="cuda", dtype=torch.float32))
    elif case["routing"] == "k_hot":
        hot = torch.rand(rows, 1, device="cuda", generator=gen) < 0.9
        score[:, :max(K, E // 8)] += 1e3 * hot
    return score.topk(K, dim=-1).indices.to(torch.int64)


def _inputs(case, gen):
    R, T, H, K = case["ranks"], case["tokens"], case["hidden"], case["topk"]
    x = torch.randn(R, T, H, device="cuda", generator=gen)
    if case["outliers"] > 0:
        x *= 1.0 + 99.0 * (torch.rand(R, T, 1, device="cuda", generator=gen) < case["outliers"])
    idx = _route(case, R * T, gen).view(R, T, K)
    weights = torch.randn(R, T, K, device="cuda", generator=gen).softmax(dim=-1)
    if case["masked"] > 0:
        idx[torch.rand(R, T, device="cuda", generator=gen) < case["masked"]] = -1
    return {"x": x.to(torch.bfloat16), "topk_idx": idx.contiguous(), "topk_weights": weights.contiguous()}


def _world_batch(case, gen):
    cfg = _config(case)
    h = WorldHarness(cfg, world=ep.default_world(cfg.num_ranks), num_tokens=_token_counts(case))
    h.load(_inputs(case, gen))
    h.alloc_dispatch_outputs()
    if case["chain"] == "expert":                      # the payload is an output
        h.recv_x.zero_()
        if case["fp8"]:
            h.recv_scales_phys.zero_()
    h.src_info.zero_()
    if case["chain"] == "identity":
        h.expert_out = h.recv_x.view(torch.bfloat16)
    h.alloc_combine_io()
    if case["chain"] == "expert":
        h.expert_out.normal_(generator=gen)
    h.combined.zero_()                                 # rows beyond a rank's tokens stay
    return h


def _buffer_state(case, gen):
    R, T, H, E = case["ranks"], case["tokens"], case["hidden"], case["experts"]
    world = ep.default_world(R)
    size = Buffer.get_ep_buffer_size_hint(T, H, R, E)
    data = _inputs(case, gen)
    n = _token_counts(case)
    state = {"world": world, "bufs": [Buffer(LogicalGroup(world, r), size) for r in range(R)],
             "x": [data["x"][r, :n[r]] for r in range(R)], "idx": [data["topk_idx"][r, :n[r]] for r in range(R)],
             "weights": [data["topk_weights"][r, :n[r]] for r in range(R)],
             "active": [torch.ones(R, dtype=torch.int32, device="cuda") for _ in range(R)]}
    if case["chain"] == "cast":
        rows = torch.empty(R, E // R, R * T, H, dtype=torch.bfloat16, device="cuda")
        state["rows"] = [rows[r] for r in range(R)]
    return state


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case, "factor": torch.rand(case["experts"], device="cuda", generator=gen) + 0.5}
    if case["api"] == "buffer":
        state.update(_buffer_state(case, gen))
    else:
        state["batches"] = [_world_batch(case, gen) for _ in range(case["batches"])]
    return state


def _run_world(state):
    chain = state["case"]["chain"]
    for h in state["batches"]:
        h.dispatch()
        if chain == "cast":
            h.cast_back(state["factor"])
    outputs = []
    for h in state["batches"]:
        if chain == "packed":
            h.combine_packed(state["factor"])
        else:
            h.combine()
        out = {"combined": h.combined, "count": h.recv_count, "src_info": h.src_info, "range": h.layout_range}
        if chain == "expert":
            out["payload"] = h.recv_x
            if h.recv_scales_phys is not None:
                out["scales"] = h.recv_scales_phys
        outputs.append(out)
    return outputs


def _run_buffer(state):
    case = state["case"]
    R, T, H, E, K, fp8 = (case[k] for k in ("ranks", "tokens", "hidden", "experts", "topk", "fp8"))
    bufs, x, idx, active = state["bufs"], state["x"], state["idx"], state["active"]
    sent = [bufs[r].dispatch(x[r], idx[r], active[r], T, E, -1, use_fp8=fp8, async_finish=True) for r in range(R)]
    for s in sent:
        s[3].current_stream_wait()
    if case["chain"] == "cast":
        rows = state["rows"]
        state["world"].cast_back([s[0][0].data_ptr() for s in sent], [s[0][1].data_ptr() for s in sent],
                                 [s[1].data_ptr() for s in sent], state["factor"].data_ptr(),
                                 [t.data_ptr() for t in rows], H, K, T, E,
                                 int(torch.cuda.current_stream().cuda_stream))
    else:
        rows = [s[0] for s in sent]
    done = [bufs[r].combine(rows[r], idx[r], state["weights"][r], active[r], -1, sent[r][2], async_finish=True)
            for r in range(R)]
    for d in done:
        d[1].current_stream_wait()
    return {"combined": [d[0] for d in done], "count": [s[1] for s in sent], "range": [s[2][1] for s in sent]}


def run(state):
    return _run_buffer(state) if state["case"]["api"] == "buffer" else _run_world(state)


def work(case):
    """Bytes of one pass.  Dispatch reads every token row and its indices and writes a payload row (and, fp8, its
    scales) and a source index per selection, a count and R ranges per expert; combine reads a row per selection and
    the routing of every token and writes the token rows; the mock expert on its own reads the payload and writes the
    bf16 rows combine then reads."""
    H, K, E, R = case["hidden"], case["topk"], case["experts"], case["ranks"]
    N = sum(_token_counts(case))
    S = N * K * (1.0 - case["masked"])
    payload = H + H // 128 * 4 if case["fp8"] else 2 * H
    total = N * H * 2 + N * K * 8 + S * (payload + 4) + E * 4 + E * R * 8
    if case["chain"] == "cast":
        total += S * (payload + 2 * H)
    total += S * (payload if case["chain"] == "packed" else 2 * H) + S * 4 + N * K * 12 + N * H * 2
    flops = 2 * S * H + (3 * N * H if case["fp8"] else 0) + (2 * S * H if case["chain"] in ("cast", "packed") else 0)
    return {"bytes": total * case["batches"], "flops": flops * case["batches"]}


def tolerance(case):
    # The contract is bit for bit: counts, slots, payload and scales, and combine's fused multiply-adds in k order.
    return "exact"
