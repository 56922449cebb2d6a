"""Workloads of one expert-parallel rank, as a program that uses this package runs them.

Three paths, each a whole step of a MoE layer between its router and its output, without the experts and the wire:

  step      deep_ep.Buffer.low_latency_dispatch + low_latency_combine: decode, and the batches past it
  exchange  the five calls of a step over an all-to-all shaped transport (ll_runtime.AllToAllState)
  prefill   the normal-mode steps: layout, FP8 cast, routing sort, channel prefix, pack, top-k remap, source
            metadata, and the reduce of the rows that come back

The other ranks' rows and answers are in HBM before a pass, where a transport would have put them.
"""
import math

import torch

import deep_ep
from deepep_efa_amd import deep_ep_cpp, ll_runtime, loopback, normal

_FORMATS = {"bf16": (False, False, False), "fp8": (True, False, False), "fp8_pow2": (True, True, False),
            "fp8_ue8m0": (True, True, True)}  # use_fp8, round_scale, use_ue8m0
_NUM_CHANNELS = 10  # Buffer.num_sms / 2


def _step(tokens, max_tokens, hidden, topk, experts, ranks, rank, fmt="fp8", popularity="uniform", masked=False,
          zero_copy=False, graph=False):
    return {"path": "step", "tokens": tokens, "max_tokens": max_tokens, "hidden": hidden, "topk": topk,
            "experts": experts, "ranks": ranks, "rank": rank, "fmt": fmt, "popularity": popularity, "masked": masked,
            "zero_copy": zero_copy, "graph": graph}


def _exchange(tokens, max_tokens, hidden, topk, experts, ranks, rank, fmt="fp8", masked=False):
    return {"path": "exchange", "tokens": tokens, "max_tokens": max_tokens, "hidden": hidden, "topk": topk,
            "experts": experts, "ranks": ranks, "rank": rank, "fmt": fmt, "popularity": "uniform", "masked": masked}


def _prefill(tokens, hidden, topk, experts, ranks, rank, fmt, masked=False):
    return {"path": "prefill", "tokens": tokens, "hidden": hidden, "topk": topk, "experts": experts, "ranks": ranks,
            "rank": rank, "fmt": fmt, "popularity": "uniform", "masked": masked}


def listed():
    return [
        # one sequence being decoded on this rank of a 32-rank group: nothing but latency
        dict(_step(1, 128, 7168, 8, 256, 32, 5), name="step_1"),
        # the headline decode step, called from Python layer by layer
        dict(_step(128, 128, 7168, 8, 256, 32, 5), name="step_128"),
        # the same step captured once and replayed, as a decode loop does
        dict(_step(128, 128, 7168, 8, 256, 32, 5, graph=True), name="step_128_graph"),
        # a ragged decode batch with padded selections, rows sent unquantised, 9 experts a rank
        dict(_step(77, 128, 5120, 6, 288, 32, 7, "bf16", masked=True), name="step_77_bf16"),
        # a chunked-prefill sized batch with power-of-two scale bytes, experts writing into the combine buffer
        dict(_step(509, 512, 4096, 8, 128, 16, 11, "fp8_ue8m0", zero_copy=True), name="step_509_ue8m0"),
        # a throughput batch: every phase bound by memory
        dict(_step(4096, 4096, 7168, 8, 64, 8, 3), name="step_4096"),
        # skewed routing seen by the rank that owns the hottest experts: some twenty times the balanced rows
        dict(_step(1000, 1024, 7168, 8, 256, 64, 0, popularity="zipf"), name="step_1000_skewed"),
        # decode over one contiguous message per peer
        dict(_exchange(128, 128, 7168, 8, 256, 32, 5), name="exchange_128"),
        # a throughput batch over the same transport
        dict(_exchange(2047, 2048, 7168, 8, 64, 8, 3), name="exchange_2047"),
        # a short prompt on a 16-rank, two-node group, rows sent as bf16
        dict(_prefill(131, 7168, 8, 256, 16, 3, "bf16", masked=True), name="prefill_131"),
        # the 4096-token layout + pack configuration, rows cast to FP8 before they are packed
        dict(_prefill(4096, 7168, 8, 256, 8, 2, "fp8"), name="prefill_4096_fp8"),
        # a long prompt batch
        dict(_prefill(12289, 7168, 8, 256, 8, 2, "bf16"), name="prefill_12289"),
    ]


def _spread(rng, low, high):
    return min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 0.49))))))


def draw(rng):
    path = rng.choice(["decode"] * 3 + ["batch"] * 2 + ["skewed"] + ["exchange"] * 2 + ["prefill"] * 2)
    hidden = rng.choice([2048, 4096, 5120, 7168])
    topk = rng.choice([4, 6, 8])
    masked = rng.random() < 0.3
    if path == "decode":  # up to 256 tokens: one launch per direction
        experts, ranks = rng.choice([(64, 8), (128, 16), (256, 16), (256, 32), (288, 32), (256, 64)])
        tokens = _spread(rng, 1, 256)
        return _step(tokens, 128 if tokens <= 128 else 256, hidden, topk, experts, ranks, rng.randrange(ranks),
                     rng.choice(["fp8", "fp8", "bf16", "fp8_pow2", "fp8_ue8m0"]), masked=masked,
                     zero_copy=rng.random() < 0.2, graph=rng.random() < 0.25)
    if path == "batch":  # chunked prefill and throughput batches
        experts, ranks = rng.choice([(64, 8), (64, 16), (32, 8)])
        tokens = _spread(rng, 257, 4096)
        return _step(tokens, (tokens + 63) // 64 * 64, hidden, topk, experts, ranks, rng.randrange(ranks),
                     rng.choice(["fp8", "fp8", "bf16", "fp8_pow2", "fp8_ue8m0"]), masked=masked,
                     zero_copy=rng.random() < 0.3)
    if path == "skewed":
        tokens = _spread(rng, 100, 1000)
        return _step(tokens, (tokens + 63) // 64 * 64, hidden, topk, 256, 64, rng.choice([0, 0, 1, 7]),
                     rng.choice(["fp8", "bf16"]), popularity="zipf", masked=masked)
    if path == "exchange":
        experts, ranks = rng.choice([(64, 8), (128, 16), (256, 32)])
        tokens = _spread(rng, 1, 2048 if ranks == 8 else 256)
        return _exchange(tokens, (tokens + 63) // 64 * 64, hidden, topk, experts, ranks, rng.randrange(ranks),
                         rng.choice(["fp8", "fp8", "bf16"]), masked)
    ranks = rng.choice([8, 8, 16, 32])
    return _prefill(_spread(rng, 64, 12000), hidden, topk, 256, ranks, rng.randrange(ranks),
                    rng.choice(["fp8", "bf16"]), masked)


def _world(case, seed, num_ranks, rank):
    """Every rank's tokens and routing, from the seed."""
    world = loopback.LoopbackWorld(num_ranks, rank, seed)
    world.synthesise(case["tokens"], case["hidden"], case["topk"], case["experts"], case["popularity"], 100)
    if case["masked"]:  # one selection in fifty is padding
        g = torch.Generator(device="cuda").manual_seed(seed + 1)
        topk = world.topk_idx_all
        topk[torch.rand(topk.shape, device="cuda", generator=g) < 0.02] = -1
    return world


def _weights(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed + 2)
    return torch.softmax(torch.randn((case["tokens"], case["topk"]), device="cuda", generator=g), dim=-1)


def _prepare_step(case, seed):
    ranks, rank, experts, max_tokens = case["ranks"], case["rank"], case["experts"], case["max_tokens"]
    fmt = _FORMATS[case["fmt"]]
    options = dict(use_fp8=fmt[0], round_scale=fmt[1], use_ue8m0=fmt[2])
    world = _world(case, seed, ranks, rank)
    x, topk_idx = (v.clone() for v in world.own_inputs())
    weights = _weights(case, seed)
    buffer = deep_ep.Buffer(None, low_latency_mode=True, num_qps_per_rank=experts // ranks, sim_num_ranks=ranks,
                            sim_rank=rank, sim_seed=seed)
    # the exchange: the peers' rows, and for the combine their experts' answers
    buffer.loopback_set_world(world.x_all, world.topk_idx_all)
    buffer.loopback_set_combine_mode(1, seed + 3)
    recv, count, handle, _, _ = buffer.low_latency_dispatch(x, topk_idx, max_tokens, experts, **options)
    g = torch.Generator(device="cuda").manual_seed(seed + 4)
    if case["zero_copy"]:
        y = buffer.get_next_low_latency_combine_buffer(handle)
    else:
        y = torch.empty((experts // ranks, ranks * max_tokens, case["hidden"]), dtype=torch.bfloat16, device="cuda")
    y.normal_(generator=g)  # what the experts computed
    combined, _, _ = buffer.low_latency_combine(y, topk_idx, weights, handle)
    torch.cuda.synchronize()
    buffer.loopback_clear_world()
    # rows past an expert's count are never written: give them a value
    for v in (*(recv if fmt[0] else (recv,)), count, handle[0], handle[1], combined):
        v.view(torch.uint8).zero_()
    state = {"path": "step", "buffer": buffer, "x": x, "topk_idx": topk_idx, "weights": weights, "y": y,
             "max_tokens": max_tokens, "experts": experts, "options": options, "zero_copy": case["zero_copy"]}
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _run_step(state)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outputs = _run_step(state)
        state["graph"], state["outputs"] = graph, outputs
    return state


def _run_step(s):
    recv, count, handle, _, _ = s["buffer"].low_latency_dispatch(s["x"], s["topk_idx"], s["max_tokens"], s["experts"],
                                                                 **s["options"])
    combined, _, _ = s["buffer"].low_latency_combine(s["y"], s["topk_idx"], s["weights"], handle,
                                                     zero_copy=s["zero_copy"])
    return recv, count, handle[0], handle[1], combined


def _prepare_exchange(case, seed):
    ranks, rank, experts, hidden = case["ranks"], case["rank"], case["experts"], case["hidden"]
    fmt = ll_runtime.row_format(*_FORMATS[case["fmt"]])
    world = _world(case, seed, ranks, rank)
    x, topk_idx = (v.clone() for v in world.own_inputs())

    def state_of(r):
        return ll_runtime.AllToAllState(ll_runtime.LLShape(ranks, r, experts, case["max_tokens"], hidden, case["topk"],
                                                           fmt))

    me = state_of(rank)
    for v in (me.send_rows, me.recv_by_source, me.packed_recv_x, me.packed_recv_src_info, me.send_flat,
              me.record_packed_row) + (() if me.packed_recv_scales is None else (me.packed_recv_scales,)):
        v.view(torch.uint8).zero_()  # rows past the counts are never written: give them a value
    # the exchange: every rank's message for this one, and the gathered route counts
    routed = []
    for r in range(ranks):
        peer = state_of(r)
        peer.dispatch_send(world.x_all[r], world.topk_idx_all[r])
        low, high = (int(v) for v in peer.send_cumsum[rank:rank + 2].cpu())
        me.recv_by_source[r * me.slot_rows:r * me.slot_rows + high - low] = peer.send_rows[low:high]
        routed.append(peer.send_count.clone())
        del peer
    routed = torch.stack(routed)
    per_rank = experts // ranks
    g = torch.Generator(device="cuda").manual_seed(seed + 4)
    me.recv_flat.normal_(generator=g)  # the peers' answers, one row per row sent
    y = torch.empty((per_rank, ranks * case["max_tokens"], hidden), dtype=torch.bfloat16, device="cuda")
    y.normal_(generator=g)
    return {"path": "exchange", "a2a": me, "x": x, "topk_idx": topk_idx, "weights": _weights(case, seed), "y": y,
            "routed": routed, "out": torch.empty((case["tokens"], hidden), dtype=torch.bfloat16, device="cuda")}


def _run_exchange(s):
    a2a = s["a2a"]
    a2a.dispatch_send(s["x"], s["topk_idx"])
    meta = a2a.exchange_metadata(s["routed"])
    a2a.dispatch_recv_ordered(s["routed"])
    a2a.combine_send(s["y"])
    a2a.combine_recv(s["topk_idx"], s["weights"], s["out"])
    return (a2a.send_rows, a2a.send_count, a2a.send_expert_prefix, a2a.send_counts, a2a.send_cumsum,
            meta["recv_counts"], meta["totals"], meta["combine_remote_recv_offset"], a2a.packed_recv_x,
            a2a.packed_recv_scales, a2a.packed_recv_count, a2a.packed_recv_src_info, a2a.packed_recv_layout_range,
            a2a.record_packed_row, a2a.send_flat, s["out"])


def _prefill_routing(case, seed):
    """One draw of the routing, its tokens in another order and its experts under other names for every seed (the
    experts of a rank stay together): the rows sent to the ranks change places but not their number."""
    ranks, experts = case["ranks"], case["experts"]
    topk_idx = _world(dict(case, hidden=128), 2024, 1, 0).topk_idx_all[0]
    g = torch.Generator(device="cuda").manual_seed(seed + 5)
    names = torch.arange(experts, device="cuda").view(ranks, -1)
    names = names[torch.randperm(ranks, device="cuda", generator=g)]
    names = names[:, torch.randperm(experts // ranks, device="cuda", generator=g)].reshape(-1)
    topk_idx = topk_idx[torch.randperm(topk_idx.shape[0], device="cuda", generator=g)]
    return torch.where(topk_idx >= 0, names[topk_idx.clamp(min=0)], topk_idx).contiguous()


def _prepare_prefill(case, seed):
    ranks, rank, experts = case["ranks"], case["rank"], case["experts"]
    x, _ = _world(case, seed, 1, 0).own_inputs()
    topk_idx = _prefill_routing(case, seed)
    weights = _weights(case, seed)
    buffer = deep_ep.Buffer(None, sim_num_ranks=ranks, sim_rank=rank, sim_seed=seed)
    _, _, _, is_in, _ = buffer.get_dispatch_layout(topk_idx, experts)
    _, counts, cumsum, total = normal.moe_routing_sort(is_in)
    g = torch.Generator(device="cuda").manual_seed(seed + 4)
    returned = torch.empty((total, case["hidden"]), dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    # what this rank receives: as many rows from each rank as it sends there
    return {"path": "prefill", "buffer": buffer, "x": x, "topk_idx": topk_idx, "weights": weights,
            "returned": returned, "experts": experts, "ranks": ranks, "fp8": case["fmt"] == "fp8",
            "recv_counts": counts, "recv_cumsum": cumsum, "recv_tokens": total}


def _run_prefill(s):
    ranks, topk_idx = s["ranks"], s["topk_idx"]
    per_rank, per_node, per_expert, is_in, _ = s["buffer"].get_dispatch_layout(topk_idx, s["experts"])
    rows, scales = deep_ep_cpp.per_token_cast_to_fp8(s["x"], False, False) if s["fp8"] else (s["x"], None)
    ids, counts, cumsum, total, row_of_pair = normal.moe_routing_sort_with_positions(is_in)
    channels = normal.channel_prefix_matrix(is_in, _NUM_CHANNELS)
    send_x, send_scales = normal.pack_rows(rows, scales, ids, cumsum)
    send_topk, send_weights = normal.topk_remap(topk_idx, s["weights"], ids, cumsum, total, ranks, s["experts"] // ranks)
    meta = normal.build_recv_src_meta(s["recv_counts"], s["recv_cumsum"], s["recv_tokens"], ranks, 8)
    combined, combined_weights = normal.combine_reduce(s["returned"], send_weights, ids, cumsum, is_in,
                                                       row_of_pair=row_of_pair)
    return (per_rank, per_node, per_expert, is_in, ids, counts, cumsum, total, row_of_pair, channels, send_x,
            send_scales, send_topk, send_weights, meta, combined, combined_weights)


def prepare(case, seed):
    return {"step": _prepare_step, "exchange": _prepare_exchange, "prefill": _prepare_prefill}[case["path"]](case, seed)


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    if state["path"] == "step":
        return _run_step(state)
    return _run_exchange(state) if state["path"] == "exchange" else _run_prefill(state)


def _routed_share(case):
    """Selections of a token that go to this rank's experts, and the ranks it goes to, on average."""
    experts, ranks, topk = case["experts"], case["ranks"], case["topk"]
    per_rank = experts // ranks
    popularity = [1.0 / (e + 1) ** 1.2 if case["popularity"] == "zipf" else 1.0 for e in range(experts)]
    low, high = 0.0, 1e9  # expert e is among the topk distinct ones with about 1 - exp(-rate * popularity)
    for _ in range(200):
        rate = (low + high) / 2
        if sum(1 - math.exp(-rate * p) for p in popularity) < topk:
            low = rate
        else:
            high = rate
    share = [(1 - math.exp(-low * p)) * (0.98 if case["masked"] else 1.0) for p in popularity]
    mine = sum(share[case["rank"] * per_rank:(case["rank"] + 1) * per_rank])
    reached = sum(1 - math.prod(1 - s for s in share[r * per_rank:(r + 1) * per_rank]) for r in range(ranks))
    return mine, reached


def work(case):
    t, h, k, e, ranks = case["tokens"], case["hidden"], case["topk"], case["experts"], case["ranks"]
    mine, reached = _routed_share(case)
    pairs = t * k * (0.98 if case["masked"] else 1.0)
    if case["path"] == "prefill":
        sent = t * reached
        row = h + h // 32 if case["fmt"] == "fp8" else 2 * h
        bytes_ = t * k * 12 + t * ranks * 5 + t * 2 * h + sent * (row + 8 + 12 * k + 8)  # dispatch side
        bytes_ += sent * 2 * h + t * 2 * h + t * k * 4  # the reduce
        return {"bytes": bytes_, "flops": sent * h}
    received = t * ranks * mine
    own = t * mine
    row = {"bf16": 2 * h, "fp8_ue8m0": h + h // 128}.get(case["fmt"], h + h // 32) + 16
    bytes_ = t * 2 * h + t * k * 12 + pairs * row + e * 4  # tokens in, a row out for each selection
    bytes_ += (received - (own if case["path"] == "step" else 0)) * 2 * row  # peers' rows into the packed tensors
    bytes_ += pairs * 2 * h + t * 2 * h + t * k * 16  # the weighted reduce
    if not case.get("zero_copy"):
        bytes_ += (received - (own if case["path"] == "step" else 0)) * 4 * h  # expert outputs back to their senders
    if case["path"] == "exchange":
        bytes_ += ranks * e * 4 + received * 20
    return {"bytes": bytes_, "flops": 2 * pairs * h}


def tolerance(case):
    """Quantised rows, scales, counts and indices are the same whoever computes them (the FP8 values and scales are
    covered by their own dtype's steps, far above `max`); sums of bf16 rows in float32 rounded once to bf16 may round
    the other way where their order differs."""
    return {"rel": 4e-3, "max": 2e-2, "differ": 0.0}
