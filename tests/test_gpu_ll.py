"""GPU parity of the low-latency dispatch + combine path, through the C ABI.

One GPU plays rank `rank` of an R-rank world; the other ranks' rows are put
in HBM by the loopback entry points.  Expected values come from the CPU
oracle restated from the reference.  Integer outputs, FP8 bytes and scales
must be bit-exact; the combine must match the float32 FMA-chain definition
bit for bit and the float64 sum within 1e-2 relative.
"""
import ctypes
import os
import re

import numpy as np
import pytest
import torch

from oracle import deepep_oracle as O
from tiny_world import load_tiny_world, tiny_world_expected

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from deepep_efa_amd import _capi, ll_runtime, loopback
    _capi.load()
    assert torch.cuda.is_available(), "these tests need the MI355X"

    class NS:
        pass

    ns = NS()
    ns.capi, ns.ll, ns.lb = _capi, ll_runtime, loopback
    return ns


def make_world(r, t, h, k, e, seed, drop=10, recipe="randn"):
    g = torch.Generator().manual_seed(seed)
    if recipe == "rank_const":  # tests/test_low_latency.py:59-60
        xs = []
        for rank in range(r):
            x = torch.ones((t, h), dtype=torch.bfloat16) * (rank - 128)
            x[:, -128:] = torch.arange(t).to(torch.bfloat16).view(-1, 1)
            xs.append(x)
        x_all = torch.stack(xs)
    else:
        x_all = torch.randn((r, t, h), generator=g).to(torch.bfloat16)
        x_all[:, ::9] *= 30
    scores = torch.rand((r, t, e), generator=g)
    topk = torch.topk(scores, k, dim=-1)[1].contiguous()
    for _ in range(drop):
        s, i, j = [int(torch.randint(0, n, (1,), generator=g)) for n in (r, t, k)]
        topk[s, i, j] = -1
    w = torch.randn((r, t, k), generator=g).abs()
    return x_all, topk, w


ONE_CALL = pytest.mark.parametrize("one_call", [False, True], ids=["two_calls", "one_call"])


def poison_outputs(st):
    """Fresh tensors may reuse memory that an earlier test left holding the right answer."""
    st.packed_recv_x.view(torch.uint8).fill_(0xEE)
    if st.packed_recv_scales is not None:
        st.packed_recv_scales.view(torch.uint8).fill_(0xEE)
    st.packed_recv_src_info.fill_(-7)
    st.packed_recv_count.fill_(-7)
    st.packed_recv_layout_range.fill_(-7)
    st.pair_slot.fill_(-7)


def run_dispatch(st, world, x, topk, stats=None, one_call=False):
    poison_outputs(st)
    if one_call:
        world.dispatch_from_peers(st)
        st.dispatch(x, topk, stats)
    else:
        st.dispatch_send(x, topk)
        world.dispatch_from_peers(st)
        st.dispatch_recv(stats)
    torch.cuda.synchronize()


def run_combine(st, world, y, topk, w, out, mode, seed=0, one_call=False):
    out.view(torch.int16).fill_(0x7FC0)  # NaN
    if one_call:
        world.combine_from_peers(st, mode=mode, seed=seed)
        st.combine(y, topk, w, out)
    else:
        world.combine_from_peers(st, mode=mode, seed=seed)
        st.combine_send(y)
        st.combine_recv(topk, w, out)
    torch.cuda.synchronize()


def dispatch_on_gpu(rt, x_all, topk_all, rank, e, m, fmt, stats=None, one_call=False):
    r, t, h = x_all.shape
    k = topk_all.shape[2]
    shape = rt.ll.LLShape(num_ranks=r, rank=rank, num_experts=e, max_tokens=m, hidden=h, num_topk=k, fmt=fmt)
    st = rt.ll.LowLatencyState(shape)
    world = rt.lb.LoopbackWorld(r, rank, seed=0)
    world.set_inputs(x_all.cuda(), topk_all.cuda())
    x, topk = world.own_inputs()
    run_dispatch(st, world, x, topk, stats, one_call)
    return st, world


def takes_one_launch(rt, st, t):
    """Whether a one-call dispatch of t tokens takes the single launch."""
    s = st.shape
    return rt.capi.load().deepep_ll_dispatch_takes_one_launch(t, s.hidden, s.num_topk, s.num_experts, s.max_tokens, s.fmt,
                                                              st.expected_rows) == 1


def kernels_launched(call, tmp_path):
    """The low-latency kernels of a call and their workgroups, by the nodes of a captured graph."""
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    graph.enable_debug_mode()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        call()
    graph.debug_dump(str(tmp_path / "graph.dot"))
    found = re.findall(r"(ll_[a-z_]*?kernel)[^\n(]*\((\d+),(\d+),(\d+)\)", (tmp_path / "graph.dot").read_text())
    return {name: int(x) * int(y) * int(z) for name, x, y, z in found}


def check_dispatch(st, want, fmt):
    count = st.packed_recv_count.cpu()
    assert torch.equal(count, want["packed_recv_count"])
    assert torch.equal(st.packed_recv_layout_range.cpu(), want["packed_recv_layout_range"])
    px = st.packed_recv_x.view(torch.uint8).view(want["packed_recv_x"].shape).cpu()
    src = st.packed_recv_src_info.cpu()
    ps = None if st.packed_recv_scales is None else \
        st.packed_recv_scales.view(torch.uint8).view(want["packed_recv_scales"].shape).cpu()
    for le in range(count.numel()):
        n = int(count[le])
        assert torch.equal(src[le, :n], want["packed_recv_src_info"][le, :n]), f"src_info expert {le}"
        assert torch.equal(px[le, :n], want["packed_recv_x"][le, :n]), f"payload bytes expert {le}"
        if ps is not None:
            assert torch.equal(ps[le, :n], want["packed_recv_scales"][le, :n]), f"scale bytes expert {le}"


@pytest.mark.parametrize("fmt", [O.ROW_FP8, O.ROW_BF16, O.ROW_FP8_POW2, O.ROW_FP8_UE8M0])
@pytest.mark.parametrize("r,rank,t,h,k,e", [
    (4, 1, 8, 512, 3, 16), (8, 7, 33, 1024, 4, 64), (2, 0, 1, 512, 1, 2),
    (4, 1, 40, 512, 9, 64),    # K > 8
    (2, 1, 600, 512, 8, 16),   # a mid-sized batch: the send side sweeps every earlier entry, in the single launch too
    (4, 3, 300, 512, 11, 32),  # both
    (2, 0, 1500, 512, 8, 16),  # more entries than one launch takes: chunk histograms ahead of the send, index kernel + flat row copy
    (8, 5, 4200, 512, 4, 64),  # the same on 8 ranks
    (8, 2, 20, 512, 4, 512),   # more than 256 segments: 16 counts per lane in the register segment table
    (16, 9, 12, 512, 6, 1024),  # the most experts the path takes
    (1, 0, 16, 512, 2, 4),     # a world of one rank: every row is the rank's own
    (4, 1, 12, 512, 2, 4),     # one expert per rank
    (2, 1, 9, 512, 64, 128),   # the most selections per token
    (4, 2, 24, 1536, 4, 16),   # hidden not a multiple of 1024: the last row piece is partly empty
    (8, 3, 17, 5120, 8, 64),
    (128, 77, 9, 512, 4, 128),   # many ranks, one expert each
    (256, 3, 5, 512, 2, 512),
    (512, 500, 3, 512, 2, 1024),  # the widest world the path takes
    (3, 1, 801, 512, 5, 9),    # odd entries a token and in all: the sweeps read them in pairs; 9 segments, not whole vectors
])
@ONE_CALL
def test_dispatch_small_worlds(rt, fmt, r, rank, t, h, k, e, one_call):
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=r * 100 + t, drop=min(5, t))
    st, _ = dispatch_on_gpu(rt, x_all, topk_all, rank, e, t, fmt, one_call=one_call)
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, fmt)
    check_dispatch(st, want, fmt)
    send_count, pair_slot = O.route(topk_all[rank], e, t)
    assert torch.equal(st.send_count.cpu(), send_count)
    assert torch.equal(st.pair_slot[:t].cpu(), pair_slot)


@pytest.mark.parametrize("rows", [1024, 1025])
@pytest.mark.parametrize("fmt,h", [(O.ROW_BF16, 2048), (O.ROW_BF16, 2176), (O.ROW_FP8, 4096), (O.ROW_FP8, 4224)])
@pytest.mark.parametrize("t,k", [(192, 8), (193, 8)])
def test_single_launch_dispatch_around_its_split_bounds(rt, rows, fmt, h, t, k):
    """Whole and split rows of 4096 bytes and just past it, expected rows and entries (1536) on both sides."""
    r, rank, e = 4, 2, 32
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=t + h, drop=20)
    shape = rt.ll.LLShape(num_ranks=r, rank=rank, num_experts=e, max_tokens=t, hidden=h, num_topk=k, fmt=fmt)
    st = rt.ll.LowLatencyState(shape)
    st.expected_rows = rows
    world = rt.lb.LoopbackWorld(r, rank, seed=0)
    world.set_inputs(x_all.cuda(), topk_all.cuda())
    run_dispatch(st, world, *world.own_inputs(), one_call=True)
    check_dispatch(st, O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, fmt), fmt)


@pytest.mark.parametrize("key,rank", [("rank0_ascending", 0), ("rank1_ascending", 1)])
@ONE_CALL
@pytest.mark.parametrize("fmt", [O.ROW_BF16, O.ROW_FP8])
def test_hand_derived_world(rt, key, rank, one_call, fmt):
    """The HIP path against values worked out on paper (tests/golden/ll_tiny_world.json): no oracle involved."""
    g, x_all, topk_all = load_tiny_world()
    e, m, h, t, k = g["num_experts"], g["max_tokens"], g["hidden"], g["num_tokens"], g["num_topk"]
    st, world = dispatch_on_gpu(rt, torch.stack(x_all), torch.stack(topk_all), rank, e, m, fmt, one_call=one_call)
    want, layout = tiny_world_expected(g, key)
    assert st.packed_recv_count.cpu().tolist() == want["count"]
    assert torch.equal(st.packed_recv_layout_range.cpu(), layout)
    for le, n in enumerate(want["count"]):
        assert st.packed_recv_src_info[le, :n].cpu().tolist() == want["src_info"][le]
        values = torch.tensor(want["row_value"][le], dtype=torch.float32)
        if fmt == O.ROW_BF16:
            assert torch.equal(st.packed_recv_x[le, :n].cpu().float(), values.view(-1, 1).expand(-1, h))
        else:
            assert (st.packed_recv_x[le, :n].view(torch.uint8).cpu() == g["fp8"]["payload_byte"]).all()
            assert torch.equal(st.packed_recv_scales[le, :n].cpu().view(-1), values / torch.tensor(448.0))
    if rank != 0:
        return
    assert st.send_count.cpu().tolist() == g["route_rank0"]["send_count"]
    assert st.pair_slot[:t].cpu().tolist() == g["route_rank0"]["pair_slot"]
    if fmt == O.ROW_BF16:  # identity experts: what comes back is what was sent
        y = st.packed_recv_x.clone()
        out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
        w = torch.tensor(g["topk_weights_rank0"], dtype=torch.float32, device="cuda")
        run_combine(st, world, y, topk_all[0].cuda(), w, out, mode=0, one_call=one_call)
        expect = torch.tensor(g["combine_rank0_identity_experts"]).view(-1, 1).expand(-1, h)
        assert torch.equal(out.cpu().float(), expect)


def check_exchange_metadata(got, want, capacity):
    assert got["send_counts"].cpu().tolist() == want["send_counts"].tolist()
    assert got["recv_counts"].cpu().tolist() == want["recv_counts"].tolist()
    assert got["totals"].cpu().tolist() == [want["total_send"], want["total_recv"], int(want["corrupt"])]
    assert got["combine_remote_recv_offset"].cpu().tolist() == want["combine_remote_recv_offset"].tolist()
    n = min(want["total_recv"], capacity)
    assert got["num_recv_tokens"].cpu().tolist() == [want["total_recv"], n]
    for key in ("source_rank", "source_offset", "padded_index", "combine_send_offset"):
        assert got[key][:n].cpu().tolist() == want[key][:n].tolist(), key
        assert (got[key][n:] == -7).all(), key  # nothing written past the records
    assert (got["tokens_per_expert"] == 0).all()


@pytest.mark.parametrize("r,e,m,k,rank,capacity", [(2, 4, 3, 2, 1, 16), (6, 24, 40, 5, 4, 400), (32, 256, 128, 8, 5, 4096),
                                                   (64, 256, 8192, 8, 63, 70000), (8, 64, 300, 6, 0, 100),
                                                   (1, 4, 9, 2, 0, 32), (160, 160, 20, 3, 77, 64)])
def test_exchange_metadata(rt, r, e, m, k, rank, capacity):
    """Counts, combine offsets and row records from the gathered route counts, against the reference's host loops."""
    g = torch.Generator().manual_seed(r * 7 + e)
    if r * m <= 4096:
        topk_all = [torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(m)]) for _ in range(r)]
        routed = torch.stack([O.route(tk, e, m)[0] for tk in topk_all]).to(torch.int32)
    else:  # any matrix of plausible counts will do
        routed = torch.randint(0, min(m, 60) + 1, (r, e), generator=g, dtype=torch.int32)
    for name, mat in (("clean", routed), ("corrupt", routed.clone())):
        if name == "corrupt":
            mat[r // 2, e // 3] = m + 1
        got = {}
        out = rt.ll.exchange_metadata(mat.cuda(), rank, m, capacity)
        torch.cuda.synchronize()
        want = O.ll_exchange_metadata(mat, rank, m)
        assert want["corrupt"] == (name == "corrupt")
        # poison-free check of "nothing written past the records": run again into pre-filled buffers
        for key in ("source_rank", "source_offset", "padded_index", "combine_send_offset"):
            got[key] = torch.full((capacity,), -7, dtype=torch.int32, device="cuda")
        lib, capi = rt.capi.load(), rt.capi
        for key in ("send_counts", "recv_counts", "totals", "combine_remote_recv_offset", "num_recv_tokens",
                    "tokens_per_expert"):
            got[key] = torch.full_like(out[key], -7)
        capi.check(lib.deepep_ll_exchange_metadata(
            capi.ptr(mat.cuda()), e, r, rank, m, capacity, capi.ptr(got["send_counts"]), capi.ptr(got["recv_counts"]),
            capi.ptr(got["totals"]), capi.ptr(got["combine_remote_recv_offset"]), capi.ptr(got["source_rank"]),
            capi.ptr(got["source_offset"]), capi.ptr(got["padded_index"]), capi.ptr(got["combine_send_offset"]),
            capi.ptr(got["num_recv_tokens"]), capi.ptr(got["tokens_per_expert"]),
            torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        check_exchange_metadata(got, want, capacity)
        for key in got:
            n = min(want["total_recv"], capacity) if got[key].numel() == capacity else got[key].numel()
            assert torch.equal(out[key][:n], got[key][:n]), key


@pytest.mark.parametrize("r,e,rank,capacity", [(1, 1, 0, 8), (1, 7, 0, 0), (3, 9, 2, 300), (2, 10, 1, 40), (5, 255, 4, 2100),
                                               (7, 259, 3, 2049), (32, 256, 31, 4096), (4, 2048, 3, 70000),
                                               (64, 1024, 1, 300000), (300, 300, 299, 500), (1024, 1024, 700, 20000),
                                               (2, 128, 1, 900), (1, 320, 0, 2000), (3, 576, 1, 700), (5, 480, 2, 700)])
def test_exchange_metadata_of_every_count(rt, r, e, rank, capacity):
    """Lists of counts that end within a vector, pass a workgroup's loads, or name more experts than it has threads:
    every count is added up, and one too large anywhere is seen."""
    g = torch.Generator().manual_seed(r * 1000 + e)
    m = 9
    routed = torch.randint(0, m + 1, (r, e), generator=g, dtype=torch.int32)
    routed[torch.rand((r, e), generator=g) > 8 * r / e] = 0  # no more in all than is possible
    spots = [None, (0, 0), (r - 1, e - 1), (r // 2, e // 2), (r - 1, max(0, e - 2))]
    for spot in spots:
        mat = routed.clone()
        if spot is not None:
            mat[spot] = m + 1 if spot != (0, 0) else -5  # -5: 2^32 - 5 as the count that it is read as
        want = O.ll_exchange_metadata(mat, rank, m)
        out = rt.ll.exchange_metadata(mat.cuda(), rank, m, capacity)
        torch.cuda.synchronize()
        assert out["totals"].cpu().tolist() == [want["total_send"], want["total_recv"], int(spot is not None)]
        assert out["send_counts"].cpu().tolist() == want["send_counts"].tolist()
        assert out["recv_counts"].cpu().tolist() == want["recv_counts"].tolist()
        first = rank * (e // r)
        assert out["combine_remote_recv_offset"].cpu().tolist() == (mat[:, :first].long() & 0xffffffff).sum(1).tolist()
        n = min(want["total_recv"], capacity)
        assert out["num_recv_tokens"].cpu().tolist() == [want["total_recv"], n]
        assert (out["tokens_per_expert"] == 0).all()
        for key in ("source_rank", "source_offset", "padded_index", "combine_send_offset"):
            assert out[key][:n].cpu().tolist() == want[key][:n].tolist(), key


@pytest.mark.parametrize("capacity,record_blocks", [(0, 0), (1024, 1), (1025, 2), (262144, 256), (300000, 256)])
@pytest.mark.filterwarnings("ignore:DEBUG")  # the graph is written out
def test_exchange_metadata_workgroups(rt, capacity, record_blocks, tmp_path):
    """A workgroup for every 1024 records there is room for, up to 256: full to the last record."""
    r, e, rank, m = 6, 48, 4, 8192
    routed = torch.randint(5000, 6300, (r, e), generator=torch.Generator().manual_seed(capacity), dtype=torch.int32)
    dev, lib, capi = routed.cuda(), rt.capi.load(), rt.capi
    out = {name: torch.full((max(1, n),), -7, dtype=torch.int64 if name == "combine_remote_recv_offset" else torch.int32, device="cuda")
           for name, n in (("send_counts", r), ("recv_counts", r), ("totals", 3), ("combine_remote_recv_offset", r),
                           ("source_rank", capacity), ("source_offset", capacity), ("padded_index", capacity),
                           ("combine_send_offset", capacity), ("num_recv_tokens", 2), ("tokens_per_expert", e // r))}

    def call():
        capi.check(lib.deepep_ll_exchange_metadata(capi.ptr(dev), e, r, rank, m, capacity, *(capi.ptr(v) for v in out.values()),
                                                   torch.cuda.current_stream().cuda_stream))

    assert kernels_launched(call, tmp_path) == {"ll_exchange_meta_kernel": 1 + 2 + record_blocks}
    call()
    torch.cuda.synchronize()
    want = O.ll_exchange_metadata(routed, rank, m)
    n = min(want["total_recv"], capacity)
    assert n == min(capacity, int(routed[:, rank * (e // r):(rank + 1) * (e // r)].sum()))
    assert out["num_recv_tokens"].cpu().tolist() == [want["total_recv"], n]
    for key in ("source_rank", "source_offset", "padded_index", "combine_send_offset"):
        assert torch.equal(out[key][:n].cpu().long(), torch.as_tensor(want[key][:n]).long()), key
        assert (out[key][n:] == -7).all()


def test_exchange_metadata_hand_derived_world(rt):
    g, _, _ = load_tiny_world()
    routed = torch.tensor(g["all_num_routed"], dtype=torch.int32)
    for rank in (0, 1):
        out = rt.ll.exchange_metadata(routed.cuda(), rank, g["max_tokens"], 8)
        torch.cuda.synchronize()
        want = g["exchange_metadata"][f"rank{rank}"]
        n = want["total_recv"]
        assert out["send_counts"].cpu().tolist() == want["send_counts"]
        assert out["recv_counts"].cpu().tolist() == want["recv_counts"]
        assert out["totals"].cpu().tolist() == [want["total_send"], n, 0]
        assert out["combine_remote_recv_offset"].cpu().tolist() == want["combine_remote_recv_offset"]
        assert out["num_recv_tokens"].cpu().tolist() == [n, n]
        for key in ("source_rank", "source_offset", "padded_index", "combine_send_offset"):
            assert out[key][:n].cpu().tolist() == want[key], key


def rows_by_source(x_all, topk_all, rank, e, m, fmt, slot_rows):
    """What an all-to-all leaves on rank `rank`: for every source s, the rows it sends to this rank's experts,
    in the sender's (token, k) order, at the start of slot s of one buffer (rows past the slot are lost)."""
    r, _, h = x_all.shape
    epr = e // r
    stride = O.row_stride(h, fmt)
    buf = torch.full((r * slot_rows, stride), 0xEE, dtype=torch.uint8)
    for s in range(r):
        _, _, experts, _, rows = O.staged_rows(x_all[s], topk_all[s], s, e, m, fmt, r)
        mine = rows[(experts // epr) == rank][:slot_rows]
        buf[s * slot_rows:s * slot_rows + mine.shape[0]] = mine
    return buf


def recv_by_source_on_gpu(rt, buf, routed, rank, e, m, h, fmt, slot_rows, capacity):
    """The exchange-metadata records for `routed`, then the receive side fed from the per-source buffer."""
    lib, capi = rt.capi.load(), rt.capi
    r = routed.shape[0]
    meta = rt.ll.exchange_metadata(routed.cuda(), rank, slot_rows, capacity)
    shape = rt.ll.LLShape(num_ranks=r, rank=rank, num_experts=e, max_tokens=m, hidden=h, num_topk=1, fmt=fmt)
    st = rt.ll.LowLatencyState(shape, keep_remote_rows=False)
    poison_outputs(st)
    ws = torch.empty(lib.deepep_ll_by_source_workspace_bytes(e, capacity), dtype=torch.uint8, device="cuda")
    tokens_per_expert = torch.full((e // r,), 77, dtype=torch.int32, device="cuda")
    dev = buf.cuda()
    capi.check(lib.deepep_ll_dispatch_recv_by_source(
        capi.ptr(dev), slot_rows, capi.ptr(meta["recv_counts"]), capi.ptr(meta["source_offset"]),
        capi.ptr(meta["num_recv_tokens"]), capacity, h, e, r, m, fmt, capi.ptr(st.packed_recv_x),
        capi.ptr(st.packed_recv_scales), capi.ptr(st.packed_recv_src_info), capi.ptr(st.packed_recv_layout_range),
        capi.ptr(st.packed_recv_count), None, capi.ptr(tokens_per_expert), None, 0, capi.ptr(ws), ws.numel(),
        torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return st, tokens_per_expert, meta


@pytest.mark.parametrize("fmt", [O.ROW_FP8, O.ROW_BF16, O.ROW_FP8_UE8M0])
@pytest.mark.parametrize("r,rank,t,h,k,e", [
    (4, 1, 8, 512, 3, 16), (8, 7, 33, 1024, 4, 64), (2, 0, 1, 512, 1, 2),
    (32, 5, 128, 7168, 8, 256),   # the headline shape
    (8, 3, 700, 512, 8, 256),     # past 4096 records: chunk histograms, sources of two chunks each
    (4, 1, 900, 512, 4, 16),      # up to 4096 records: one workgroup per source walks its two chunks, running counts
    (16, 2, 1200, 512, 8, 64),    # 9600 records in chunks of 512, about 600 per source
    (16, 5, 4096, 512, 8, 64),    # 32768 records: four chunks per source, 80 chunk workgroups
    (1, 0, 16, 512, 2, 4),        # a world of one rank
    (4, 2, 64, 512, 2, 4),        # one expert per rank
    (2, 1, 40, 512, 6, 2048),     # 1024 local experts: ten bits of expert id
])
def test_dispatch_recv_by_source(rt, fmt, r, rank, t, h, k, e):
    """Rows delivered grouped by source rank + the exchange-metadata records give the packed outputs of
    the staged receive, i.e. the same oracle outputs (csrc/kernels/efa_kernels.cu:877-1052,1227-1389)."""
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=r * 31 + t, drop=min(5, t))
    m = t
    slot_rows = t * min(k, e // r)  # the most one source can send to one rank
    buf = rows_by_source(x_all, topk_all, rank, e, m, fmt, slot_rows)
    routed = torch.stack([O.route(topk_all[s], e, m)[0] for s in range(r)]).to(torch.int32)
    capacity = int(routed[:, rank * (e // r):(rank + 1) * (e // r)].sum()) + 5
    st, tokens_per_expert, meta = recv_by_source_on_gpu(rt, buf, routed, rank, e, m, h, fmt, slot_rows, capacity)
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, m, fmt)
    check_dispatch(st, want, fmt)
    assert torch.equal(tokens_per_expert.cpu(), want["packed_recv_count"])
    assert int(meta["num_recv_tokens"][0]) == int(want["packed_recv_count"].sum())


@pytest.mark.parametrize("seed", range(int(os.environ.get("DEEPEP_TEST_RANDOM_SHAPES", "24"))))
def test_dispatch_recv_by_source_seeded_random_shapes(rt, seed):
    """The by-source receive on shapes nobody picked by hand, on both sides of its 4096-record bound."""
    r, rank, t, _, h, k, e, fmt, drop = _random_shape(seed)
    if seed % 3 == 0:
        t = t * 7  # more records: sources of several chunks
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=2000 + seed, drop=drop)
    m = t
    slot_rows = t * min(k, e // r)
    buf = rows_by_source(x_all, topk_all, rank, e, m, fmt, slot_rows)
    routed = torch.stack([O.route(topk_all[s], e, m)[0] for s in range(r)]).to(torch.int32)
    capacity = int(routed[:, rank * (e // r):(rank + 1) * (e // r)].sum()) + seed % 4
    st, tokens_per_expert, meta = recv_by_source_on_gpu(rt, buf, routed, rank, e, m, h, fmt, slot_rows, capacity)
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, m, fmt)
    check_dispatch(st, want, fmt)
    assert torch.equal(tokens_per_expert.cpu(), want["packed_recv_count"])


@pytest.mark.parametrize("t", [24, 1500], ids=["one_workgroup_per_source", "chunked"])
def test_dispatch_recv_by_source_drops_what_does_not_fit(rt, t):
    """A slot of M rows per source, as the reference sizes it (csrc/transport/ll_pipeline.cpp:1527): rows a
    source sends beyond it are lost, the others land as if the lost ones had not been sent; and with fewer
    record slots than rows, only the rows that have a record are received."""
    r, rank, h, k, e, fmt = 2, 0, 512, 4, 8, O.ROW_FP8
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=3, drop=0)
    topk_all[1, :, :] = torch.tensor([0, 1, 2, 3])  # every token of source 1 names all of rank 0's experts
    slot_rows = t  # source 1 sends 4 * t rows
    buf = rows_by_source(x_all, topk_all, rank, e, t, fmt, slot_rows)
    routed = torch.stack([O.route(topk_all[s], e, t)[0] for s in range(r)]).to(torch.int32)
    for capacity in (4 * t * r, t // 2 + 3):
        st, _, meta = recv_by_source_on_gpu(rt, buf, routed, rank, e, t, h, fmt, slot_rows, capacity)
        recv_counts = meta["recv_counts"].cpu().tolist()
        # expected: walk the records the way the kernel may use them
        epr, n = e // r, 0
        want_rows = [[[] for _ in range(r)] for _ in range(epr)]
        tail_at = O.row_payload(h, fmt) - 16
        tail = buf[:, tail_at:tail_at + 16].contiguous().view(torch.int32)
        for s in range(r):
            for j in range(recv_counts[s]):
                if n < capacity and j < slot_rows:
                    row = s * slot_rows + j
                    want_rows[int(tail[row, 3])][s].append(row)
                n += 1
        count = st.packed_recv_count.cpu().tolist()
        layout = st.packed_recv_layout_range.cpu()
        px = st.packed_recv_x.view(torch.uint8).cpu()
        for le in range(epr):
            begin = 0
            for s in range(r):
                rows = want_rows[le][s]
                assert int(layout[le, s]) == (((begin << 32) | len(rows)) if rows else 0), (capacity, le, s)
                if rows:
                    idx = torch.tensor(rows)
                    assert torch.equal(px[le, begin:begin + len(rows)], buf[idx, :h])
                    assert torch.equal(st.packed_recv_src_info[le, begin:begin + len(rows)].cpu(), tail[idx, 0])
                begin += len(rows)
            assert count[le] == begin


def _random_shape(seed):
    g = np.random.default_rng(seed)
    r = int(g.choice([1, 2, 3, 4, 5, 6, 8, 12, 16, 24]))
    epr = int(g.choice([1, 2, 3, 5, 8, 16]))
    e = r * epr
    k = int(g.integers(1, min(e, 12) + 1))
    t = int(g.choice([1, 2, 7, 31, 64, 100, 129, 257, 300, 1100]))
    m = t + int(g.choice([0, 0, 1, 13, 64]))  # room for more tokens than the batch holds
    h = int(g.choice([128, 256, 384, 640, 1024, 2048, 2176]))
    fmt = int(g.choice([O.ROW_FP8, O.ROW_BF16, O.ROW_FP8_POW2]))
    rank, drop = int(g.integers(0, r)), int(g.integers(0, min(40, t * k) + 1))
    if h % 512 == 0 and int(g.integers(0, 3)) == 0:
        fmt = O.ROW_FP8_UE8M0  # packed exponent bytes need whole groups of four scales
    return r, rank, t, m, h, k, e, fmt, drop


@pytest.mark.parametrize("seed", range(int(os.environ.get("DEEPEP_TEST_RANDOM_SHAPES", "24"))))
@ONE_CALL
def test_dispatch_and_combine_seeded_random_shapes(rt, seed, one_call):
    """Shapes nobody picked by hand: odd world sizes, hidden sizes with a ragged last piece, more slots
    than tokens, many or no dropped selections.  Dispatch bit-exact, combine against the float32 chain."""
    r, rank, t, m, h, k, e, fmt, drop = _random_shape(seed)
    x_all, topk_all, w_all = make_world(r, t, h, k, e, seed=1000 + seed, drop=drop)
    st, world = dispatch_on_gpu(rt, x_all, topk_all, rank, e, m, fmt, one_call=one_call)
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, m, fmt)
    check_dispatch(st, want, fmt)
    send_count, pair_slot = O.route(topk_all[rank], e, m)
    assert torch.equal(st.send_count.cpu(), send_count)
    assert torch.equal(st.pair_slot[:t].cpu(), pair_slot)
    # combine with the identity expert: every pair returns the row it was sent, so out = x * sum of weights
    epr = e // r
    y = torch.zeros((epr, r * m, h), dtype=torch.bfloat16)
    count = st.packed_recv_count.cpu()
    for le in range(epr):
        n = int(count[le])
        if fmt == O.ROW_BF16:
            y[le, :n] = st.packed_recv_x[le, :n].cpu()
        else:
            y[le, :n] = O.per_token_cast_back(st.packed_recv_x[le, :n].cpu(), st.packed_recv_scales[le, :n].cpu())
    out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
    run_combine(st, world, y.cuda(), topk_all[rank].cuda(), w_all[rank].cuda(), out, mode=0, one_call=one_call)
    wsum = w_all[rank].masked_fill(topk_all[rank] == -1, 0).sum(1).view(-1, 1)
    expect = x_all[rank].float() * wsum
    got = out.cpu().float()
    assert torch.isnan(got).sum().item() == 0
    live = wsum.view(-1) > 0
    assert (got[~live] == 0).all()  # a token with no valid selection combines to zero
    if live.any():
        diff = O.calc_diff(expect[live], got[live])
        assert diff < (2e-3 if fmt != O.ROW_BF16 else 1e-4), (diff, (r, rank, t, m, h, k, e, fmt))


def test_dispatch_send_staging_and_send_slots(rt):
    """The send side alone: own rows for own experts land in recv_staging, the rest in send_slots."""
    r, rank, t, h, k, e, m = 4, 2, 20, 512, 4, 32, 24
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=5, drop=6)
    shape = rt.ll.LLShape(r, rank, e, m, h, k, O.ROW_FP8)
    st = rt.ll.LowLatencyState(shape)
    st.recv_staging.fill_(0xAB)
    st.send_slots.fill_(0xCD)
    st.dispatch_send(x_all[rank].cuda(), topk_all[rank].cuda())
    torch.cuda.synchronize()
    send_count, pair_slot, experts, slots, rows = O.staged_rows(x_all[rank], topk_all[rank], rank, e, m, O.ROW_FP8, r)
    assert torch.equal(st.send_count.cpu(), send_count)
    assert torch.equal(st.pair_slot[:t].cpu(), pair_slot)
    stride = st.stride
    staging = st.recv_staging.cpu().view(e // r, r, m, stride)
    sendbuf = st.send_slots.cpu().view(e, m, stride)
    epr = e // r
    touched_stage = torch.zeros((epr, r, m), dtype=torch.bool)
    touched_send = torch.zeros((e, m), dtype=torch.bool)
    payload = O.row_payload(h, O.ROW_FP8)
    assert stride == O.row_stride(h, O.ROW_FP8) == 640 and payload == 544  # a row takes whole 128-byte lines
    for i in range(rows.shape[0]):
        ex, sl = int(experts[i]), int(slots[i])
        if ex // epr == rank:
            got, fill = staging[ex % epr, rank, sl], 0xAB
            touched_stage[ex % epr, rank, sl] = True
        else:
            got, fill = sendbuf[ex, sl], 0xCD
            touched_send[ex, sl] = True
        assert torch.equal(got[:payload], rows[i, :payload])
        assert (got[payload:] == fill).all()  # nothing is written behind the tail
    assert (staging[~touched_stage] == 0xAB).all() and (sendbuf[~touched_send] == 0xCD).all()
    rc = st.recv_count.cpu().view(epr, r)
    assert torch.equal(rc[:, rank], send_count[rank * epr:(rank + 1) * epr])
    assert (rc[:, [s for s in range(r) if s != rank]] == 0).all()


@ONE_CALL
@pytest.mark.parametrize("use_fp8", [True, False])
def test_reference_recipe_roundtrip(rt, use_fp8, one_call):
    """tests/test_low_latency.py:59-60,113-147,181-184 on one rank of an 8-rank world."""
    r, rank, t, h, k, e = 8, 3, 64, 2048, 6, 64
    fmt = O.ROW_FP8 if use_fp8 else O.ROW_BF16
    x_all, topk_all, w_all = make_world(r, t, h, k, e, seed=77, drop=10, recipe="rank_const")
    stats = torch.zeros(e // r, dtype=torch.int32, device="cuda")
    st, world = dispatch_on_gpu(rt, x_all, topk_all, rank, e, t, fmt, stats, one_call=one_call)
    epr = e // r
    count = st.packed_recv_count.cpu()
    lr_all = st.packed_recv_layout_range.cpu()
    assert torch.equal(stats.cpu(), count)
    for i in range(epr):
        expert = rank * epr + i
        n = int(count[i])
        lr = lr_all[i]
        assert n == int((lr & 0xFFFFFFFF).sum()) == int((topk_all == expert).sum())
        if n == 0:
            continue
        if use_fp8:
            recv = O.per_token_cast_back(st.packed_recv_x[i, :n].cpu(), st.packed_recv_scales[i, :n].cpu()).float()
        else:
            recv = st.packed_recv_x[i, :n].cpu().float()
        src = st.packed_recv_src_info[i, :n].cpu()
        assert torch.equal(recv[:, :-128].amin(-1), recv[:, :-128].amax(-1))
        assert (recv[:, -128:] - src.view(-1, 1) % t).sum().item() == 0
        for j in range(r):
            begin, cnt = int(lr[j] >> 32), int(lr[j] & 0xFFFFFFFF)
            assert int((recv[:, :-128].amin(-1) == j - 128).sum()) == int((topk_all[j] == expert).sum())
            assert (recv[begin:begin + cnt, :-128] - j + 128).sum().item() == 0
    # combine with an identity expert (simulated_gemm_x = dequantised recv)
    if use_fp8:
        el, n_slots = st.packed_recv_x.shape[:2]
        q = st.packed_recv_x.view(-1, h).cpu()
        sc = st.packed_recv_scales.view(-1, h // 128).cpu()
        live = torch.zeros((el, n_slots), dtype=torch.bool)
        for i in range(el):
            live[i, :int(count[i])] = True
        y = torch.zeros((el * n_slots, h), dtype=torch.bfloat16)
        y[live.view(-1)] = O.per_token_cast_back(q[live.view(-1)], sc[live.view(-1)])
        y = y.view(el, n_slots, h).cuda()
    else:
        y = st.packed_recv_x.clone()
    out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
    topk, w = topk_all[rank].cuda(), w_all[rank].cuda()
    run_combine(st, world, y, topk, w, out, mode=0, one_call=one_call)
    x = x_all[rank]
    wsum = w_all[rank].masked_fill(topk_all[rank] == -1, 0).sum(1).view(-1, 1)
    diff = O.calc_diff(x.float() * wsum, out.cpu())
    assert torch.isnan(out.float()).sum().item() == 0
    assert diff < (9e-4 if use_fp8 else 1e-5), diff


@pytest.mark.parametrize("r,rank,t,h,k,e", [(32, 5, 128, 7168, 8, 256), (4, 0, 16, 512, 3, 8),
                                            (8, 3, 4200, 512, 4, 64),   # large-batch combine-send path
                                            (8, 3, 1024, 4096, 8, 64),  # the largest single launch: moves > 192 MB, so it streams
                                            (4, 2, 40, 512, 11, 64),    # more than eight selections per token
                                            (8, 6, 20, 512, 4, 512),    # more than 256 segments
                                            (4, 1, 33, 1536, 5, 32),    # hidden not a multiple of 512
                                            (128, 77, 9, 512, 4, 128),  # many ranks, one expert each
                                            (512, 500, 3, 512, 2, 1024)])
@ONE_CALL
def test_combine_random_expert_outputs(rt, oracle_c, r, rank, t, h, k, e, one_call):
    """Seeded expert outputs along the dispatch routing; combine vs the float32 chain and the float64 sum."""
    x_all, topk_all, w_all = make_world(r, t, h, k, e, seed=31 + r, drop=10)
    st, world = dispatch_on_gpu(rt, x_all, topk_all, rank, e, t, O.ROW_FP8, one_call=one_call)
    epr, n_slots, lib, capi = e // r, r * t, rt.capi.load(), rt.capi
    seed_local, seed_remote = 1234, 4321
    # local experts' outputs: row key = local_expert * N + slot
    y = torch.zeros((epr, n_slots, h), dtype=torch.bfloat16, device="cuda")
    capi.check(lib.deepep_synth_bf16_rows(capi.ptr(y), epr * n_slots, h, h * 2, None, 0, seed_local, 0,
                                          torch.cuda.current_stream().cuda_stream))
    out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
    run_combine(st, world, y, topk_all[rank].cuda(), w_all[rank].cuda(), out, mode=1, seed=seed_remote,
                one_call=one_call)
    # oracle: which row does each of this rank's pairs get back?
    topk, w = topk_all[rank], w_all[rank]
    _, pair_slot = O.route(topk, e, t)
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, O.ROW_FP8)
    keys_local, keys_remote = [], []
    pair_rows = torch.zeros((t, k, h), dtype=torch.bfloat16)
    live = pair_slot >= 0
    idx_local, idx_remote = [], []
    for ti in range(t):
        for ki in range(k):
            if not live[ti, ki]:
                continue
            ex, sl = int(topk[ti, ki]), int(pair_slot[ti, ki])
            if ex // epr == rank:
                begin = int(want["packed_recv_layout_range"][ex % epr, rank] >> 32)
                keys_local.append((ex % epr) * n_slots + begin + sl)
                idx_local.append((ti, ki))
            else:
                keys_remote.append(ex * t + sl)
                idx_remote.append((ti, ki))
    if idx_local:
        rows = O.synth_bf16_rows(np.array(keys_local, dtype=np.uint32), h, seed_local)
        ii = torch.tensor(idx_local)
        pair_rows[ii[:, 0], ii[:, 1]] = rows
    if idx_remote:
        rows = O.synth_bf16_rows(np.array(keys_remote, dtype=np.uint32), h, seed_remote)
        ii = torch.tensor(idx_remote)
        pair_rows[ii[:, 0], ii[:, 1]] = rows
    chain = torch.empty((t, h), dtype=torch.int16)
    live8 = live.to(torch.uint8).contiguous()
    oracle_c.oracle_combine_chain(ctypes.c_void_p(pair_rows.view(torch.int16).data_ptr()),
                                  ctypes.c_void_p(w.contiguous().data_ptr()), ctypes.c_void_p(live8.data_ptr()), t, k,
                                  h, ctypes.c_void_p(chain.data_ptr()))
    got = out.cpu()
    assert torch.equal(got.view(torch.int16), chain), "combine differs from the float32 FMA chain"
    # accumulate: the sum starts from what `out` holds (csrc/kernels/coop_combine_recv.cuh:174-179)
    prev = torch.randn((t, h), generator=torch.Generator().manual_seed(3)).to(torch.bfloat16)
    out2 = prev.cuda()
    if one_call:
        st.combine(y, topk_all[rank].cuda(), w_all[rank].cuda(), out2, accumulate=True)
    else:
        st.combine_recv(topk_all[rank].cuda(), w_all[rank].cuda(), out2, accumulate=True)
    torch.cuda.synchronize()
    want2 = O.ll_combine_f32_chain(pair_rows, w, live, initial=prev)
    assert torch.equal(out2.cpu().view(torch.int16), want2.view(torch.int16)), "accumulating combine"
    ref = O.ll_combine(pair_rows, topk, w, live)
    err = (got.double() - ref).abs()
    assert (err <= 1e-2 * ref.abs() + 1e-2 * ref.abs().mean()).all()
    assert O.calc_diff(got, ref) < 1e-5


def bf16_bits_of(x):
    """float32 -> bf16 bits by integer arithmetic, to nearest with ties to even; any NaN as 0x7FC0."""
    b = x.contiguous().view(torch.int32).long() & 0xFFFFFFFF
    r = (b + 0x7FFF + ((b >> 16) & 1)) >> 16
    return torch.where(x.isnan(), torch.full_like(r, 0x7FC0), r).int()


def bf16_bits(x):
    return torch.where(x.isnan(), torch.full(x.shape, 0x7FC0, dtype=torch.int32, device=x.device), x.view(torch.int16).int() & 0xFFFF)


def reduce_rows(rt, staging, topk_weights, out):
    """combine_recv of one expert's rows: token t adds up weight * row over the selections, rows 0, 1, .. in turn."""
    t, k = topk_weights.shape
    slot = torch.arange(k, dtype=torch.int32, device="cuda").repeat(t, 1).contiguous()
    expert = torch.zeros((t, k), dtype=torch.int64, device="cuda")
    rt.capi.check(rt.capi.load().deepep_ll_combine_recv(
        rt.capi.ptr(staging), rt.capi.ptr(expert), rt.capi.ptr(topk_weights), rt.capi.ptr(slot), t, staging.shape[1], k, 1,
        staging.shape[0], 0, rt.capi.ptr(out), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()


def test_combine_rounds_every_float_to_the_nearest_bf16(rt):
    """Sums that take every float32 value of a normal size: each is three bf16 values added without a rounding.  The values
    too small for that, infinities and NaN follow as weights of a row of ones, one lower half for each way to round."""
    n = 1 << 24
    one, low = torch.ones((1, 3), device="cuda"), torch.arange(n, dtype=torch.int64, device="cuda")
    out = torch.empty((1, n), dtype=torch.bfloat16, device="cuda")
    for top in range(256):
        bits = (low + (top << 24))
        exponent = (bits >> 23) & 255
        bits = torch.where((exponent >= 24) & (exponent < 255), bits, 0x3F800000 + (bits & 0x7FFFFF))
        x = torch.where(bits >= 1 << 31, bits - (1 << 32), bits).int().view(torch.float32)
        high = (x.view(torch.int32) & -65536).view(torch.float32)
        middle = ((x - high).view(torch.int32) & -65536).view(torch.float32)
        rows = torch.stack([v.view(torch.int32) >> 16 for v in (high, middle, x - high - middle)]).short().view(torch.bfloat16)
        reduce_rows(rt, rows, one, out)
        assert torch.equal(bf16_bits(out[0]), bf16_bits_of(x)), hex(top)
    upper = torch.arange(65536, dtype=torch.int64, device="cuda").view(-1, 1) << 16
    bits = (upper + torch.tensor([0, 1, 0x7FFF, 0x8000, 0x8001, 0xFFFF], device="cuda")).view(-1, 1)
    w = torch.where(bits >= 1 << 31, bits - (1 << 32), bits).int().view(torch.float32)
    out = torch.empty((w.shape[0], 128), dtype=torch.bfloat16, device="cuda")
    reduce_rows(rt, torch.ones((1, 128), dtype=torch.bfloat16, device="cuda"), w, out)
    want = bf16_bits_of(torch.where(w == 0, 0.0, w))  # +0 + -0 is +0
    assert torch.equal(bf16_bits(out), want.expand(-1, 128))


# zeros, the smallest and largest subnormal, the smallest normal, 1, the next two and half a step, the largest and half a
# step of it, infinities, a quiet and two signalling NaN
SPECIAL = [0x0000, 0x8000, 0x0001, 0x8001, 0x007F, 0x0080, 0x3F80, 0xBF80, 0x3F81, 0x3F82, 0x3B80, 0xBB80, 0x7F7F, 0xFF7F, 0x7B00,
           0xFB00, 0x7F80, 0xFF80, 0x7FC0, 0x7F81, 0xFFFF]


def test_combine_of_ties_infinities_and_nan(rt):
    """Every pair of special values as one sum of two rows."""
    v = torch.tensor(SPECIAL, dtype=torch.int32).short().view(torch.bfloat16)
    a, b = (m.reshape(-1) for m in torch.meshgrid(v, v, indexing="ij"))
    rows = torch.zeros((2, 512), dtype=torch.bfloat16)
    rows[0, :a.numel()], rows[1, :a.numel()] = a, b
    out = torch.empty((1, 512), dtype=torch.bfloat16, device="cuda")
    reduce_rows(rt, rows.cuda(), torch.ones((1, 2), device="cuda"), out)
    assert torch.equal(bf16_bits(out[0]).cpu(), bf16_bits_of((rows[0].float() + 0.0) + rows[1].float()))


@ONE_CALL
@pytest.mark.parametrize("e,rank", [(256, 11), (288, 7)])  # 288 experts: the reference's own LL test, nine per rank
def test_ll_config_full_size(rt, one_call, e, rank):
    """One GPU's share of EP=32 at 128 tokens x 7168, top-8 of 256 (or 288) experts, seeded world."""
    r, t, h, k = 32, 128, 7168, 8
    shape = rt.ll.LLShape(r, rank, e, t, h, k, O.ROW_FP8)
    st = rt.ll.LowLatencyState(shape)
    world = rt.lb.LoopbackWorld(r, rank, seed=2024)
    world.synthesise(t, h, k, e)
    x, topk = world.own_inputs()
    run_dispatch(st, world, x, topk, one_call=one_call)
    # the oracle regenerates the same world from the seed
    topk_all = O.synth_topk_idx(O.uniform_cdf(e), np.arange(r), t, k, 2024)
    assert torch.equal(world.topk_idx_all.cpu(), topk_all)
    x_all = O.synth_bf16_rows(np.arange(r * t, dtype=np.uint32), h, 2024).view(r, t, h)
    assert torch.equal(world.x_all.cpu().view(torch.int16), x_all.view(torch.int16))
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, O.ROW_FP8)
    check_dispatch(st, want, O.ROW_FP8)
    assert int(st.packed_recv_count.sum()) == int(((topk_all // (e // r)) == rank).sum())


@ONE_CALL
def test_skewed_routing_roundtrip(rt, one_call):
    """Zipf(1.2) popularity, 1 % outlier rows, EP=64 with 4 local experts, hot experts past half their slots."""
    r, rank, t, h, k, e = 64, 0, 256, 1024, 8, 256
    shape = rt.ll.LLShape(r, rank, e, t, h, k, O.ROW_FP8)
    st = rt.ll.LowLatencyState(shape)
    world = rt.lb.LoopbackWorld(r, rank, seed=99)
    world.synthesise(t, h, k, e, popularity="zipf", outlier_period=100)
    x, topk = world.own_inputs()
    run_dispatch(st, world, x, topk, one_call=one_call)
    topk_all = O.synth_topk_idx(O.zipf_cdf(e), np.arange(r), t, k, 99)
    x_all = O.synth_bf16_rows(np.arange(r * t, dtype=np.uint32), h, 99, outlier_period=100).view(r, t, h)
    assert torch.equal(world.topk_idx_all.cpu(), topk_all)
    assert torch.equal(world.x_all.cpu().view(torch.int16), x_all.view(torch.int16))
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, O.ROW_FP8)
    check_dispatch(st, want, O.ROW_FP8)
    assert int(st.packed_recv_count[0]) > r * t // 2, "the hottest expert should fill over half its slots"
    # round trip with identity experts: combined == x * sum(w) within FP8 error
    count = st.packed_recv_count.cpu()
    el, n_slots = st.packed_recv_x.shape[:2]
    y = torch.zeros((el, n_slots, h), dtype=torch.bfloat16)
    for i in range(el):
        n = int(count[i])
        y[i, :n] = O.per_token_cast_back(st.packed_recv_x[i, :n].cpu(), st.packed_recv_scales[i, :n].cpu())
    g = torch.Generator().manual_seed(1)
    w = torch.softmax(torch.randn((t, k), generator=g), dim=-1)
    out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
    run_combine(st, world, y.cuda(), topk, w.cuda(), out, mode=0, one_call=one_call)
    diff = O.calc_diff(x_all[rank].float() * w.sum(1, keepdim=True), out.cpu())
    assert diff < 9e-4, diff


def test_ll_argument_errors(rt):
    lib, capi = rt.capi.load(), rt.capi
    z = torch.zeros(4096, dtype=torch.uint8, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    # tokens beyond num_max_dispatch_tokens_per_rank
    rc = lib.deepep_ll_dispatch_send(capi.ptr(z), capi.ptr(z), 9, 128, 2, 8, 2, 0, 8, 1, capi.ptr(z), capi.ptr(z),
                                     capi.ptr(z), capi.ptr(z), capi.ptr(z), capi.ptr(z), 4096, s)
    assert rc != 0 and "num_tokens <= max_tokens" in lib.deepep_last_error().decode()
    # experts not divisible by ranks
    rc = lib.deepep_ll_dispatch_recv(capi.ptr(z), capi.ptr(z), 128, 9, 2, 8, 1, capi.ptr(z), capi.ptr(z), capi.ptr(z),
                                     capi.ptr(z), capi.ptr(z), None, 0, None, 0, s)
    assert rc != 0 and "num_experts % num_ranks == 0" in lib.deepep_last_error().decode()
    # workspace too small
    rc = lib.deepep_ll_dispatch_send(capi.ptr(z), capi.ptr(z), 8, 128, 2, 8, 2, 0, 8, 1, capi.ptr(z), capi.ptr(z),
                                     capi.ptr(z), capi.ptr(z), capi.ptr(z), capi.ptr(z), 16, s)
    assert rc != 0 and "workspace_bytes" in lib.deepep_last_error().decode()
    torch.cuda.synchronize()


@ONE_CALL
def test_empty_batch(rt, one_call):
    """No tokens on this rank: counts come from the peers alone, combine returns nothing."""
    r, rank, t, h, k, e = 4, 2, 6, 512, 2, 8
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=8, drop=0)
    shape = rt.ll.LLShape(r, rank, e, t, h, k, O.ROW_FP8)
    st = rt.ll.LowLatencyState(shape)
    world = rt.lb.LoopbackWorld(r, rank)
    world.set_inputs(x_all.cuda(), topk_all.cuda())
    run_dispatch(st, world, x_all[rank, :0].cuda(), topk_all[rank, :0].cuda(), one_call=one_call)
    xs, tks = list(x_all), list(topk_all)
    xs[rank], tks[rank] = xs[rank][:0], tks[rank][:0]
    want = O.ll_dispatch(xs, tks, rank, e, t, O.ROW_FP8)
    check_dispatch(st, want, O.ROW_FP8)
    assert (st.send_count == 0).all()


@pytest.mark.parametrize("hint", [180, 9000, 18000], ids=["one_launch", "past_8192_rows", "past_72_MB"])
@pytest.mark.parametrize("rank", [0, 1, 3])
def test_empty_batch_after_one_with_own_rows(rt, rank, hint):
    """A rank that ran out of tokens: the counts of its own rows that the call before left are gone from ranges, counts,
    statistics and the places of the higher ranks' rows.  An empty tensor's address is null, which says nothing else."""
    r, t, m, h, k, e = 4, 60, 1200, 4096, 3, 16
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=8 + rank, drop=3)
    st = rt.ll.LowLatencyState(rt.ll.LLShape(r, rank, e, m, h, k, O.ROW_FP8))
    st.expected_rows = hint
    st.segment_workspace = torch.empty(rt.capi.load().deepep_ll_segment_workspace_bytes(e, m), dtype=torch.uint8, device="cuda")
    world = rt.lb.LoopbackWorld(r, rank)
    world.set_inputs(x_all.cuda(), topk_all.cuda())
    xs, topks = list(x_all), list(topk_all)
    for tokens in (t, 0, t, 0):
        x, topk = x_all[rank, :tokens].cuda(), topk_all[rank, :tokens].cuda()
        assert (x.data_ptr() == 0) == (tokens == 0)
        stats = torch.zeros(e // r, dtype=torch.int32, device="cuda")
        run_dispatch(st, world, x, topk, stats, one_call=True)
        xs[rank], topks[rank] = x_all[rank, :tokens], topk_all[rank, :tokens]
        want = O.ll_dispatch(xs, topks, rank, e, m, O.ROW_FP8)
        check_dispatch(st, want, O.ROW_FP8)
        assert torch.equal(stats.cpu(), want["packed_recv_count"])
        send_count, _ = O.route(topks[rank], e, m)
        assert torch.equal(st.send_count.cpu(), send_count)
        own = st.recv_count.view(e // r, r)[:, rank].cpu()
        assert torch.equal(own, send_count[rank * (e // r):(rank + 1) * (e // r)])


def test_large_batch_without_the_segment_workspace(rt, oracle_c):
    """A large batch but no workspace for the row index: receive and row return fall back to the
    kernels of the small-batch path and must give the same answers."""
    r, rank, t, h, k, e = 8, 5, 4200, 512, 4, 64
    x_all, topk_all, w_all = make_world(r, t, h, k, e, seed=77, drop=10)
    shape = rt.ll.LLShape(num_ranks=r, rank=rank, num_experts=e, max_tokens=t, hidden=h, num_topk=k, fmt=O.ROW_FP8)
    st = rt.ll.LowLatencyState(shape)
    assert st.segment_workspace is not None
    st.segment_workspace = None
    world = rt.lb.LoopbackWorld(r, rank, seed=0)
    world.set_inputs(x_all.cuda(), topk_all.cuda())
    x, topk = world.own_inputs()
    run_dispatch(st, world, x, topk)
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, O.ROW_FP8)
    check_dispatch(st, want, O.ROW_FP8)
    # identity experts: the round trip returns x * sum(w) within the FP8 error
    count = st.packed_recv_count.cpu()
    y = torch.zeros((e // r, r * t, h), dtype=torch.bfloat16)
    for le in range(e // r):
        n = int(count[le])
        y[le, :n] = O.per_token_cast_back(st.packed_recv_x[le, :n].cpu(), st.packed_recv_scales[le, :n].cpu())
    out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
    w = torch.softmax(w_all[rank], dim=-1)
    run_combine(st, world, y.cuda(), topk, w.cuda(), out, mode=0)
    wsum = w.masked_fill(topk_all[rank] == -1, 0).sum(1, keepdim=True)
    assert O.calc_diff(x_all[rank].float() * wsum, out.cpu()) < 9e-4


@pytest.mark.parametrize("zero_copy", [False, True], ids=["rows_returned", "zero_copy"])
@pytest.mark.parametrize("fmt", [O.ROW_FP8, O.ROW_BF16])
def test_every_rank_on_one_gpu_with_a_real_exchange(rt, fmt, zero_copy):
    """All R ranks run on the one GPU, each with its own buffers, and the exchange between them is a
    plain copy of what the send sides produced (send_slots -> the peer's recv_staging, then
    combine_send_slots -> the peer's combine_staging).  Nothing is synthesised "in a peer's name":
    this is the data flow of a multi-GPU run with the transport replaced by device copies.
    zero_copy: the combine returns no rows; the exchange takes each (expert, source) range straight
    from the expert outputs, where layout_range says it lies."""
    r, t, h, k, e = 4, 12, 512, 3, 16
    epr = e // r
    x_all, topk_all, w_all = make_world(r, t, h, k, e, seed=123, drop=4)
    states = []
    for rank in range(r):
        st = rt.ll.LowLatencyState(rt.ll.LLShape(r, rank, e, t, h, k, fmt))
        st.recv_count.zero_()
        st.dispatch_send(x_all[rank].cuda(), topk_all[rank].cuda())
        states.append(st)
    torch.cuda.synchronize()
    # the dispatch exchange: rank s's rows for expert e travel to the rank that owns e
    for s in range(r):
        src = states[s]
        slots = src.send_slots.view(e, t, src.stride)
        counts = src.send_count.cpu()
        for ex in range(e):
            dst_rank, le = ex // epr, ex % epr
            if dst_rank == s:
                continue
            cnt = int(counts[ex])
            dst = states[dst_rank]
            dst.recv_staging.view(epr, r, t, dst.stride)[le, s, :cnt] = slots[ex, :cnt]
            dst.recv_count.view(epr, r)[le, s] = cnt
    outs = []
    for rank in range(r):
        st = states[rank]
        poison_outputs_keep_pair_slot(st)
        st.dispatch_recv()
        torch.cuda.synchronize()
        want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, fmt)
        check_dispatch(st, want, fmt)
        # identity experts
        if fmt == O.ROW_BF16:
            y = st.packed_recv_x.clone()
        else:
            q = st.packed_recv_x.float().view(epr, r * t, h // 128, 128)
            y = (q * st.packed_recv_scales.unsqueeze(-1)).view(epr, r * t, h).to(torch.bfloat16)
        y = torch.nan_to_num(y, nan=0.0, posinf=0.0, neginf=0.0)  # rows past the counts hold poison
        if not zero_copy:
            st.combine_send(y)
        outs.append(y)
    torch.cuda.synchronize()
    # the combine exchange: what rank q returns for rank s's pairs goes to s's staging for q's experts
    for q in range(r):
        src = states[q]
        back = src.combine_send_slots  # [E_l, R, M, H]
        lr = src.packed_recv_layout_range.cpu()
        for le in range(epr):
            for s in range(r):
                if s == q:
                    continue
                begin, cnt = int(lr[le, s] >> 32), int(lr[le, s] & 0xFFFFFFFF)
                if zero_copy:
                    states[s].combine_staging[q * epr + le, :cnt] = outs[q][le, begin:begin + cnt]
                else:
                    states[s].combine_staging[q * epr + le, :cnt] = back[le, s, :cnt]
    for rank in range(r):
        st = states[rank]
        out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
        out.view(torch.int16).fill_(0x7FC0)
        topk, w = topk_all[rank].cuda(), w_all[rank].cuda()
        if zero_copy:
            st.combine_send_slots.view(torch.int16).fill_(0x7FC0)
            st.combine(outs[rank], topk, w, out, zero_copy=True)  # the own experts' rows are read from the outputs
        else:
            st.combine_recv(topk, w, out)
        torch.cuda.synchronize()
        if zero_copy:
            assert (st.combine_send_slots.view(torch.int16) == 0x7FC0).all()
        wsum = w_all[rank].masked_fill(topk_all[rank] == -1, 0).sum(1, keepdim=True)
        diff = O.calc_diff(x_all[rank].float() * wsum, out.cpu())
        assert not torch.isnan(out.float()).any()
        assert diff < (9e-4 if fmt != O.ROW_BF16 else 1e-5), (rank, diff)


def poison_outputs_keep_pair_slot(st):
    st.packed_recv_x.view(torch.uint8).fill_(0xEE)
    if st.packed_recv_scales is not None:
        st.packed_recv_scales.view(torch.uint8).fill_(0xEE)
    st.packed_recv_src_info.fill_(-7)
    st.packed_recv_count.fill_(-7)
    st.packed_recv_layout_range.fill_(-7)


def test_exchange_metadata_through_the_host_module(rt):
    """The pybind11 binding returns the same values as the C-ABI call, and rejects a host tensor."""
    from deepep_efa_amd import deep_ep_cpp
    r, e, m, rank, cap = 8, 64, 50, 3, 512
    g = torch.Generator().manual_seed(77)
    routed = torch.randint(0, m + 1, (r, e), generator=g, dtype=torch.int32)
    send, recv, totals, remote, records, num_recv, per_expert = deep_ep_cpp.ll_exchange_metadata(routed.cuda(), rank, m, cap)
    torch.cuda.synchronize()
    want = O.ll_exchange_metadata(routed, rank, m)
    n = min(want["total_recv"], cap)
    assert send.cpu().tolist() == want["send_counts"].tolist() and recv.cpu().tolist() == want["recv_counts"].tolist()
    assert totals.cpu().tolist() == [want["total_send"], want["total_recv"], 0]
    assert remote.cpu().tolist() == want["combine_remote_recv_offset"].tolist()
    assert num_recv.cpu().tolist() == [want["total_recv"], n] and (per_expert == 0).all()
    for i, key in enumerate(("source_rank", "source_offset", "padded_index", "combine_send_offset")):
        assert records[i, :n].cpu().tolist() == want[key][:n].tolist(), key
    with pytest.raises(RuntimeError, match="Assertion"):
        deep_ep_cpp.ll_exchange_metadata(routed, rank, m, cap)
    for odd in (cap, cap + 3, 0):  # by name: the same launch, its records one by one
        named = rt.ll.exchange_metadata(routed.cuda(), rank, m, odd)
        whole = deep_ep_cpp.ll_exchange_metadata(routed.cuda(), rank, m, odd)
        n = min(want["total_recv"], odd)
        for got, key in zip(whole[:4] + whole[5:], ("send_counts", "recv_counts", "totals", "combine_remote_recv_offset",
                                                    "num_recv_tokens", "tokens_per_expert")):
            assert torch.equal(named[key], got), key
        for i, key in enumerate(("source_rank", "source_offset", "padded_index", "combine_send_offset")):
            assert named[key].shape == (odd,) and torch.equal(named[key][:n], whole[4][i, :n]), key
    with pytest.raises(RuntimeError):
        rt.ll.exchange_metadata(routed.cuda(), rank, m, -1)


@pytest.mark.parametrize("hint", ["batch", "unknown", "huge"])
def test_capacity_far_above_the_batch(rt, hint):
    """A caller may size M for its largest batch and dispatch a small one.  The kernels are picked from the
    expected-rows hint or, without one, a thirty-second of the capacity, and every hint gives the same result."""
    r, rank, t, m, h, k, e = 8, 2, 40, 5000, 512, 4, 64
    x_all, topk_all, w_all = make_world(r, t, h, k, e, seed=4242, drop=7)
    shape = rt.ll.LLShape(num_ranks=r, rank=rank, num_experts=e, max_tokens=m, hidden=h, num_topk=k, fmt=O.ROW_FP8)
    st = rt.ll.LowLatencyState(shape)
    st.expected_rows = {"batch": t * k, "unknown": 0, "huge": 10 ** 6}[hint]
    if st.segment_workspace is None:
        st.segment_workspace = torch.empty(rt.capi.load().deepep_ll_segment_workspace_bytes(e, m), dtype=torch.uint8,
                                           device="cuda")
    world = rt.lb.LoopbackWorld(r, rank, seed=0)
    world.set_inputs(x_all.cuda(), topk_all.cuda())
    x, topk = world.own_inputs()
    run_dispatch(st, world, x, topk, None, one_call=True)
    single = rt.capi.load().deepep_ll_dispatch_is_single_launch(t, k, e, m, st.expected_rows) == 1
    assert single == (hint == "batch")
    assert takes_one_launch(rt, st, t) == (hint != "huge")
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, m, O.ROW_FP8)
    check_dispatch(st, want, O.ROW_FP8)
    # combine with identity experts
    epr = e // r
    y = torch.zeros((epr, r * m, h), dtype=torch.bfloat16)
    count = st.packed_recv_count.cpu()
    for le in range(epr):
        n = int(count[le])
        y[le, :n] = O.per_token_cast_back(st.packed_recv_x[le, :n].cpu(), st.packed_recv_scales[le, :n].cpu())
    out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
    run_combine(st, world, y.cuda(), topk_all[rank].cuda(), w_all[rank].cuda(), out, mode=0, one_call=True)
    wsum = w_all[rank].masked_fill(topk_all[rank] == -1, 0).sum(1).view(-1, 1)
    live = wsum.view(-1) > 0
    assert O.calc_diff((x_all[rank].float() * wsum)[live], out.cpu().float()[live]) < 2e-3


@ONE_CALL
@pytest.mark.parametrize("fmt", [O.ROW_FP8, O.ROW_BF16])
def test_tokens_naming_an_expert_more_than_once(rt, fmt, one_call):
    """Top-k never does it, but the path defines it: every pair gets its own slot in (token, k) order, and
    pairs beyond the M slots of a (source, expert) segment are dropped (slot -1, not counted, not combined)."""
    r, rank, t, m, h, k, e = 2, 1, 6, 6, 256, 4, 4
    g = torch.Generator().manual_seed(5)
    x_all = torch.randn((r, t, h), generator=g).to(torch.bfloat16)
    topk_all = torch.tensor([[[3, 3, 3, 3]] * t,                       # 24 pairs for expert 3: 6 kept, 18 dropped
                             [[2, 2, 0, -1], [2, 3, 3, 1], [0, 0, 0, 0], [2, 1, 2, 1], [-1, -1, 3, 3], [2, 2, 2, 2]]])
    w_all = torch.rand((r, t, k), generator=g) + 0.1
    st, world = dispatch_on_gpu(rt, x_all, topk_all, rank, e, m, fmt, one_call=one_call)
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, m, fmt)
    check_dispatch(st, want, fmt)
    send_count, pair_slot = O.route(topk_all[rank], e, m)
    assert torch.equal(st.send_count.cpu(), send_count) and torch.equal(st.pair_slot[:t].cpu(), pair_slot)
    # what rank 0 sent to expert 3 (on rank 1): exactly M rows, the first M pairs in (token, k) order
    lr = int(st.packed_recv_layout_range[1, 0])
    assert lr & 0xFFFFFFFF == m
    assert st.packed_recv_src_info[1, (lr >> 32):(lr >> 32) + m].cpu().tolist() == [0, 0, 0, 0, 1, 1]
    # combine: identity experts on the received rows; dropped pairs contribute nothing
    epr = e // r
    y = torch.zeros((epr, r * m, h), dtype=torch.bfloat16)
    count = st.packed_recv_count.cpu()
    for le in range(epr):
        n = int(count[le])
        if fmt == O.ROW_BF16:
            y[le, :n] = st.packed_recv_x[le, :n].cpu()
        else:
            y[le, :n] = O.per_token_cast_back(st.packed_recv_x[le, :n].cpu(), st.packed_recv_scales[le, :n].cpu())
    out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
    run_combine(st, world, y.cuda(), topk_all[rank].cuda(), w_all[rank].cuda(), out, mode=0, one_call=one_call)
    live = pair_slot >= 0
    back = x_all[rank] if fmt == O.ROW_BF16 else O.per_token_cast_back(*O.per_token_cast_to_fp8(x_all[rank]))
    chain = O.ll_combine_f32_chain(back.unsqueeze(1).expand(-1, k, -1).contiguous(), w_all[rank], live)
    assert torch.equal(out.cpu().view(torch.int16), chain.view(torch.int16))


@ONE_CALL
@pytest.mark.parametrize("fmt", [O.ROW_FP8, O.ROW_BF16])
def test_send_past_the_streaming_bound(rt, one_call, fmt):
    """2800 tokens x 7168, top-8: the send moves more than 192 MB, so its payload stores carry the
    non-temporal hint (a different kernel instantiation); every output must be what the oracle says."""
    r, rank, t, h, k, e = 2, 1, 2800, 7168, 8, 16
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=2800, drop=10)
    assert t * (2 * h + k * O.row_payload(h, fmt)) > 192 * 2 ** 20
    st, _ = dispatch_on_gpu(rt, x_all, topk_all, rank, e, t, fmt, one_call=one_call)
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, fmt)
    check_dispatch(st, want, fmt)
    send_count, pair_slot = O.route(topk_all[rank], e, t)
    assert torch.equal(st.send_count.cpu(), send_count)
    assert torch.equal(st.pair_slot.cpu(), pair_slot)
    # the rows for the other rank's experts, byte for byte, on a sample of pairs
    _, _, experts, slots, rows = O.staged_rows(x_all[rank][:64], topk_all[rank][:64], rank, e, t, fmt, r)
    payload = O.row_payload(h, fmt)
    sendbuf = st.send_slots.view(e, t, st.stride)
    for i in range(0, rows.shape[0], 7):
        ex, sl = int(experts[i]), int(slots[i])
        if ex // (e // r) != rank:
            assert torch.equal(sendbuf[ex, sl, :payload].cpu(), rows[i, :payload]), (ex, sl)


@pytest.mark.parametrize("fmt", [O.ROW_FP8, O.ROW_BF16])
def test_every_rank_on_one_gpu_through_an_all_to_all(rt, fmt):
    """The data flow of the all_to_all_single fallback (deep_ep/buffer.py:2268,2297) with all R ranks on the
    one GPU: every rank's send side fills its per-expert slots; the "all-gather" of the route counts is the
    stack of the ranks' send_count; each rank's message to rank d is its rows for d's experts, expert by
    expert, copied into slot `source` of d's receive buffer; deepep_ll_exchange_metadata turns the gathered
    counts into the records and deepep_ll_dispatch_recv_by_source unpacks.  The packed outputs must be the
    oracle's (csrc/kernels/efa_kernels.cu:877-1052,1227-1389; csrc/transport/ll_pipeline.cpp:1204-1361)."""
    r, t, h, k, e = 4, 40, 512, 3, 16
    epr = e // r
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=321, drop=6)
    lib, capi = rt.capi.load(), rt.capi
    states = []
    for rank in range(r):
        st = rt.ll.LowLatencyState(rt.ll.LLShape(r, rank, e, t, h, k, fmt))
        st.dispatch_send(x_all[rank].cuda(), topk_all[rank].cuda())
        states.append(st)
    torch.cuda.synchronize()
    routed = torch.stack([st.send_count for st in states])  # [R, E]: what an all-gather of the counts leaves everywhere
    slot_rows = t * min(k, epr)
    stride = states[0].stride
    for rank in range(r):
        # the messages: source s -> this rank, rows in expert-major order (inside an expert, slot order)
        buf = torch.full((r * slot_rows, stride), 0xEE, dtype=torch.uint8, device="cuda")
        for s in range(r):
            src = states[s]
            counts = src.send_count.cpu()
            if s == rank:  # a rank's rows for its own experts were staged, not put into send slots
                own = src.recv_staging.view(epr, r, t, stride)
                parts = [own[le, rank, :int(counts[rank * epr + le])] for le in range(epr)]
            else:
                slots = src.send_slots.view(e, t, stride)
                parts = [slots[ex, :int(counts[ex])] for ex in range(rank * epr, (rank + 1) * epr)]
            msg = torch.cat(parts)
            buf[s * slot_rows:s * slot_rows + msg.shape[0]] = msg
        capacity = int(routed[:, rank * epr:(rank + 1) * epr].sum())
        meta = rt.ll.exchange_metadata(routed, rank, slot_rows, capacity)
        st = states[rank]
        poison_outputs_keep_pair_slot(st)
        ws = torch.empty(lib.deepep_ll_by_source_workspace_bytes(e, capacity), dtype=torch.uint8, device="cuda")
        capi.check(lib.deepep_ll_dispatch_recv_by_source(
            capi.ptr(buf), slot_rows, capi.ptr(meta["recv_counts"]), capi.ptr(meta["source_offset"]),
            capi.ptr(meta["num_recv_tokens"]), capacity, h, e, r, t, fmt, capi.ptr(st.packed_recv_x),
            capi.ptr(st.packed_recv_scales), capi.ptr(st.packed_recv_src_info), capi.ptr(st.packed_recv_layout_range),
            capi.ptr(st.packed_recv_count), None, None, None, 0, capi.ptr(ws), ws.numel(),
            torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, fmt)
        check_dispatch(st, want, fmt)
        assert int(meta["num_recv_tokens"][0]) == int(want["packed_recv_count"].sum())


@pytest.mark.parametrize("fmt", [O.ROW_FP8, O.ROW_BF16])
def test_single_launch_dispatch_past_the_streaming_bound(rt, fmt):
    """700 tokens x 7168, top-8 on two ranks: 5600 entries, so the dispatch is one launch, and more than
    64 MB of traffic, so that launch is the streaming instantiation."""
    r, rank, t, h, k, e = 2, 0, 700, 7168, 8, 16
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=700, drop=10)
    lib = rt.capi.load()
    assert lib.deepep_ll_dispatch_is_single_launch(t, k, e, t, t * k) == 1
    e_l = e // r
    received = sum(int(((tk >= rank * e_l) & (tk < (rank + 1) * e_l)).sum()) for tk in topk_all)
    assert t * (2 * h + k * O.row_payload(h, fmt)) + 2 * received * O.row_payload(h, fmt) > 64 * 2 ** 20
    st, _ = dispatch_on_gpu(rt, x_all, topk_all, rank, e, t, fmt, one_call=True)
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, fmt)
    check_dispatch(st, want, fmt)
    send_count, pair_slot = O.route(topk_all[rank], e, t)
    assert torch.equal(st.send_count.cpu(), send_count)
    assert torch.equal(st.pair_slot.cpu(), pair_slot)


@pytest.mark.parametrize("r,rank,t,h,k,e", [(8, 3, 64, 1024, 6, 64), (8, 3, 1500, 512, 8, 64)],
                         ids=["one_launch", "large_batch"])
def test_combine_without_row_return_reduces_the_same(rt, r, rank, t, h, k, e):
    """NULL send slots (zero copy): the call is the reduce alone; `out` is bit-identical to the full call's
    and no returned row is written."""
    x_all, topk_all, w_all = make_world(r, t, h, k, e, seed=91, drop=7)
    st, world = dispatch_on_gpu(rt, x_all, topk_all, rank, e, t, O.ROW_BF16, one_call=True)
    y = torch.randn((e // r, r * t, h), generator=torch.Generator().manual_seed(9)).to(torch.bfloat16).cuda()
    world.combine_from_peers(st, mode=1, seed=5)
    topk, w = topk_all[rank].cuda(), torch.softmax(w_all[rank], dim=-1).cuda()
    outs = []
    for zero_copy in (False, True):
        st.combine_send_slots.view(torch.int16).fill_(0x7FC0)
        out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
        out.view(torch.int16).fill_(0x7FC0)
        st.combine(y, topk, w, out, zero_copy=zero_copy)
        torch.cuda.synchronize()
        outs.append(out)
        touched = bool((st.combine_send_slots.view(torch.int16) != 0x7FC0).any())
        assert touched != zero_copy
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


# ---------------------------------------------------------------------------------------------
# The all-to-all shaped transport: one contiguous message per peer in both directions
# ---------------------------------------------------------------------------------------------
def send_by_dest_on_gpu(rt, x, topk, rank, r, e, m, fmt):
    t, h = x.shape
    k = topk.shape[1]
    st = rt.ll.AllToAllState(rt.ll.LLShape(r, rank, e, m, h, k, fmt))
    st.send_rows.fill_(0xEE)
    st.pair_slot.fill_(-7)
    for name in ("send_count", "send_expert_prefix", "send_counts", "send_cumsum"):
        getattr(st, name).fill_(-7)
    st.dispatch_send(x.cuda(), topk.cuda())
    torch.cuda.synchronize()
    return st


def check_send_by_dest(st, want, t):
    payload = st.lib.deepep_ll_row_payload_bytes(st.shape.hidden, st.shape.fmt)
    assert torch.equal(st.send_count.cpu(), want["send_count"])
    assert torch.equal(st.send_expert_prefix.cpu(), want["send_expert_prefix"])
    assert torch.equal(st.send_counts.cpu(), want["send_counts"])
    assert torch.equal(st.send_cumsum.cpu(), want["send_cumsum"])
    assert torch.equal(st.pair_slot[:t].cpu(), want["pair_slot"])
    n = want["rows"].shape[0]
    got = st.send_rows.cpu()
    h, fmt = st.shape.hidden, st.shape.fmt
    db, sb = O.row_data_bytes(h, fmt), O.row_scale_bytes(h, fmt)
    dp, sp = O.align_up(db, 16), O.align_up(sb, 16)
    touched = torch.zeros(got.shape[1], dtype=torch.bool)
    for lo, hi in ((0, db), (dp, dp + sb), (dp + sp, dp + sp + 16)):  # data, scales, tail: the padding is nobody's
        assert torch.equal(got[:n, lo:hi], want["rows"][:, lo:hi]), (lo, hi)
        touched[lo:hi] = True
    assert payload == dp + sp + 16
    assert (got[:n, ~touched] == 0xEE).all() and (got[n:] == 0xEE).all()  # nothing between the parts or behind the rows


@pytest.mark.parametrize("fmt", [O.ROW_FP8, O.ROW_BF16, O.ROW_FP8_UE8M0])
@pytest.mark.parametrize("r,rank,t,h,k,e", [
    (4, 1, 8, 512, 3, 16), (8, 7, 33, 1024, 4, 64), (2, 0, 1, 512, 1, 2),
    (32, 5, 128, 7168, 8, 256),  # the headline shape
    (2, 0, 1100, 512, 8, 16),    # T * K > 8192: the tables come from the chunk histograms
    (8, 5, 4200, 512, 4, 64),
    (16, 9, 12, 512, 6, 1024),   # the most experts
    (1, 0, 16, 512, 2, 4),       # a world of one rank
    (4, 2, 24, 1536, 4, 16),     # hidden not a multiple of 1024
    (512, 500, 3, 512, 2, 1024),
    (4, 3, 256, 512, 8, 32),     # 2048 entries: the last batch whose tables are built inside the send launch past 1024 experts
    (4, 3, 257, 512, 8, 32),     # 2056 entries
    (16, 9, 257, 512, 8, 1024),  # the most experts whose tables the send launch makes past 2048 entries
    (16, 9, 257, 512, 8, 1040),  # and the first with a launch for them
    (2, 1, 1024, 512, 8, 32),    # 8192 entries: the last without chunk histograms
    (8, 5, 1030, 512, 8, 816),   # five chunk histograms of 4080 words: the send launch makes the tables
    (8, 5, 1030, 512, 8, 824),   # 4120 words: a launch for them
    (4, 3, 8191, 512, 8, 8),     # the last batch whose entries a half word counts
    (4, 3, 8192, 512, 8, 8),
    (32, 7, 77, 512, 6, 288),    # five experts a lane, the last lanes without any; an odd number of entries before tokens
    (3, 2, 67, 512, 5, 195),     # as many experts as no lane's share divides, tokens of an odd number of entries
])
def test_send_by_dest(rt, fmt, r, rank, t, h, k, e):
    """One buffer, contiguous per destination rank, rows by expert and slot; counts, prefixes and every
    row byte against the oracle (csrc/kernels/efa_kernels.cu:2332-2400, row tail :797-800)."""
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=r * 17 + t, drop=min(5, t))
    st = send_by_dest_on_gpu(rt, x_all[rank], topk_all[rank], rank, r, e, t, fmt)
    check_send_by_dest(st, O.ll_send_by_dest(x_all[rank], topk_all[rank], rank, e, t, fmt, r), t)


@pytest.mark.parametrize("t,k,h,fmt", [
    (479, 8, 2048, O.ROW_FP8), (480, 8, 2048, O.ROW_FP8),  # one token a workgroup, two
    (481, 16, 512, O.ROW_FP8_POW2), (511, 8, 4096, O.ROW_FP8_UE8M0),
    (959, 8, 1024, O.ROW_BF16), (960, 8, 1024, O.ROW_BF16),  # two, four
    (963, 5, 640, O.ROW_FP8), (1021, 7, 2048, O.ROW_FP8), (1024, 8, 512, O.ROW_FP8), (1024, 8, 4096, O.ROW_FP8)])
def test_several_tokens_a_workgroup(rt, t, k, h, fmt):
    """From 480 tokens on a workgroup that ranks its own slots has two or four of them: experts that its tokens share,
    or one names twice, hot ones past a segment's room, entries that name none, and a last workgroup that is not full;
    by destination and in the single-launch dispatch."""
    r, rank, e, m = 4, 2, 20, t
    g = torch.Generator().manual_seed(t * k)
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=t + k, drop=0)
    topk_all[:] = torch.randint(0, e, topk_all.shape, generator=g)
    topk_all[torch.rand(topk_all.shape, generator=g) < 0.2] = 11  # the rank's own, and more often than it has slots
    topk_all[torch.rand(topk_all.shape, generator=g) < 0.05] = -1
    topk_all[rank, 3, 0], topk_all[rank, t - 1, k - 1] = e, (1 << 32) + 1
    live = (topk_all >= 0) & (topk_all < e)
    topk = torch.where(live, topk_all, -1)  # the same to the oracle
    st = send_by_dest_on_gpu(rt, x_all[rank], topk_all[rank], rank, r, e, m, fmt)
    check_send_by_dest(st, O.ll_send_by_dest(x_all[rank], topk[rank], rank, e, m, fmt, r), t)
    got, _ = dispatch_on_gpu(rt, x_all, topk_all, rank, e, m, fmt, one_call=True)
    check_dispatch(got, O.ll_dispatch(list(x_all), list(topk), rank, e, m, fmt), fmt)
    assert torch.equal(got.pair_slot.cpu().view(-1)[:t * k], st.pair_slot.cpu().view(-1)[:t * k])


@pytest.mark.parametrize("t,k,h,fmt,staged,by_dest", [
    (479, 8, 2048, O.ROW_FP8, 1, 1), (480, 8, 2048, O.ROW_FP8, 2, 2), (960, 8, 2048, O.ROW_FP8, 4, 4),  # four waves a token
    (959, 8, 3072, O.ROW_FP8, 1, 1), (960, 8, 3072, O.ROW_FP8, 2, 2),  # six: from 480 workgroups
    (1365, 3, 2560, O.ROW_FP8, 1, 1), (1365, 4, 2560, O.ROW_FP8, 2, 2),  # and 4096 entries
    (1000, 8, 7168, O.ROW_FP8, 1, 1), (600, 8, 7168, O.ROW_FP8, 1, 1),  # seven
    (959, 8, 4096, O.ROW_FP8, 1, 1), (960, 8, 4096, O.ROW_FP8, 1, 2), (1000, 8, 4096, O.ROW_BF16, 1, 2),  # eight
    (1000, 8, 4224, O.ROW_FP8, 2, 2), (1024, 8, 4096, O.ROW_FP8, 4, 4)])  # five, and four again
@pytest.mark.filterwarnings("ignore:DEBUG")  # the graph is written out
def test_tokens_of_a_send_workgroup(rt, t, k, h, fmt, staged, by_dest, tmp_path):
    """How many tokens a workgroup of a send takes, by the workgroups of its launch; the slots are the same."""
    r, rank, e = 4, 2, 64
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=t + k, drop=20)
    x, topk = x_all[rank].cuda(), topk_all[rank].cuda()
    send_count, pair_slot = O.route(topk_all[rank], e, t)
    shape = rt.ll.LLShape(r, rank, e, t, h, k, fmt)
    for st, tokens in ((rt.ll.LowLatencyState(shape), staged), (rt.ll.AllToAllState(shape), by_dest)):
        launched = kernels_launched(lambda: st.dispatch_send(x, topk), tmp_path)
        assert launched == {"ll_send_kernel": -(-t // tokens) + 1}
        st.dispatch_send(x, topk)
        assert torch.equal(st.send_count.cpu(), send_count) and torch.equal(st.pair_slot[:t].cpu(), pair_slot)


@pytest.mark.parametrize("t,k,h,fmt", [
    (13, 8, 4608, O.ROW_BF16), (224, 8, 4608, O.ROW_BF16), (225, 8, 4608, O.ROW_BF16),  # 9 pieces: five waves of a workgroup, eight
    (200, 6, 5120, O.ROW_BF16), (150, 8, 6144, O.ROW_BF16), (40, 8, 7168, O.ROW_BF16),  # 10, 12 and 14: five, six, eight
    (100, 7, 9216, O.ROW_FP8), (31, 3, 8832, O.ROW_FP8_POW2), (20, 5, 17408, O.ROW_FP8_UE8M0)])  # fp8; three workgroups a row
def test_rows_cut_evenly_between_workgroups(rt, t, k, h, fmt):
    """A row of more pieces than a workgroup has waves, cut evenly up to 1792 entries: the oracle's rows, sent and kept."""
    r, rank, e, m = 4, 2, 20, t
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=t + k, drop=5)
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, m, fmt)
    (got, _), (two, _) = (dispatch_on_gpu(rt, x_all, topk_all, rank, e, m, fmt, one_call=c) for c in (True, False))
    check_dispatch(got, want, fmt)
    check_dispatch(two, want, fmt)
    assert torch.equal(got.pair_slot, two.pair_slot) and torch.equal(got.send_count, two.send_count)
    data, own = (2 * h if fmt == O.ROW_BF16 else h), e // r
    for expert in range(e):  # rows to other ranks leave through the slots
        n = min(m, int(got.send_count[expert])) if expert // own != rank else 0
        a, b = (s.send_slots.view(torch.uint8).view(e, m, s.stride)[expert, :n, :data] for s in (got, two))
        assert torch.equal(a, b), f"rows sent to expert {expert}"


@pytest.mark.parametrize("t,k,h,fmt", [
    (576, 8, 4096, O.ROW_FP8), (577, 8, 4096, O.ROW_FP8), (1024, 8, 3072, O.ROW_FP8_UE8M0), (1536, 5, 2048, O.ROW_BF16),
    (1537, 5, 2048, O.ROW_BF16)])
@pytest.mark.parametrize("skew", [False, True])
def test_fewer_receive_workgroups(rt, t, k, h, fmt, skew):
    """Either side of where the single-launch dispatch has half as many receive workgroups, which go round for the rows:
    as many as were expected, and twice as many."""
    r, rank, e, m = 4, 1, 16, t
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=t + k, drop=9)
    if skew:  # every token's first two selections are this rank's
        topk_all[:, :, 0], topk_all[:, :, 1] = 4, 6
    st, world = dispatch_on_gpu(rt, x_all, topk_all, rank, e, m, fmt, one_call=True)
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, m, fmt)
    check_dispatch(st, want, fmt)
    x, topk = world.own_inputs()
    st.expected_rows = 1  # far too few
    run_dispatch(st, world, x, topk, None, one_call=True)
    check_dispatch(st, want, fmt)


@pytest.mark.parametrize("t,k,h,fmt", [
    (1024, 8, 2048, O.ROW_FP8), (1025, 8, 2048, O.ROW_FP8),  # 8192 entries, more
    (1025, 8, 4096, O.ROW_BF16), (1291, 7, 640, O.ROW_FP8_POW2), (1100, 8, 3584, O.ROW_FP8_UE8M0),
    (1773, 8, 2176, O.ROW_FP8), (1774, 8, 2176, O.ROW_FP8),  # 24 M entries for a token a workgroup to go through
    (3546, 8, 1024, O.ROW_BF16), (3547, 8, 1024, O.ROW_BF16),  # and for four tokens a workgroup
    (3546, 8, 512, O.ROW_BF16), (1408, 8, 512, O.ROW_BF16), (1409, 8, 512, O.ROW_BF16)])  # rows of one wave: 11264 entries
@pytest.mark.filterwarnings("ignore:DEBUG")  # the graph is written out
def test_one_call_dispatch_past_8192_entries(rt, t, k, h, fmt, tmp_path):
    """One launch or several, by entries, rows expected and what these hold in all: the oracle's rows either way, also
    where far more or fewer of them arrive than were expected; and the launches that a caller is told of."""
    r, rank, e, m = 4, 2, 20, t
    g = torch.Generator().manual_seed(t * k)
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=t + k, drop=0)
    topk_all[torch.rand(topk_all.shape, generator=g) < 0.1] = 11  # the rank's own, and more often than a token has slots for
    topk_all[torch.rand(topk_all.shape, generator=g) < 0.05] = -1
    most = min(96 << 10, (72 << 20) // rt.capi.load().deepep_ll_row_payload_bytes(h, fmt))
    st, world = dispatch_on_gpu(rt, x_all, topk_all, rank, e, m, fmt, one_call=True)
    x, topk = world.own_inputs()
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, m, fmt)
    check_dispatch(st, want, fmt)
    slots = st.pair_slot.clone()
    if st.segment_workspace is None:
        st.segment_workspace = torch.empty(rt.capi.load().deepep_ll_segment_workspace_bytes(e, m), dtype=torch.uint8,
                                           device="cuda")
    few = t * k <= 8192 or (t, h) in ((1025, 4096), (1025, 2048), (1291, 640), (1100, 3584), (1773, 2176), (3546, 1024), (1408, 512))
    for hint in (8192, 8193, most, most + 1):
        st.expected_rows = hint
        run_dispatch(st, world, x, topk, None, one_call=True)
        check_dispatch(st, want, fmt)
        assert torch.equal(st.pair_slot, slots)
        one = takes_one_launch(rt, st, t)
        assert one == (few and hint <= most)
        launched = kernels_launched(lambda: st.dispatch(x, topk), tmp_path)
        assert set(launched) == {"ll_dispatch_fused_kernel"} if one else "ll_rank_chunk_kernel" in launched


@pytest.mark.parametrize("receive", ["from_tails", "ordered"])
def test_all_to_all_with_an_empty_batch(rt, receive):
    """No token anywhere: the tables are zeros, nothing is received, the records stay untouched, and the reduce of
    no tokens is a no-op."""
    r, rank, m, h, k, e = 4, 2, 8, 512, 2, 8
    x = torch.empty((0, h), dtype=torch.bfloat16)
    topk = torch.empty((0, k), dtype=torch.int64)
    st = send_by_dest_on_gpu(rt, x, topk, rank, r, e, m, O.ROW_FP8)
    assert (st.send_count == 0).all() and (st.send_expert_prefix == 0).all()
    assert (st.send_counts == 0).all() and (st.send_cumsum == 0).all()
    assert (st.send_rows == 0xEE).all()
    routed = torch.zeros((r, e), dtype=torch.int32, device="cuda")
    st.exchange_metadata(routed)
    poison_outputs_keep_pair_slot(st)
    st.record_packed_row.fill_(-7)
    if receive == "ordered":
        st.dispatch_recv_ordered(routed)
    else:
        st.dispatch_recv()
    torch.cuda.synchronize()
    assert (st.packed_recv_count == 0).all() and (st.packed_recv_layout_range == 0).all()
    assert (st.tokens_per_expert == 0).all() and (st.record_packed_row == -7).all()
    y = torch.zeros((e // r, r * m, h), dtype=torch.bfloat16, device="cuda")
    st.send_flat.view(torch.int16).fill_(0x7FC0)
    st.combine_send(y)
    out = torch.empty((0, h), dtype=torch.bfloat16, device="cuda")
    st.combine_recv(topk.cuda(), torch.empty((0, k), dtype=torch.float32, device="cuda"), out)
    torch.cuda.synchronize()
    assert (st.send_flat.view(torch.int16) == 0x7FC0).all()


@pytest.mark.parametrize("t,k,e", [(1025, 8, 64), (1171, 7, 96), (1100, 8, 66), (2400, 5, 256), (1025, 64, 260),
                                   (8193, 1, 8), (8192, 8, 64), (8193, 8, 64), (13200, 5, 256), (1025, 8, 4096),
                                   (1088, 8, 64), (1089, 8, 128), (1240, 8, 128)])
def test_slots_of_batches_ranked_ahead_of_their_rows(rt, t, k, e):
    """Past 8192 entries a launch of its own ranks them, whole tokens of up to 2048 entries a chunk and 512 a workgroup,
    and what the chunks before a token's hold is added by the waves that store its rows: for up to 32 chunks and, by destination, up to
    64 experts or 256 in fours; beyond by a launch between the two.  With odd numbers of entries, experts named more than
    once by a token, hot ones, and entries that name none."""
    g = torch.Generator().manual_seed(t * 10 + e)
    topk = torch.randint(0, e, (t, k), generator=g)
    topk[torch.rand((t, k), generator=g) < 0.3] = e // 2
    topk[torch.rand((t, k), generator=g) < 0.05] = -1
    topk[3, 0], topk[t - 1, k - 1] = e, (1 << 32) + 1
    live = (topk >= 0) & (topk < e)
    flat = torch.where(live, topk, 0).view(-1).numpy()
    ok = live.view(-1).numpy()
    order = np.argsort(np.where(ok, flat, e), kind="stable")
    total = np.bincount(flat[ok], minlength=e)
    first = np.concatenate([[0], np.cumsum(total)])
    slot = np.full(t * k, -1, dtype=np.int64)
    mine = order[:int(ok.sum())]
    slot[mine] = np.arange(mine.size) - first[flat[mine]]
    m, h, r, rank = t, 128, 4 if e % 4 == 0 else 2, 1
    slot[slot >= m] = -1
    count = np.minimum(total, m)

    x = torch.randn((t, h), generator=g).to(torch.bfloat16)
    by_dest = send_by_dest_on_gpu(rt, x, topk, rank, r, e, m, O.ROW_BF16)
    assert np.array_equal(by_dest.pair_slot.cpu().numpy().reshape(-1)[:t * k], slot)
    assert np.array_equal(by_dest.send_count.cpu().numpy(), count)
    prefix = np.concatenate([[0], np.cumsum(count)])
    assert np.array_equal(by_dest.send_expert_prefix.cpu().numpy(), prefix)
    stride = rt.capi.load().deepep_ll_row_stride(h, O.ROW_BF16)
    rows = by_dest.send_rows.cpu().view(-1, stride)
    pair = np.flatnonzero(slot >= 0)
    at = torch.from_numpy(prefix[flat[pair]] + slot[pair])
    token = torch.from_numpy(pair // k)
    assert torch.equal(rows[at, :2 * h], x.view(torch.uint8)[token])
    tail = rows[at, 2 * h:2 * h + 16].contiguous().view(torch.int32)
    per_rank = e // r
    expert = torch.from_numpy(flat[pair])
    want = torch.stack([token, torch.from_numpy(pair % k), torch.full_like(token, rank), expert % per_rank], dim=1)
    assert torch.equal(tail, want.to(torch.int32))

    lib = rt.capi.load()
    n_src = 2  # two sources at once, whose slots nobody asked for, and the slots alone
    staging = torch.empty((e // r) * r * m * stride, dtype=torch.uint8, device="cuda")
    recv_count = torch.full((e // r, r), -7, dtype=torch.int32, device="cuda")
    ws = torch.empty(n_src * lib.deepep_ll_dispatch_workspace_bytes(t, k, e), dtype=torch.uint8, device="cuda")
    both_x = torch.stack([x, x.flip(0)]).cuda()
    both_topk = torch.stack([topk, topk]).cuda()
    src = torch.tensor([0, r - 1], dtype=torch.int32, device="cuda")
    if staging.numel() < 2 ** 32:
        rt.capi.check(lib.deepep_loopback_dispatch_from_peers(
            rt.capi.ptr(both_x), rt.capi.ptr(both_topk), rt.capi.ptr(src), n_src, t, h, k, e, r, rank, m, O.ROW_BF16,
            rt.capi.ptr(staging), rt.capi.ptr(recv_count), rt.capi.ptr(ws), ws.numel(), rt.ll.current_stream_ptr()))
        mine = torch.from_numpy(count[rank * per_rank:(rank + 1) * per_rank]).to(torch.int32)
        assert torch.equal(recv_count[:, 0].cpu(), mine) and torch.equal(recv_count[:, r - 1].cpu(), mine)
        assert (recv_count[:, 1:r - 1] == -7).all()
        le = per_rank // 2
        got = staging.view(per_rank, r, m, stride)[le, r - 1, :int(mine[le]), 2 * h:2 * h + 4].contiguous().view(torch.int32)
        of_expert = (expert == rank * per_rank + le).numpy()
        assert torch.equal(got.view(-1).cpu(), token[torch.from_numpy(of_expert)].to(torch.int32))
        for name, scratch in (("deepep_ll_dispatch_send", (rt.capi.ptr(ws), ws.numel())), ("deepep_ll_dispatch_send_static", ())):
            sent = torch.full((e,), -7, dtype=torch.int32, device="cuda")
            pair_slot = torch.full((t, k), -7, dtype=torch.int32, device="cuda")
            recv_count.fill_(-7)
            rt.capi.check(getattr(lib, name)(
                rt.capi.ptr(both_x), rt.capi.ptr(both_topk), t, h, k, e, r, rank, m, O.ROW_BF16, rt.capi.ptr(staging),
                rt.capi.ptr(recv_count), None, rt.capi.ptr(sent), rt.capi.ptr(pair_slot), *scratch, rt.ll.current_stream_ptr()))
            assert np.array_equal(pair_slot.cpu().numpy().reshape(-1), slot), name
            assert np.array_equal(sent.cpu().numpy(), count), name
            assert torch.equal(recv_count[:, rank].cpu(), mine), name


@pytest.mark.parametrize("rank", [0, 5])
def test_one_call_dispatch_of_few_entries_and_many_rows(rt, rank):
    """Fewer than 8192 entries but more rows than a single launch takes: the slots ahead, the index beside the rows."""
    r, t, h, k, e = 8, 300, 256, 8, 64
    g = torch.Generator().manual_seed(77)
    x_all = torch.randn((r, t, h), generator=g).to(torch.bfloat16)
    topk = torch.topk(torch.rand((r, t, e), generator=g) + (torch.arange(e) // 8 == rank) * 0.6, k, dim=-1)[1]
    topk[:, ::7, 2] = -1
    want = O.ll_dispatch(x_all, topk.contiguous(), rank, e, t, O.ROW_FP8)
    shape = rt.ll.LLShape(num_ranks=r, rank=rank, num_experts=e, max_tokens=t, hidden=h, num_topk=k, fmt=O.ROW_FP8)
    st = rt.ll.LowLatencyState(shape)
    st.expected_rows = 96 * 1024 + 1
    assert not takes_one_launch(rt, st, t)
    st.segment_workspace = torch.empty(rt.capi.load().deepep_ll_segment_workspace_bytes(e, t), dtype=torch.uint8,
                                       device="cuda")
    world = rt.lb.LoopbackWorld(r, rank, seed=0)
    world.set_inputs(x_all.cuda(), topk.contiguous().cuda())
    x, own = world.own_inputs()
    run_dispatch(st, world, x, own, None, True)
    assert int(want["packed_recv_count"].sum()) > 8192
    check_dispatch(st, want, O.ROW_FP8)


@pytest.mark.parametrize("t,k,e,rows", [(300, 8, 64, 99000), (1500, 8, 64, 0), (1500, 8, 64, 12000), (1611, 7, 96, 12000),
                                        (8300, 8, 64, 70000)])  # the last of more than 32 chunks
def test_workspace_that_holds_the_chunk_histograms_alone(rt, t, k, e, rows):
    """ceil(T / floor(2048 / K)) * E * 4 bytes, rounded up to 256, for each source: every send works with them."""
    r, rank, h, fmt = 4, 2, 256, O.ROW_FP8
    lib = rt.capi.load()
    g = torch.Generator().manual_seed(t + e)
    x_all = torch.randn((r, t, h), generator=g).to(torch.bfloat16).cuda()
    topk = torch.randint(0, e, (r, t, k), generator=g)
    topk[torch.rand((r, t, k), generator=g) < 0.05] = -1
    topk = topk.cuda()
    hist_bytes = (-(-t // (2048 // k)) * e * 4 + 255) // 256 * 256
    assert hist_bytes < lib.deepep_ll_dispatch_workspace_bytes(t, k, e)
    per_rank = e // r

    def guarded(nbytes):
        whole = torch.full((nbytes + 4096,), 0x5A, dtype=torch.uint8, device="cuda")
        return whole[:nbytes], whole[nbytes:]

    def dispatch(small):
        st = rt.ll.LowLatencyState(rt.ll.LLShape(num_ranks=r, rank=rank, num_experts=e, max_tokens=t, hidden=h, num_topk=k, fmt=fmt))
        st.expected_rows = rows
        assert not takes_one_launch(rt, st, t)
        st.segment_workspace = (torch.empty(lib.deepep_ll_segment_workspace_bytes(e, t), dtype=torch.uint8, device="cuda")
                                if rows > 0 else None)
        world = rt.lb.LoopbackWorld(r, rank, seed=0)
        world.set_inputs(x_all, topk)
        x, own = world.own_inputs()
        guard = torch.empty(0, device="cuda")
        if small:
            st.workspace, guard = guarded(hist_bytes)
        st.recv_staging.fill_(0x5A)
        st.send_slots.fill_(0)  # a row's padding is not written
        stats = torch.zeros(per_rank, dtype=torch.int32, device="cuda")
        run_dispatch(st, world, x, own, stats, True)
        count = st.packed_recv_count
        written = torch.arange(r * t, device="cuda") < count.view(-1, 1)
        assert (guard == 0x5A).all()
        own_staged = st.recv_staging.view(per_rank, r, -1)[:, rank]
        assert (own_staged == 0x5A).all()
        return [count, stats, st.recv_count, st.send_count, st.pair_slot, st.packed_recv_layout_range,
                st.packed_recv_x.view(torch.uint8)[written], st.packed_recv_scales[written], st.packed_recv_src_info[written],
                st.send_slots]

    for i, (a, b) in enumerate(zip(dispatch(False), dispatch(True))):
        assert torch.equal(a, b), i

    src = torch.tensor([0, 3], dtype=torch.int32, device="cuda")
    stride = lib.deepep_ll_row_stride(h, fmt)
    staged = []
    for size in (lib.deepep_ll_dispatch_workspace_bytes(t, k, e), hist_bytes):
        ws, guard = guarded(2 * size)
        staging = torch.zeros((per_rank, r, t, stride), dtype=torch.uint8, device="cuda")
        recv_count = torch.zeros((per_rank, r), dtype=torch.int32, device="cuda")
        rt.capi.check(lib.deepep_loopback_dispatch_from_peers(
            rt.capi.ptr(x_all[[0, 3]].contiguous()), rt.capi.ptr(topk[[0, 3]].contiguous()), rt.capi.ptr(src), 2, t, h, k, e, r, rank, t,
            fmt, rt.capi.ptr(staging), rt.capi.ptr(recv_count), rt.capi.ptr(ws), ws.numel(), rt.ll.current_stream_ptr()))
        assert (guard == 0x5A).all()
        staged.append((staging, recv_count))
    assert all(torch.equal(a, b) for a, b in zip(*staged))


def test_send_by_dest_with_repeated_experts_and_full_pairs(rt):
    """Tokens naming an expert more than once: pairs beyond a pair's M slots are dropped from the counts,
    the prefixes and the buffer alike."""
    r, rank, t, m, h, k, e = 2, 1, 6, 6, 256, 4, 4
    g = torch.Generator().manual_seed(5)
    x = torch.randn((t, h), generator=g).to(torch.bfloat16)
    topk = torch.tensor([[2, 2, 0, -1], [2, 3, 3, 1], [3, 3, 3, 3], [2, 1, 2, 1], [-1, -1, 3, 3], [3, 3, 3, 3]])
    st = send_by_dest_on_gpu(rt, x, topk, rank, r, e, m, O.ROW_FP8)
    want = O.ll_send_by_dest(x, topk, rank, e, m, O.ROW_FP8, r)
    assert int(want["send_count"][3]) == m and int((want["pair_slot"] == -1).sum()) > 3
    check_send_by_dest(st, want, t)


def all_to_all_dispatch(states, fmt):
    """The dispatch all-to-all between ranks that share the GPU: the gathered counts, then one slice copy per
    (source, destination) pair -- no regrouping of rows on the way."""
    r = len(states)
    routed = torch.stack([st.send_count for st in states])
    cums = [st.send_cumsum.cpu().tolist() for st in states]
    for d, dst in enumerate(states):
        dst.recv_by_source.fill_(0xEE)
        dst.exchange_metadata(routed)
        for s, src in enumerate(states):
            lo, hi = cums[s][d], cums[s][d + 1]
            assert hi - lo <= dst.slot_rows
            dst.recv_by_source[s * dst.slot_rows:s * dst.slot_rows + hi - lo] = src.send_rows[lo:hi]
    return routed


@pytest.mark.parametrize("receive", ["from_tails", "ordered", "ordered_as_a_large_batch"])
@pytest.mark.parametrize("delivery", ["flat", "slotted", "direct"])
@pytest.mark.parametrize("fmt", [O.ROW_FP8, O.ROW_BF16])
@pytest.mark.parametrize("r,t,h,k,e", [(4, 40, 512, 3, 16), (8, 700, 512, 8, 64), (3, 5, 256, 2, 3)],
                         ids=["small", "chunked_receive", "one_expert_per_rank"])
def test_all_to_all_round_trip_on_one_gpu(rt, oracle_c, fmt, delivery, receive, r, t, h, k, e):
    """Every rank on the one GPU, the transport replaced by slice copies of contiguous ranges: send by
    destination, exchange metadata from the gathered counts, receive by source, experts, return by
    destination (into a flat buffer that is copied range by range, or -- `direct` -- straight into the
    peers' receive buffers), reduce from the flat (or slotted) buffer.  Dispatch outputs bit-exact against
    the oracle, per-record rows against its loops, the combine against the float32 chain.
    (deep_ep/buffer.py:2266-2301,2601-2608,2735; csrc/transport/ll_pipeline.cpp:1204-1361)"""
    run_all_to_all_round_trip(rt, oracle_c, fmt, delivery, receive, r, t, h, k, e)


@pytest.mark.parametrize("delivery,receive", [("flat", "ordered"), ("direct", "from_tails")])
def test_all_to_all_round_trip_at_the_headline_shape(rt, oracle_c, delivery, receive):
    """The same with all 32 ranks of the headline world (128 tokens x 7168, top-8 of 256 experts, FP8) on the one
    GPU; the dispatch outputs of three ranks and the combined rows of the same three against the oracle."""
    run_all_to_all_round_trip(rt, oracle_c, O.ROW_FP8, delivery, receive, 32, 128, 7168, 8, 256, check_ranks=(0, 5, 31))


@pytest.mark.parametrize("seed", range(16))
def test_all_to_all_round_trip_random_worlds(rt, oracle_c, seed):
    """Seeded random small worlds through the same flow: odd rank counts, one to five experts a rank, one token
    to a few hundred (both sides of the 2048 entries up to which the send builds its own tables), every format,
    receive and delivery."""
    rng = np.random.default_rng(1000 + seed)
    r = int(rng.choice([1, 2, 3, 4, 6, 8, 16]))
    epr = int(rng.choice([1, 2, 3, 5]))
    e = r * epr
    k = int(rng.integers(1, min(8, e) + 1))
    t = int(rng.choice([1, 2, 7, 33, 64, 129, 260, 300]))
    h = int(rng.choice([128, 256, 512, 1024, 1536, 2048]))
    fmt = [O.ROW_FP8, O.ROW_BF16, O.ROW_FP8_POW2, O.ROW_FP8_UE8M0][int(rng.integers(4))]
    if fmt == O.ROW_FP8_UE8M0 and (h // 128) % 4:
        h = 512  # packed UE8M0 scales come four to a word
    delivery = ["flat", "slotted", "direct"][int(rng.integers(3))]
    receive = ["from_tails", "ordered", "ordered_as_a_large_batch"][int(rng.integers(3))]
    run_all_to_all_round_trip(rt, oracle_c, fmt, delivery, receive, r, t, h, k, e)


@pytest.mark.parametrize("t", [48, 1100], ids=["decode_size", "large_batch"])
def test_all_to_all_step_replays_in_a_hip_graph(rt, t):
    """A rank's five calls over the all-to-all surface captured once and replayed: they must allocate nothing
    and record no memset, and every replay, with eager work and synchronisations in between, must leave what the
    eager calls left (the peers' messages and answers stay where the eager exchange put them)."""
    r, rank, h, k, e, fmt = 4, 1, 1024, 8, 32, O.ROW_FP8
    epr = e // r
    x_all, topk_all, w_all = make_world(r, t, h, k, e, seed=77, drop=5)
    states = []
    for s_ in range(r):
        st = rt.ll.AllToAllState(rt.ll.LLShape(r, s_, e, t, h, k, fmt))
        st.dispatch_send(x_all[s_].cuda(), topk_all[s_].cuda())
        states.append(st)
    torch.cuda.synchronize()
    routed = all_to_all_dispatch(states, fmt)  # also runs every rank's exchange_metadata
    me = states[rank]
    x, topk, w = x_all[rank].cuda(), topk_all[rank].cuda(), w_all[rank].cuda()
    y = torch.empty((epr, r * t, h), dtype=torch.bfloat16, device="cuda")
    rt.capi.check(rt.capi.load().deepep_synth_bf16_rows(rt.capi.ptr(y), epr * r * t, h, h * 2, None, 0, 31, 0,
                                                        torch.cuda.current_stream().cuda_stream))
    me.recv_flat.normal_()  # the peers' answers
    out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
    meta = me.meta
    lib, capi = rt.capi.load(), rt.capi
    meta_args = [capi.ptr(routed), e, r, rank, me.slot_rows, me.row_capacity] + [capi.ptr(meta[n]) for n in (
        "send_counts", "recv_counts", "totals", "combine_remote_recv_offset", "source_rank", "source_offset",
        "padded_index", "combine_send_offset", "num_recv_tokens", "tokens_per_expert")]

    def step():
        me.dispatch_send(x, topk)
        capi.check(lib.deepep_ll_exchange_metadata(*meta_args, torch.cuda.current_stream().cuda_stream))
        me.dispatch_recv_ordered(routed)
        me.combine_send(y)
        me.combine_recv(topk, w, out)

    n_records = int(meta["num_recv_tokens"][1])  # the records past them are nobody's to write
    outputs = lambda: (me.send_rows, me.send_expert_prefix, me.send_cumsum, me.pair_slot, me.packed_recv_count,
                       me.packed_recv_layout_range, me.record_packed_row[:n_records], me.send_flat.view(torch.int16),
                       out.view(torch.int16))
    me.send_rows.fill_(0xEE)
    me.send_flat.view(torch.int16).fill_(0x7FC0)
    step()
    torch.cuda.synchronize()
    want = [v.clone() for v in outputs()]
    n_rows = int(me.packed_recv_count.sum())
    assert n_rows > (8192 if t > 1024 else 0)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        step()
    for replay in range(4):
        me.send_rows.fill_(0xEE)  # eager work between the replays: scribble over what the step writes
        me.send_flat.view(torch.int16).fill_(0x7FC0)
        out.zero_()
        me.packed_recv_count.fill_(-1)
        me.record_packed_row.fill_(-7)
        me.pair_slot.fill_(-9)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for i, (got, exp) in enumerate(zip(outputs(), want)):
            assert torch.equal(got, exp), f"replay {replay}: output {i}"


def test_all_to_all_round_trip_with_large_batches(rt, oracle_c):
    """4096 tokens a rank, 8 ranks x 32 experts, hidden 2048 (every rank on the one GPU needs ~9 GB then): the
    send runs on chunk histograms with the prefix launch, the receive on the ordered index and the flat row copy,
    the return and the reduce on their streaming forms; one rank against the oracle."""
    import gc
    gc.collect()
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    if free < 90 * 2 ** 30:
        pytest.skip(f"needs ~75 GB of free HBM, {free >> 30} GiB are free")
    run_all_to_all_round_trip(rt, oracle_c, O.ROW_FP8, "flat", "ordered", 8, 4096, 2048, 8, 256, check_ranks=(3,))


def run_all_to_all_round_trip(rt, oracle_c, fmt, delivery, receive, r, t, h, k, e, check_ranks=None):
    epr = e // r
    checked = range(r) if check_ranks is None else check_ranks
    x_all, topk_all, w_all = make_world(r, t, h, k, e, seed=555 + r, drop=min(6, t))
    states = []
    for rank in range(r):
        st = rt.ll.AllToAllState(rt.ll.LLShape(r, rank, e, t, h, k, fmt))
        st.dispatch_send(x_all[rank].cuda(), topk_all[rank].cuda())
        states.append(st)
    torch.cuda.synchronize()
    routed = all_to_all_dispatch(states, fmt)
    ys = []
    for rank, st in enumerate(states):
        poison_outputs_keep_pair_slot(st)
        st.record_packed_row.fill_(-7)
        st.tokens_per_expert.fill_(-7)
        if receive.startswith("ordered"):  # the messages are in this build's own order: placed from the counts alone
            if receive == "ordered_as_a_large_batch":  # the index launch + flat row copy instead of the single launch
                st.expected_rows = 9000
            st.dispatch_recv_ordered(routed)
        else:
            st.dispatch_recv()
        torch.cuda.synchronize()
        assert torch.equal(st.tokens_per_expert, st.packed_recv_count)
        if rank in checked:
            want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, fmt)
            check_dispatch(st, want, fmt)
            n = int(st.meta["num_recv_tokens"][1])
            rec = O.ll_record_packed_rows(list(topk_all), rank, e, t)
            assert n == rec.numel() and torch.equal(st.record_packed_row[:n].cpu().long(), rec)
            assert (st.record_packed_row[n:] == -7).all()
        # the experts: a seeded row per packed slot
        y = torch.empty((epr, r * t, h), dtype=torch.bfloat16, device="cuda")
        rt.capi.check(rt.capi.load().deepep_synth_bf16_rows(rt.capi.ptr(y), epr * r * t, h, h * 2, None, 0, 900 + rank,
                                                            0, torch.cuda.current_stream().cuda_stream))
        ys.append(y)
    peer_table = torch.tensor([st.recv_flat.data_ptr() for st in states], dtype=torch.int64, device="cuda")
    peer_rows = torch.tensor([st.recv_flat.shape[0] for st in states], dtype=torch.int64, device="cuda")
    for st in states:
        st.recv_flat.view(torch.int16).fill_(0x7FC0)
        st.send_flat.view(torch.int16).fill_(0x7FC0)
    for rank, st in enumerate(states):
        if delivery == "direct":
            st.combine_send(ys[rank], peer_table, peer_rows)
        else:
            st.combine_send(ys[rank])
    torch.cuda.synchronize()
    slot_rows = t * min(k, epr)
    slotted = [torch.full((r * slot_rows, h), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in states]
    if delivery != "direct":  # the all-to-all back: one slice copy per (answering rank, asking rank) pair
        cums = [st.send_cumsum.cpu().tolist() for st in states]
        for d, ans in enumerate(states):
            recv_counts = ans.meta["recv_counts"].cpu().tolist()
            first = 0
            for s, ask in enumerate(states):
                n = recv_counts[s]
                assert n == cums[s][d + 1] - cums[s][d]
                assert int(ans.meta["combine_remote_recv_offset"][s]) == cums[s][d]
                ask.recv_flat[cums[s][d]:cums[s][d] + n] = ans.send_flat[first:first + n]
                slotted[s][d * slot_rows:d * slot_rows + n] = ans.send_flat[first:first + n]
                first += n
    else:
        assert all((st.send_flat.view(torch.int16) == 0x7FC0).all() for st in states)  # nothing went the long way
    for rank, st in enumerate(states):
        if rank not in checked:
            continue
        topk, w = topk_all[rank], w_all[rank]
        out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
        out.view(torch.int16).fill_(0x7FC0)
        if delivery == "slotted":
            st.combine_recv(topk.cuda(), w.cuda(), out, recv=slotted[rank], slot_rows=slot_rows)
        else:
            st.combine_recv(topk.cuda(), w.cuda(), out)
        torch.cuda.synchronize()
        # which seeded row answers each pair: the packed row the owner of the expert gave it
        _, pair_slot = O.route(topk, e, t)
        live = pair_slot >= 0
        pair_rows = torch.zeros((t, k, h), dtype=torch.bfloat16)
        for d in range(r):
            lr = states[d].packed_recv_layout_range.cpu()
            sel = live & (topk // epr == d)
            ti, ki = torch.nonzero(sel, as_tuple=True)
            if ti.numel() == 0:
                continue
            le = (topk[ti, ki] % epr)
            begin = (lr[le, rank] >> 32)
            keys = (le * (r * t) + begin + pair_slot[ti, ki].long()).numpy().astype(np.uint32)
            pair_rows[ti, ki] = O.synth_bf16_rows(keys, h, 900 + d)
        chain = torch.empty((t, h), dtype=torch.int16)
        live8 = live.to(torch.uint8).contiguous()
        oracle_c.oracle_combine_chain(ctypes.c_void_p(pair_rows.view(torch.int16).data_ptr()),
                                      ctypes.c_void_p(w.contiguous().data_ptr()), ctypes.c_void_p(live8.data_ptr()),
                                      t, k, h, ctypes.c_void_p(chain.data_ptr()))
        assert torch.equal(out.cpu().view(torch.int16), chain), (rank, delivery)
        ref = O.ll_combine(pair_rows, topk, w, live)
        err = (out.cpu().double() - ref).abs()
        assert (err <= 1e-2 * ref.abs() + 1e-2 * ref.abs().mean()).all()  # the 1e-2 bar against the float64 sum


def test_all_to_all_hand_derived_world(rt):
    """The same flow on the two-rank world worked out on paper (tests/golden/ll_tiny_world.json): message order,
    tables, per-record packed rows, the flat buffers of both directions and the combined rows -- no oracle."""
    g, x_all, topk_all = load_tiny_world()
    e, m, h, t, k, r = g["num_experts"], g["max_tokens"], g["hidden"], g["num_tokens"], g["num_topk"], g["num_ranks"]
    states = []
    for rank in range(r):
        st = rt.ll.AllToAllState(rt.ll.LLShape(r, rank, e, m, h, k, O.ROW_BF16))
        st.dispatch_send(x_all[rank].cuda(), topk_all[rank].cuda())
        states.append(st)
    torch.cuda.synchronize()
    tail_at = O.row_payload(h, O.ROW_BF16) - 16
    for rank, st in enumerate(states):
        want = g["send_by_dest"][f"rank{rank}"]
        assert st.send_expert_prefix.cpu().tolist() == want["send_expert_prefix"]
        assert st.send_counts.cpu().tolist() == want["send_counts"]
        assert st.send_cumsum.cpu().tolist() == want["send_cumsum"]
        n = want["send_cumsum"][-1]
        tails = st.send_rows[:n, tail_at:tail_at + 16].cpu().contiguous().view(torch.int32)
        assert tails[:, 0].tolist() == want["row_token"] and tails[:, 1].tolist() == want["row_topk_slot"]
        assert tails[:, 3].tolist() == want["row_local_expert"]
        slot = st.pair_slot[:t].cpu()
        prefix = torch.tensor(want["send_expert_prefix"])
        row = torch.where(slot >= 0, prefix[topk_all[rank].clamp(min=0)] + slot, torch.full_like(slot, -1))
        assert row.tolist() == want["pair_send_row"]
    all_to_all_dispatch(states, O.ROW_BF16)
    for rank, st in enumerate(states):
        st.dispatch_recv()
        torch.cuda.synchronize()
        rec = g["record_packed_row"][f"rank{rank}"]
        assert st.record_packed_row[:len(rec)].cpu().tolist() == rec
        want, layout = tiny_world_expected(g, f"rank{rank}_ascending")
        assert st.packed_recv_count.cpu().tolist() == want["count"]
        assert torch.equal(st.packed_recv_layout_range.cpu(), layout)
        st.combine_send(st.packed_recv_x)  # identity experts
        torch.cuda.synchronize()
        flat = g["combine_send_flat_identity_experts"][f"rank{rank}"]
        assert st.send_flat[:len(flat)].cpu().float()[:, 0].tolist() == flat
    cums = [st.send_cumsum.cpu().tolist() for st in states]
    for d, ans in enumerate(states):
        recv_counts, first = ans.meta["recv_counts"].cpu().tolist(), 0
        for s, ask in enumerate(states):
            ask.recv_flat[cums[s][d]:cums[s][d] + recv_counts[s]] = ans.send_flat[first:first + recv_counts[s]]
            first += recv_counts[s]
    want_back = g["combine_recv_flat_rank0_identity_experts"]
    assert states[0].recv_flat[:len(want_back)].cpu().float()[:, 0].tolist() == want_back
    out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
    w = torch.tensor(g["topk_weights_rank0"], dtype=torch.float32, device="cuda")
    states[0].combine_recv(topk_all[0].cuda(), w, out)
    torch.cuda.synchronize()
    expect = torch.tensor(g["combine_rank0_identity_experts"]).view(-1, 1).expand(-1, h)
    assert torch.equal(out.cpu().float(), expect)


@pytest.mark.parametrize("t,hint", [(24, 0), (1500, 0), (1500, 1500)],
                         ids=["one_workgroup_per_source", "chunked", "one_workgroup_per_source_past_its_hint"])
def test_dispatch_recv_by_source_clamps_a_pair_to_max_tokens(rt, t, hint):
    """Slots wider than M and senders that put more than M rows into one (expert, source) pair: the pair keeps
    its first M rows in arrival order, the counts and ranges count only those, and an expert's ranges stay
    inside its R * M packed slots -- what the staged receive does with an over-full count."""
    r, rank, h, k, e, fmt = 2, 0, 512, 4, 8, O.ROW_FP8
    m = t // 3  # what the receiver was built for; the senders route as if M were t
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=11, drop=0)
    topk_all[1, :, :] = torch.tensor([0, 1, 2, 3])  # source 1: t rows for each of rank 0's experts
    slot_rows = 4 * t
    buf = rows_by_source(x_all, topk_all, rank, e, t, fmt, slot_rows)
    routed = torch.stack([O.route(topk_all[s], e, t)[0] for s in range(r)]).to(torch.int32)
    capacity = 8 * t
    lib, capi = rt.capi.load(), rt.capi
    meta = rt.ll.exchange_metadata(routed.clamp(max=slot_rows).cuda(), rank, slot_rows, capacity)
    st = rt.ll.LowLatencyState(rt.ll.LLShape(r, rank, e, m, h, 1, fmt), keep_remote_rows=False)
    poison_outputs(st)
    ws = torch.empty(lib.deepep_ll_by_source_workspace_bytes(e, capacity), dtype=torch.uint8, device="cuda")
    rec = torch.full((capacity,), -7, dtype=torch.int32, device="cuda")
    capi.check(lib.deepep_ll_dispatch_recv_by_source(
        capi.ptr(buf.cuda()), slot_rows, capi.ptr(meta["recv_counts"]), capi.ptr(meta["source_offset"]),
        capi.ptr(meta["num_recv_tokens"]), capacity, h, e, r, m, fmt, capi.ptr(st.packed_recv_x),
        capi.ptr(st.packed_recv_scales), capi.ptr(st.packed_recv_src_info), capi.ptr(st.packed_recv_layout_range),
        capi.ptr(st.packed_recv_count), None, None, capi.ptr(rec), hint, capi.ptr(ws), ws.numel(),
        torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    epr, n_slots = e // r, r * m
    tail_at = O.row_payload(h, fmt) - 16
    tail = buf[:, tail_at:tail_at + 16].contiguous().view(torch.int32)
    recv_counts = meta["recv_counts"].cpu().tolist()
    kept = [[[] for _ in range(r)] for _ in range(epr)]
    want_rec, i = [], 0
    for s in range(r):
        for j in range(recv_counts[s]):
            row = s * slot_rows + j
            le = int(tail[row, 3])
            if len(kept[le][s]) < m:
                kept[le][s].append((row, i))
            i += 1
    want_rec = [-1] * i
    count = st.packed_recv_count.cpu().tolist()
    layout = st.packed_recv_layout_range.cpu()
    px = st.packed_recv_x.view(torch.uint8).cpu()
    for le in range(epr):
        begin = 0
        for s in range(r):
            rows = kept[le][s]
            assert int(layout[le, s]) == (((begin << 32) | len(rows)) if rows else 0), (le, s)
            if rows:
                idx = torch.tensor([row for row, _ in rows])
                assert torch.equal(px[le, begin:begin + len(rows)], buf[idx, :h])
                for pos, (_, rec_i) in enumerate(rows):
                    want_rec[rec_i] = le * n_slots + begin + pos
            begin += len(rows)
        assert count[le] == begin and begin <= n_slots
    assert max(count) == n_slots or t < 30  # source 1 alone fills its half of every expert
    assert rec[:i].cpu().tolist() == want_rec


def test_ordered_receive_with_slots_too_small_and_counts_too_large(rt):
    """The ordered receive on hostile inputs: a source whose message does not fit its slot loses the rows past
    it (their records read -1, the ranges count only what was kept), and a count above M is read as M."""
    r, rank, t, h, k, e, fmt = 2, 0, 30, 512, 4, 8, O.ROW_FP8
    epr = e // r
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=17, drop=0)
    topk_all[1, :, :] = torch.tensor([0, 1, 2, 3])  # source 1 sends t rows to each of rank 0's four experts
    slot_rows = 2 * t + 7  # ... but its slot holds two experts' worth and a bit
    states = []
    for s_ in range(r):
        st = rt.ll.AllToAllState(rt.ll.LLShape(r, s_, e, t, h, k, fmt), slot_rows=slot_rows)
        st.dispatch_send(x_all[s_].cuda(), topk_all[s_].cuda())
        states.append(st)
    torch.cuda.synchronize()
    routed = torch.stack([st.send_count for st in states])
    dst = states[rank]
    dst.recv_by_source.fill_(0xEE)
    for s_, src in enumerate(states):
        lo, hi = [int(v) for v in src.send_cumsum[rank:rank + 2].cpu()]
        n = min(hi - lo, slot_rows)
        dst.recv_by_source[s_ * slot_rows:s_ * slot_rows + n] = src.send_rows[lo:lo + n]
    routed_big = routed.clone()
    routed_big[0, 1] += 1000  # nonsense from source 0 for expert 1: read as M rows
    for mat, hint in ((routed, t * k), (routed_big, t * k), (routed, 9000), (routed_big, 9000)):
        poison_outputs_keep_pair_slot(dst)
        dst.record_packed_row.fill_(-7)
        dst.expected_rows = hint  # the single launch, then the index launch + flat row copy
        dst.dispatch_recv_ordered(mat)
        torch.cuda.synchronize()
        sent = mat[:, rank * epr:(rank + 1) * epr].cpu().clamp(max=t)  # [source, local expert]
        want_rec, begin = [], [0] * epr
        kept = torch.zeros((epr, r), dtype=torch.int64)
        for s_ in range(r):
            first = 0
            for le in range(epr):
                c = int(sent[s_, le])
                kept[le, s_] = max(0, min(c, slot_rows - first))
                first += c
        layout = dst.packed_recv_layout_range.cpu()
        for le in range(epr):
            b = 0
            for s_ in range(r):
                n = int(kept[le, s_])
                assert int(layout[le, s_]) == (((b << 32) | n) if n else 0)
                b += n
            assert int(dst.packed_recv_count[le]) == b
        for s_ in range(r):
            for le in range(epr):
                b = int(kept[le, :s_].sum())
                want_rec += [le * r * t + b + j if j < int(kept[le, s_]) else -1 for j in range(int(sent[s_, le]))]
        n_rec = min(len(want_rec), dst.row_capacity)
        assert dst.record_packed_row[:n_rec].cpu().tolist() == want_rec[:n_rec]
        if mat is routed:  # the rows kept are the oracle's rows, in place
            want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, fmt)
            px = dst.packed_recv_x.view(torch.uint8).cpu()
            for le in range(epr):
                n0 = int(kept[le, 0])
                assert torch.equal(px[le, :n0], want["packed_recv_x"][le, :n0])  # source 0 fits whole
                n1 = int(kept[le, 1])
                full0 = int(want["packed_recv_layout_range"][le, 0] & 0xFFFFFFFF)
                assert torch.equal(px[le, n0:n0 + n1], want["packed_recv_x"][le, full0:full0 + n1])


@pytest.mark.parametrize("hidden", [128, 1152, 7168, 16512])
@pytest.mark.parametrize("records", [0, 1, 33, 255, 257, 700])
def test_return_by_destination_over_record_counts(rt, records, hidden):
    """Record counts around the windows the rows are walked in, rows below, at and above two vectors a thread, records
    in another order than the rows, records without a row, and more records than the grid was sized for."""
    r, e, m = 4, 8, 128
    capacity = 512 if records > 512 else max(records, 1)
    g = torch.Generator().manual_seed(records * 7 + hidden)
    x = torch.randn((e * m, hidden), generator=g).bfloat16().cuda()
    packed = torch.randperm(e * m, generator=g)[:capacity].int()
    packed[::5] = -1
    padded, offset = (torch.randperm(capacity, generator=g).int() for _ in range(2))
    out = torch.full((capacity, hidden), 3.0, dtype=torch.bfloat16, device="cuda")
    num = torch.tensor([records, records], dtype=torch.int32, device="cuda")
    on_gpu = [v.cuda() for v in (packed, padded, offset)]
    rt.capi.check(rt.capi.load().deepep_ll_combine_send_by_dest(
        rt.capi.ptr(x), rt.capi.ptr(on_gpu[0]), None, rt.capi.ptr(on_gpu[1]), rt.capi.ptr(on_gpu[2]), rt.capi.ptr(num), capacity,
        hidden, e, r, m, rt.capi.ptr(out), None, None, None, None, 64, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    want = torch.full((capacity, hidden), 3.0, dtype=torch.bfloat16)
    for i in range(min(records, capacity)):
        row = int(packed[int(padded[i])])
        if row >= 0:
            want[int(offset[i])] = x[row].cpu()
    assert torch.equal(out.cpu(), want)


@pytest.mark.parametrize("hidden,hints", [(7168, (877, 878, 1755, 1756)), (8192, (768, 769, 1536, 1537))])
def test_return_by_destination_whose_accesses_stream_in_part(rt, hidden, hints):
    """24 and 48 MB of expected traffic: which accesses carry the streaming hint changes no row."""
    r, e, m, capacity, records = 4, 8, 256, 2048, 300
    g = torch.Generator().manual_seed(hidden)
    x = torch.randn((e * m, hidden), generator=g).bfloat16().cuda()
    packed = torch.randperm(e * m, generator=g)[:capacity].int()
    offset = torch.randperm(capacity, generator=g).int()
    num = torch.tensor([records, records], dtype=torch.int32, device="cuda")
    on_gpu = [v.cuda() for v in (packed, torch.arange(capacity, dtype=torch.int32), offset)]
    want = torch.full((capacity, hidden), 3.0, dtype=torch.bfloat16, device="cuda")
    want[on_gpu[2][:records].long()] = x[on_gpu[0][:records].long()]
    for hint in hints:
        out = torch.full((capacity, hidden), 3.0, dtype=torch.bfloat16, device="cuda")
        rt.capi.check(rt.capi.load().deepep_ll_combine_send_by_dest(
            rt.capi.ptr(x), rt.capi.ptr(on_gpu[0]), None, rt.capi.ptr(on_gpu[1]), rt.capi.ptr(on_gpu[2]), rt.capi.ptr(num),
            capacity, hidden, e, r, m, rt.capi.ptr(out), None, None, None, None, hint, torch.cuda.current_stream().cuda_stream))
        assert torch.equal(out, want), hint


@pytest.mark.parametrize("t", [292, 293])  # 32 MB of gathered rows, and more
def test_reduce_around_its_streaming_bound(rt, t):
    """The reduce of a batch is the reduces of its tokens."""
    h, k, e = 7168, 8, 16
    g = torch.Generator().manual_seed(t)
    topk = torch.topk(torch.rand((t, e), generator=g), k, dim=-1)[1]
    topk[5, 3] = -1
    slots = torch.arange(t, dtype=torch.int32).repeat_interleave(k).view(t, k)
    slots[topk < 0] = -1
    staging = torch.randn((e, t, h), generator=g).bfloat16().cuda()
    w, topk, slots = torch.rand((t, k), generator=g).cuda(), topk.cuda(), slots.cuda()
    lib = rt.capi.load()

    def reduce(lo, hi):
        out = torch.full((hi - lo + 1, h), 7.0, dtype=torch.bfloat16, device="cuda")
        parts = [v[lo:hi].contiguous() for v in (topk, w, slots)]
        rt.capi.check(lib.deepep_ll_combine_recv(rt.capi.ptr(staging), *[rt.capi.ptr(v) for v in parts], hi - lo, h, k, e, t, 0,
                                                 rt.capi.ptr(out), torch.cuda.current_stream().cuda_stream))
        assert (out[hi - lo] == 7.0).all()
        return out[:hi - lo]

    assert torch.equal(reduce(0, t), torch.cat([reduce(0, 100), reduce(100, t)]))


@pytest.mark.parametrize("hidden", [8192, 16512])  # a round of 1024 threads, and more than two
@pytest.mark.parametrize("records,hint", [(700, 32768), (700, 32769), (33792 + 257, 32769)])  # the last has more than workgroups
def test_return_by_destination_of_many_records(rt, records, hidden, hint):
    """Past 32768 expected records a row takes up to 1024 threads instead of 512."""
    e, r, capacity = 8, 4, 34400
    g = torch.Generator(device="cuda").manual_seed(records + hidden)
    x = torch.randint(-2 ** 15, 2 ** 15, (capacity, hidden), dtype=torch.int16, device="cuda", generator=g)
    packed, padded, offset = (torch.randperm(capacity, device="cuda", generator=g).int() for _ in range(3))
    packed[::5] = -1
    out = torch.full((capacity, hidden), 3, dtype=torch.int16, device="cuda")
    num = torch.tensor([records, records], dtype=torch.int32, device="cuda")
    rt.capi.check(rt.capi.load().deepep_ll_combine_send_by_dest(
        rt.capi.ptr(x), rt.capi.ptr(packed), None, rt.capi.ptr(padded), rt.capi.ptr(offset), rt.capi.ptr(num), capacity, hidden, e,
        r, capacity // e, rt.capi.ptr(out), None, None, None, None, hint, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    rows, to = packed[padded[:records].long()].long(), offset[:records].long()
    want = torch.full_like(out, 3)
    want[to[rows >= 0]] = x[rows[rows >= 0]]
    assert torch.equal(out, want)


@pytest.mark.parametrize("records", [1000, 16384 + 256, 20000])
def test_return_by_destination_with_room_for_a_million_records_and_no_hint(rt, records):
    """Every record is moved, also those past the 16384 workgroups, and none of the room is paid for: 820 us for 1000
    rows with a workgroup for each record there is room for, 17 with 16384 of them, 5 with the rows as a hint."""
    h, e, m, capacity = 7168, 64, 16384, 1 << 20
    lib = rt.capi.load()
    x = torch.randn((records, h), generator=torch.Generator().manual_seed(records)).bfloat16().cuda()
    out = torch.full((records, h), 3.0, dtype=torch.bfloat16, device="cuda")  # no record names a row past it
    index = torch.arange(capacity, dtype=torch.int32, device="cuda")
    num = torch.tensor([records, records], dtype=torch.int32, device="cuda")

    def move(hint):
        rt.capi.check(lib.deepep_ll_combine_send_by_dest(
            rt.capi.ptr(x), rt.capi.ptr(index), None, rt.capi.ptr(index), rt.capi.ptr(index), rt.capi.ptr(num), capacity, h, e,
            8, m, rt.capi.ptr(out), None, None, None, None, hint, torch.cuda.current_stream().cuda_stream))

    def best(hint):
        times = []
        for _ in range(10):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            move(hint)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end) * 1000)
        return min(times)

    move(0)
    torch.cuda.synchronize()
    assert torch.equal(out, x)
    assert best(0) < best(records) + 150


@pytest.mark.parametrize("t,h,fmt,hint", [
    (33, 128, O.ROW_FP8, 8193), (33, 15488, O.ROW_FP8, 8193),  # the grid is far larger than the rows; two trips a row
    (40, 8320, O.ROW_BF16, 9000), (1300, 512, O.ROW_FP8_UE8M0, 8193),  # more rows than workgroups
    (4700, 128, O.ROW_FP8, 65537),  # two rows a workgroup, and more than that
    (300, 1024, O.ROW_BF16, 65537), (300, 5120, O.ROW_BF16, 65537), (300, 5248, O.ROW_BF16, 65537),  # where one and two meet
])
def test_row_copies_over_widths_and_hints(rt, t, h, fmt, hint):
    """The flat row copy of both directions, every row and every byte around it."""
    r, rank, k, e = 2, 1, 8, 16
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=t + h, drop=20)
    st = rt.ll.LowLatencyState(rt.ll.LLShape(num_ranks=r, rank=rank, num_experts=e, max_tokens=t, hidden=h, num_topk=k,
                                             fmt=fmt))
    st.expected_rows = hint
    st.segment_workspace = torch.empty(rt.capi.load().deepep_ll_segment_workspace_bytes(e, t), dtype=torch.uint8,
                                       device="cuda")
    world = rt.lb.LoopbackWorld(r, rank, seed=0)
    world.set_inputs(x_all.cuda(), topk_all.cuda())
    run_dispatch(st, world, *world.own_inputs())
    want = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, fmt)
    check_dispatch(st, want, fmt)
    px = st.packed_recv_x.view(torch.uint8).view(e // r, r * t, -1)
    for le, n in enumerate(st.packed_recv_count.tolist()):
        assert bool((px[le, n:] == 0xEE).all())  # nothing behind the last row
    y = torch.randn((e // r, r * t, h), device="cuda").bfloat16()
    st.combine_send_slots.fill_(3.0)
    st.combine_staging.fill_(3.0)
    slots, staging = st.combine_send_slots.clone(), st.combine_staging.clone()
    st.combine_send(y)
    for le in range(e // r):
        for s in range(r):
            begin, n = int(want["packed_recv_layout_range"][le, s]) >> 32, int(want["packed_recv_layout_range"][le, s]) & 0xFFFFFFFF
            (staging[rank * (e // r) + le] if s == rank else slots[le, s])[:n] = y[le, begin:begin + n]
    assert torch.equal(st.combine_send_slots, slots) and torch.equal(st.combine_staging, staging)


def test_row_return_sized_for_more_rows_than_a_launch_has_threads(rt):
    """4.2 million expected rows of 1024 vectors, a workgroup of 1024 threads each, would be 2^32 threads, which a
    launch refuses; the six rows that are there are moved all the same."""
    r, m, h, n = 1024, 4096, 8192, 3
    lib = rt.capi.load()
    x = torch.randn((2 * n, h), generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    ranges = torch.zeros((1, r), dtype=torch.int64)
    ranges[0, 0], ranges[0, 1] = n, (n << 32) | n  # this rank's own rows and those owed to rank 1
    ranges = ranges.cuda()
    staging = torch.full((n + 1, h), 3.0, dtype=torch.bfloat16, device="cuda")
    slots = torch.full((m + n + 1, h), 3.0, dtype=torch.bfloat16, device="cuda")
    ws = torch.empty(lib.deepep_ll_segment_workspace_bytes(r, m), dtype=torch.uint8, device="cuda")
    rt.capi.check(lib.deepep_ll_combine_send(
        rt.capi.ptr(x), rt.capi.ptr(ranges), h, r, r, 0, m, rt.capi.ptr(staging), rt.capi.ptr(slots), r * m,
        rt.capi.ptr(ws), ws.numel(), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(staging[:n], x[:n]) and torch.equal(slots[m:m + n], x[n:])
    assert bool((staging[n:] == 3.0).all()) and bool((slots[:m] == 3.0).all()) and bool((slots[m + n:] == 3.0).all())


@pytest.mark.parametrize("hint", [0, 1024 * 4096])
def test_ordered_receive_sized_for_more_rows_than_a_launch_has_threads(rt, hint):
    """The same for rows whose payload takes 960 threads and whose scales take a wave more, by a hint and by capacity."""
    r, m, h, n = 1024, 4096, 15360, 3
    lib = rt.capi.load()
    stride, payload = lib.deepep_ll_row_stride(h, O.ROW_FP8), lib.deepep_ll_row_payload_bytes(h, O.ROW_FP8)
    rows = torch.randint(0, 256, (m + n, stride), dtype=torch.uint8, generator=torch.Generator().manual_seed(2)).cuda()
    routed = torch.zeros((r, r), dtype=torch.int32)
    routed[:2, 0] = n  # sources 0 and 1 send three rows each to this rank's expert
    routed = routed.cuda()
    i32 = dict(dtype=torch.int32, device="cuda")
    px = torch.full((2 * n + 1, h), 7, dtype=torch.uint8, device="cuda")
    scales, info = torch.full((2 * n + 1, h // 128), 7, **i32), torch.full((2 * n + 1,), 7, **i32)
    ranges, count = torch.empty((1, r), dtype=torch.int64, device="cuda"), torch.empty(1, **i32)
    ws = torch.empty(256 + r * m * 8, dtype=torch.uint8, device="cuda")
    rt.capi.check(lib.deepep_ll_dispatch_recv_by_source_ordered(
        rt.capi.ptr(rows), m, rt.capi.ptr(routed), h, r, r, 0, m, O.ROW_FP8, rt.capi.ptr(px), rt.capi.ptr(scales),
        rt.capi.ptr(info), rt.capi.ptr(ranges), rt.capi.ptr(count), None, None, None, r * m, hint, rt.capi.ptr(ws),
        ws.numel(), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    want = torch.cat([rows[:n], rows[m:]])
    assert count.tolist() == [2 * n]
    assert torch.equal(px[:2 * n], want[:, :h]) and bool((px[2 * n] == 7).all())
    assert torch.equal(scales[:2 * n], want[:, h:h + h // 32].contiguous().view(torch.int32)) and bool((scales[2 * n] == 7).all())
    assert torch.equal(info[:2 * n], want[:, payload - 16:payload - 12].contiguous().view(torch.int32).view(-1)) and int(info[2 * n]) == 7


@pytest.mark.parametrize("t,k", [(1025, 8), (1100, 8)])
def test_large_combine_moves_no_rows_of_a_malformed_range(rt, t, k):
    """Past 8192 rows the reduce's launch builds the row return's index; a segment whose range leaves its expert gets
    no rows moved, all others do, and the reduce does not depend on it."""
    r, rank, h, e = 8, 3, 512, 16
    x_all, topk_all, w = make_world(r, t, h, k, e, seed=t, drop=30)
    st, world = dispatch_on_gpu(rt, x_all, topk_all, rank, e, t, O.ROW_BF16, one_call=True)
    topk, weights = topk_all[rank].cuda(), w[rank].cuda()
    y = torch.randn(st.packed_recv_x.shape, generator=torch.Generator().manual_seed(t)).bfloat16().cuda()
    world.combine_from_peers(st, mode=1, seed=5)
    got = []
    sound = st.packed_recv_layout_range
    bad = sound.clone()
    le, source = 1, 6
    bad[le, source] = (int(r * t) << 32) | int(sound[le, source] & 0xffffffff)
    for lr in (sound, bad):
        st.combine_send_slots.view(torch.int16).fill_(0x7FC0)
        out = torch.zeros((t, h), dtype=torch.bfloat16, device="cuda")
        st.combine(y, topk, weights, out, layout_range=lr)
        torch.cuda.synchronize()
        got.append((st.combine_send_slots.view(torch.int16).view(e // r, r, t, h).cpu(), out.cpu()))
    want = got[0][0].clone()
    for l2 in range(e // r):  # what a row return moves, worked out from the ranges
        for s in range(r):
            n, begin = int(sound[l2, s] & 0xffffffff), int(sound[l2, s] >> 32)
            rows = y[l2, begin:begin + n].view(torch.int16).cpu()
            if s != rank:
                assert torch.equal(want[l2, s, :n], rows)
    want[le, source] = 0x7FC0
    assert torch.equal(got[1][0], want)
    assert torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("fmt,h,hints", [(O.ROW_BF16, 4096, (6656, 6657)), (O.ROW_FP8, 7168, (7606, 7607, 8193))])
def test_ordered_receive_in_one_launch_and_in_two(rt, fmt, h, hints):
    """On either side of the 52 MB of expected rows the ordered receive gives the oracle's rows and records."""
    r, rank, t, k, e = 3, 1, 40, 4, 24
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=h, drop=9)
    states = [rt.ll.AllToAllState(rt.ll.LLShape(r, s, e, t, h, k, fmt)) for s in range(r)]
    for s, st in enumerate(states):
        st.dispatch_send(x_all[s].cuda(), topk_all[s].cuda())
    torch.cuda.synchronize()
    routed, st = all_to_all_dispatch(states, fmt), states[rank]
    want, rec = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, fmt), O.ll_record_packed_rows(list(topk_all), rank, e, t)
    for hint in hints:
        poison_outputs_keep_pair_slot(st)
        st.record_packed_row.fill_(-7)
        st.expected_rows = hint
        st.dispatch_recv_ordered(routed)
        torch.cuda.synchronize()
        check_dispatch(st, want, fmt)
        assert torch.equal(st.record_packed_row[:rec.numel()].cpu().long(), rec)


@pytest.mark.parametrize("fmt,h,e,hints", [
    (O.ROW_BF16, 2048, 24, (8192, 8193, 10240, 10241)),  # 40 MB past 8192 rows
    (O.ROW_FP8, 2048, 24, (16384, 16385)), (O.ROW_FP8, 1920, 24, (8192, 8193)),  # the last rows, and too narrow ones
    (O.ROW_FP8, 2048, 256, (8193, 16385)), (O.ROW_FP8, 2048, 260, (8192, 8193))])  # the last experts, and too many
@pytest.mark.filterwarnings("ignore:DEBUG")  # the graph is written out
def test_ordered_receive_past_8192_rows(rt, fmt, h, e, hints, tmp_path):
    """One launch or two past 8192 expected rows: the oracle's rows and records either way.  All hints but the last take
    one launch."""
    r, rank, t, k = 4, 3, 33, 5
    x_all, topk_all, _ = make_world(r, t, h, k, e, seed=h, drop=9)
    states = [rt.ll.AllToAllState(rt.ll.LLShape(r, s, e, t, h, k, fmt)) for s in range(r)]
    for s, st in enumerate(states):
        st.dispatch_send(x_all[s].cuda(), topk_all[s].cuda())
    torch.cuda.synchronize()
    routed, st = all_to_all_dispatch(states, fmt), states[rank]
    want, rec = O.ll_dispatch(list(x_all), list(topk_all), rank, e, t, fmt), O.ll_record_packed_rows(list(topk_all), rank, e, t)
    for hint in hints:
        poison_outputs_keep_pair_slot(st)
        st.record_packed_row.fill_(-7)
        st.expected_rows = hint
        st.dispatch_recv_ordered(routed)
        torch.cuda.synchronize()
        check_dispatch(st, want, fmt)
        assert torch.equal(st.record_packed_row[:rec.numel()].cpu().long(), rec)
        launched = kernels_launched(lambda: st.dispatch_recv_ordered(routed), tmp_path)
        assert set(launched) == ({"ll_recv_ordered_kernel"} if hint != hints[-1] else
                                 {"ll_by_source_ordered_index_kernel", "ll_rows_flat_kernel"}), hint


@pytest.mark.parametrize("h,hints", [
    (1024, (8192, 8193, 16400, 16401)),  # one launch, one that streams, the last before twice the selections, two launches
    (512, (12288, 12289)),  # rows below 2 KB: one launch, two
])
def test_combine_in_one_launch_and_in_two(rt, h, hints):
    """A combine's rows and its sums do not depend on which launches the expected rows choose."""
    r, rank, t, k, e = 8, 3, 1025, 8, 16
    x_all, topk_all, w = make_world(r, t, h, k, e, seed=h, drop=30)
    st, world = dispatch_on_gpu(rt, x_all, topk_all, rank, e, t, O.ROW_BF16, one_call=True)
    y = torch.randn(st.packed_recv_x.shape, generator=torch.Generator().manual_seed(h)).bfloat16().cuda()
    world.combine_from_peers(st, mode=1, seed=5)
    ranges, slots = st.packed_recv_layout_range.cpu(), torch.full((e // r, r, t, h), 0x7FC0, dtype=torch.int16)
    for le in range(e // r):
        for s in range(r):
            n, begin = int(ranges[le, s] & 0xffffffff), int(ranges[le, s] >> 32)
            if s != rank:
                slots[le, s, :n] = y[le, begin:begin + n].view(torch.int16).cpu()
    sums = []
    for hint in hints:
        st.expected_rows = hint
        st.combine_send_slots.view(torch.int16).fill_(0x7FC0)
        out = torch.zeros((t, h), dtype=torch.bfloat16, device="cuda")
        st.combine(y, topk_all[rank].cuda(), w[rank].cuda(), out)
        torch.cuda.synchronize()
        assert torch.equal(st.combine_send_slots.view(torch.int16).view(e // r, r, t, h).cpu(), slots)
        sums.append(out.cpu())
    assert all(torch.equal(sums[0], o) for o in sums[1:])


@pytest.mark.parametrize("r,e,h,hints,parts", [
    (8, 16, 512, (8192, 8193), (2, 1)), (8, 16, 1024, (8192, 8193), (2, 1)),  # rows of less than 4 KB: past 8192 whole
    (8, 16, 1920, (8192, 8193, 16384), (2, 1, 1)),
    (8, 16, 2048, (8193, 16384), (2, 2)),  # rows of 4 KB: in two parts throughout
    (8, 256, 2048, (8193,), (2,)), (8, 264, 2048, (8192, 8193), (2, 1)),  # past 256 experts whole
    (2, 16, 7168, (8192, 8193, 8629, 8630), (4, 4, 4, 0)),  # rows of 14 KB in four parts; 132 MB with the tokens' rows, two launches
    (2, 258, 7168, (8193, 15066, 15067), (1, 1, 0)),  # and 220
])
@pytest.mark.filterwarnings("ignore:DEBUG")  # the graph is written out
def test_combine_past_8192_rows_in_parts(rt, r, e, h, hints, parts, tmp_path):
    """How the rows of a single-launch combine are cut, and whether it is one, changes no row and no sum."""
    rank, t, k = 1, 1025, 8
    x_all, topk_all, w = make_world(r, t, h, k, e, seed=h + r, drop=30)
    st, world = dispatch_on_gpu(rt, x_all, topk_all, rank, e, t, O.ROW_BF16, one_call=True)
    y = torch.randn(st.packed_recv_x.shape, generator=torch.Generator().manual_seed(h)).bfloat16().cuda()
    world.combine_from_peers(st, mode=1, seed=5)
    topk, weights, got = topk_all[rank].cuda(), w[rank].cuda(), []
    for hint in (0,) + hints:
        st.combine_send_slots.view(torch.int16).fill_(0x7FC0)
        out = torch.zeros((t, h), dtype=torch.bfloat16, device="cuda")
        if hint == 0:  # the two calls, which also move the rank's own rows to the staging area
            st.expected_rows = 8192
            st.combine_send(y)
            st.combine_recv(topk, weights, out)
        else:
            st.expected_rows = hint
            st.combine(y, topk, weights, out)
            launched = kernels_launched(lambda: st.combine(y, topk, weights, out), tmp_path)
            fused = [n for name, n in launched.items() if "fused" in name]
            reduce_waves = t * -(-h // 512)
            rows = min(hint + hint // 8 + 16, e * t)
            cut = parts[hints.index(hint)]
            assert fused == ([-(-reduce_waves // 4) + min(16384, -(-rows * cut // 4))] if cut else []), hint
        torch.cuda.synchronize()
        got.append((st.combine_send_slots.view(torch.int16).clone(), out))
    assert not torch.equal(got[0][0], torch.full_like(got[0][0], 0x7FC0))
    for slots, out in got[1:]:
        assert torch.equal(slots, got[0][0]) and torch.equal(out, got[0][1])


_FORMS = ("ll_combine_fused_kernelILb0", "ll_combine_fused_kernelILb1", "ll_combine_fused_past_caches_kernel")


def combine_launched(call, tmp_path):
    """The combine kernel of a call, by its node in a captured graph."""
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    graph.enable_debug_mode()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        call()
    graph.debug_dump(str(tmp_path / "graph.dot"))
    names = set(re.findall(r"ll_combine_\w*?kernel(?:I(?:Lb[01]E)+E)?", (tmp_path / "graph.dot").read_text()))
    assert len(names) == 1
    return names.pop()


@pytest.mark.filterwarnings("ignore:DEBUG")  # the graph is written out
@pytest.mark.parametrize("h,k,hints", [(7168, 8, (1404, 1405, 6085, 6086)),  # 48 and 192 MB: three forms of the launch
                                       (5504, 8, (1876, 1877, 7972, 7973))])  # rows with a last piece of three quarters
def test_combine_whose_accesses_stream_in_part(rt, h, k, hints, tmp_path):
    """Which accesses of the single-launch combine carry the streaming hint changes no row and no sum."""
    r, rank, t, e = 8, 3, 40, 64
    x_all, topk_all, w = make_world(r, t, h, k, e, seed=h, drop=9)
    st, world = dispatch_on_gpu(rt, x_all, topk_all, rank, e, 160, O.ROW_BF16, one_call=True)
    y = torch.randn(st.packed_recv_x.shape, generator=torch.Generator().manual_seed(h)).bfloat16().cuda()
    world.combine_from_peers(st, mode=1, seed=5)
    topk, w, got = topk_all[rank].cuda(), w[rank].cuda(), []
    for hint in (0,) + hints:
        st.combine_send_slots.view(torch.int16).fill_(0x7FC0)
        out = torch.zeros((t, h), dtype=torch.bfloat16, device="cuda")
        if hint == 0:
            st.combine_send(y)
            st.combine_recv(topk, w, out)
        else:
            st.expected_rows = hint
            st.combine(y, topk, w, out)
            form = combine_launched(lambda: st.combine(y, topk, w, out), tmp_path)
            assert form.startswith(_FORMS[(0, 1, 1, 2)[hints.index(hint)]]), hint
        torch.cuda.synchronize()
        got.append((st.combine_send_slots.view(torch.int16).clone(), out.view(torch.int16).clone()))
    assert all(torch.equal(a, b) for other in got[1:] for a, b in zip(got[0], other))


@pytest.mark.filterwarnings("ignore:DEBUG")  # the graph is written out
@pytest.mark.parametrize("t,h,streams", [(164, 7168, 0), (165, 7168, 1), (214, 5504, 0), (215, 5504, 1)])
def test_combine_without_row_return_streams_by_what_it_gathers(rt, t, h, streams, tmp_path):
    """18 MB of gathered rows, whatever number of rows is expected; and the sums of the two phases."""
    r, rank, k, e = 8, 3, 8, 64
    x_all, topk_all, w = make_world(r, t, h, k, e, seed=t, drop=9)
    st, world = dispatch_on_gpu(rt, x_all, topk_all, rank, e, 256, O.ROW_BF16, one_call=True)
    y = torch.randn(st.packed_recv_x.shape, generator=torch.Generator().manual_seed(h)).bfloat16().cuda()
    world.combine_from_peers(st, mode=1, seed=5)
    topk, w = topk_all[rank].cuda(), w[rank].cuda()
    want = torch.zeros((t, h), dtype=torch.bfloat16, device="cuda")
    st.combine_send(y)
    st.combine_recv(topk, w, want)
    st.combine_send_slots.view(torch.int16).fill_(0x7FC0)
    for hint in (t * k, 8192):
        st.expected_rows = hint
        out = torch.zeros((t, h), dtype=torch.bfloat16, device="cuda")
        st.combine(y, topk, w, out, zero_copy=True)
        assert torch.equal(out.view(torch.int16), want.view(torch.int16)), hint
        form = combine_launched(lambda: st.combine(y, topk, w, out, zero_copy=True), tmp_path)
        assert form.startswith(_FORMS[streams]), hint
    assert (st.combine_send_slots.view(torch.int16) == 0x7FC0).all()


@pytest.mark.parametrize("t,h,k,e,hints", [
    (64, 4096, 8, 64, (3399, 3400)),  # 2048 workgroups, which the chip holds at once, and 2049
    (61, 1024, 3, 512, (3572, 3573)),  # the same with more than 256 segments
])
def test_combine_of_one_round_of_workgroups_and_of_more(rt, t, h, k, e, hints):
    """Both forms of the single launch give the two calls' sums and rows."""
    r, rank = 8, 3
    x_all, topk_all, w = make_world(r, t, h, k, e, seed=h, drop=9)
    st, world = dispatch_on_gpu(rt, x_all, topk_all, rank, e, t, O.ROW_BF16, one_call=True)
    y = torch.randn(st.packed_recv_x.shape, generator=torch.Generator().manual_seed(h)).bfloat16().cuda()
    world.combine_from_peers(st, mode=1, seed=5)
    topk, w, got = topk_all[rank].cuda(), w[rank].cuda(), []
    for hint in (0,) + hints:
        st.combine_send_slots.view(torch.int16).fill_(0x7FC0)
        out = torch.zeros((t, h), dtype=torch.bfloat16, device="cuda")
        if hint == 0:
            st.combine_send(y)
            st.combine_recv(topk, w, out)
        else:
            st.expected_rows = hint
            st.combine(y, topk, w, out)
        torch.cuda.synchronize()
        got.append((st.combine_send_slots.view(torch.int16).clone(), out.view(torch.int16).clone()))
    assert all(torch.equal(a, b) for other in got[1:] for a, b in zip(got[0], other))


def test_all_to_all_calls_let_other_threads_run(rt):
    """A launch of the all-to-all surface releases the GIL.  The interpreter is told never to take it away from a
    running thread, and nothing else in the loop gives it up, so the second thread gets on only through the calls."""
    import _thread
    import sys
    import time
    r, rank, t, h, k, e = 4, 1, 64, 512, 4, 16
    a2a = rt.ll.AllToAllState(rt.ll.LLShape(r, rank, e, t, h, k, O.ROW_BF16))
    world = rt.lb.LoopbackWorld(r, rank, seed=3)
    world.synthesise(t, h, k, e)
    x, topk = world.own_inputs()
    w, out = torch.ones((t, k), device="cuda"), torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
    routed = torch.zeros((r, e), dtype=torch.int32, device="cuda")
    calls = [lambda: a2a.dispatch_send(x, topk), lambda: a2a.exchange_metadata(routed),
             lambda: a2a.dispatch_recv_ordered(routed), lambda: a2a.dispatch_recv(),
             lambda: a2a.combine_send(a2a.packed_recv_x), lambda: a2a.combine_recv(topk, w, out)]
    for call in calls:
        call()
    torch.cuda.synchronize()
    interval = sys.getswitchinterval()
    for i, call in enumerate(calls):
        ran = []
        sys.setswitchinterval(1000)
        try:
            _thread.start_new_thread(lambda: ran.append(True), ())
            for _ in range(20000):
                if ran:
                    break
                call()
            got_on = bool(ran)
        finally:
            sys.setswitchinterval(interval)
        while not ran:
            time.sleep(0.001)
        torch.cuda.synchronize()
        assert got_on, i


def test_all_to_all_state_with_attributes_of_a_subclass(rt):
    """A subclass may keep an attribute where it likes (a property with a setter): the calls get what it says."""
    class Counting(rt.ll.AllToAllState):
        asked = 0

        @property
        def expected_rows(self):
            type(self).asked += 1
            return self._rows

        @expected_rows.setter
        def expected_rows(self, rows):
            self._rows = rows

    r, rank, t, h, k, e = 2, 0, 16, 256, 2, 4
    x_all, topk_all, w = make_world(r, t, h, k, e, seed=5)
    x, topk, weights = x_all[rank].cuda(), topk_all[rank].cuda(), w[rank].cuda()
    results = []
    for kind in (rt.ll.AllToAllState, Counting):
        me = kind(rt.ll.LLShape(r, rank, e, t, h, k, O.ROW_BF16))
        me.dispatch_send(x, topk)
        routed = torch.stack([me.send_count, torch.zeros_like(me.send_count)])
        lo, hi = (int(v) for v in me.send_cumsum[rank:rank + 2].cpu())
        me.recv_by_source[:hi - lo] = me.send_rows[lo:hi]
        me.exchange_metadata(routed)
        me.dispatch_recv_ordered(routed)
        me.send_flat.zero_(), me.recv_flat.fill_(1)
        me.combine_send(me.packed_recv_x)
        out = torch.empty((t, h), dtype=torch.bfloat16, device="cuda")
        me.combine_recv(topk, weights, out)
        torch.cuda.synchronize()
        results.append((me.packed_recv_count.clone(), me.send_flat.clone(), out))
    assert Counting.asked == 2
    assert all(torch.equal(a, b) for a, b in zip(*results)) and int(results[0][0].sum()) > 0
