"""CPU-only checks: the C-ABI library exports what include/deepep_hip.h declares, size
arithmetic matches the oracle, and the host module's argument checks raise the reference's
EPException text.  No kernel is launched here."""
import decimal
import os
import re
import subprocess

import numpy as np
import pytest
import torch

from oracle import deepep_oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "deepep_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(deepep_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from deepep_efa_amd import _capi
    lib = _capi.load()
    declared = _declared_symbols()
    assert len(declared) >= 20
    for name in declared:
        assert hasattr(lib, name), f"{name} is declared in include/deepep_hip.h but not exported"
        assert name in _capi.PROTOTYPES, f"{name} has no ctypes prototype"
    assert sorted(_capi.PROTOTYPES) == declared


def test_abi_revision_is_the_same_everywhere():
    """The header's revision, what the built library reports and what the integration notes tell a
    maintainer to gate on are one number."""
    from deepep_efa_amd import _capi
    header = open(os.path.join(ROOT, "include", "deepep_hip.h")).read()
    revision = int(re.search(r"#define\s+DEEPEP_HIP_ABI_VERSION\s+(\d+)", header).group(1))
    assert _capi.load().deepep_abi_version() == revision
    notes = open(os.path.join(ROOT, "INTEGRATION.md")).read()
    assert re.search(r"`deepep_abi_version\(\)` is (\d+)", notes).group(1) == str(revision)
    # every *_workspace_bytes function the header declares is named there too
    for name in _declared_symbols():
        if name.endswith("_workspace_bytes"):
            assert name in notes, f"INTEGRATION.md does not mention {name}"


@pytest.mark.parametrize("hidden", [128, 512, 2048, 7168])
def test_row_sizes_match_oracle(hidden):
    from deepep_efa_amd import _capi
    lib = _capi.load()
    for fmt in (O.ROW_BF16, O.ROW_FP8, O.ROW_FP8_POW2, O.ROW_FP8_UE8M0):
        assert lib.deepep_ll_row_data_bytes(hidden, fmt) == O.row_data_bytes(hidden, fmt)
        assert lib.deepep_ll_row_scale_bytes(hidden, fmt) == O.row_scale_bytes(hidden, fmt)
        assert lib.deepep_ll_row_stride(hidden, fmt) == O.row_stride(hidden, fmt)


@pytest.mark.parametrize("m,h,r,e", [(128, 7168, 32, 256), (1, 128, 2, 2), (8192, 7168, 64, 256), (256, 2048, 8, 288)])
def test_size_hint_matches_oracle(m, h, r, e):
    from deepep_efa_amd import _capi
    import deep_ep
    assert _capi.load().deepep_get_low_latency_rdma_size_hint(m, h, r, e) == O.get_low_latency_rdma_size_hint(m, h, r, e)
    assert deep_ep.Buffer.get_low_latency_rdma_size_hint(m, h, r, e) == O.get_low_latency_rdma_size_hint(m, h, r, e)


def test_host_argument_checks_without_a_gpu():
    from deepep_efa_amd import _capi
    lib = _capi.load()
    # shape checks run before anything touches the device
    rc = lib.deepep_per_token_cast_to_fp8(None, 4, 100, 1, None, None, None)
    assert rc != 0
    assert lib.deepep_last_error().decode() == "Failed: Assertion error cast.hip:%d 'num_rows >= 0 && num_cols > 0 && num_cols %% 128 == 0'" % \
        int(re.search(r"cast\.hip:(\d+)", lib.deepep_last_error().decode()).group(1))
    rc = lib.deepep_ll_combine_recv(None, None, None, None, 4, 7168, 0, 256, 128, 0, None, None)
    assert rc != 0 and "num_topk > 0" in lib.deepep_last_error().decode()
    rc = lib.deepep_moe_routing_sort(None, -1, 8, None, None, None, None, None, 0, None)
    assert rc != 0 and lib.deepep_last_error().decode().startswith("Failed: Assertion error layout.hip:")
    with pytest.raises(_capi.DeepEPError):
        _capi.check(rc)


def _kernel_metadata():
    """name -> metadata of every kernel in the built library: the msgpack notes of its code objects."""
    msgpack = pytest.importorskip("msgpack")
    blob = open(os.path.join(ROOT, "deepep_efa_amd", "libdeepep_hip.so"), "rb").read()
    kernels = {}
    for m in re.finditer(rb"\x07\0\0\0(....)\x20\0\0\0AMDGPU\0\0", blob, re.S):  # note: name size, data size, type 32, name
        note = blob[m.end():m.end() + int.from_bytes(m.group(1), "little")]
        for k in msgpack.unpackb(note, strict_map_key=False)["amdhsa.kernels"]:
            kernels[k[".name"]] = k
    return kernels


@pytest.mark.parametrize("kernel", ["ll_combine_fused_kernelILb0ELb1EE", "ll_combine_recv_kernelILb0EE", "combine_reduce_kernelILb0EE",
                                    "combine_reduce_kernelILb1EE"])
def test_reduces_leave_room_for_eight_waves_a_simd(kernel):
    """512 registers a lane and SIMD, eight waves: 64 each, and none kept in memory instead."""
    found = [k for name, k in _kernel_metadata().items() if kernel in name]
    assert len(found) == 1 and found[0][".vgpr_count"] <= 64 and found[0][".private_segment_fixed_size"] == 0


def test_ranked_send_leaves_room_for_eight_waves_a_simd():
    """Every row format, streaming or not: the kernel has no other way to hide its trips to memory."""
    found = [k for name, k in _kernel_metadata().items() if "ll_send_ranked_kernel" in name]
    assert len(found) == 8
    assert all(k[".vgpr_count"] <= 64 and k[".private_segment_fixed_size"] == 0 for k in found)


@pytest.mark.parametrize("tokens,seen_tokens,seen_rows,want", [
    (128, 0, 0, 1024),          # nothing seen yet: what a balanced world sends
    (0, 0, 0, 8),
    (128, 128, 900, 1024),      # less than balanced
    (128, 128, 5000, 5000),
    (4, 1, 2100, 2100),         # other ranks' rows do not grow with this rank's tokens
    (1000, 1, 2100, 8000),
    (1000, 100, 40000, 40000),
    (4, 1000, 60000, 240),      # the decode step behind a prefill
    (0, 1000, 60000, 8),
    (128, 128, 2 ** 32 - 1, 256 * 128),  # never more than there is room for
])
def test_rows_expected_of_a_batch_follow_the_last_one(tokens, seen_tokens, seen_rows, want):
    from deepep_efa_amd import _capi
    lib = _capi.load()
    got = lib.deepep_ll_expected_rows(tokens, 8, 256, 128 if tokens <= 128 else 1024, seen_tokens << 32 | seen_rows)
    assert got == want
    if tokens <= 4:  # a decode batch stays in the single launch
        assert lib.deepep_ll_dispatch_is_single_launch(tokens, 8, 256, 128, got) == 1


@pytest.mark.parametrize("t,h,k,e,fmt,rows,want", [
    (1024, 512, 8, 64, 1, 8192, 1),                                 # 8192 entries and rows, whatever these hold
    (1408, 512, 8, 64, 0, 0, 1), (1409, 512, 8, 64, 0, 0, 0),       # rows of one wave: 44 rounds of the counting workgroup
    (1408, 1024, 8, 64, 1, 0, 1), (1409, 1024, 8, 64, 1, 0, 0),
    (5416, 512, 2, 64, 1, 0, 1), (5417, 512, 2, 64, 1, 0, 0),       # and 14 M entries for the send workgroups
    (3500, 128, 8, 64, 0, 0, 0),
    (3546, 1024, 8, 64, 0, 0, 1), (3547, 1024, 8, 64, 0, 0, 0),     # four tokens a workgroup: 24 M
    (1773, 2176, 8, 64, 1, 0, 1), (1774, 2176, 8, 64, 1, 0, 0),     # one
    (768, 1152, 32, 256, 1, 0, 1), (769, 1152, 32, 256, 1, 0, 0),   # 96 rounds of four waves
    (1000, 1152, 16, 64, 1, 0, 1), (2000, 1152, 16, 64, 1, 0, 1),   # and of eight
    (140, 1920, 64, 256, 1, 0, 0), (140, 2048, 64, 256, 1, 0, 1),   # more than 32 selections: rows of 2 KB
    (140, 896, 64, 256, 0, 0, 0), (140, 1024, 64, 256, 0, 0, 1),
    (600, 2048, 8, 64, 1, (72 << 20) // 2128, 1), (600, 2048, 8, 64, 1, (72 << 20) // 2128 + 1, 0),  # 72 MB of rows
    (600, 128, 8, 256, 0, 96 << 10, 1), (600, 128, 8, 256, 0, (96 << 10) + 1, 0),
    (0, 512, 8, 64, 1, 20000, 1), (0, 7168, 8, 64, 1, 20000, 0),    # a rank without tokens
])
def test_batches_that_a_one_call_dispatch_takes_in_one_launch(t, h, k, e, fmt, rows, want):
    from deepep_efa_amd import _capi
    lib, m = _capi.load(), max(t, 4096)
    rows = rows or t * k
    assert lib.deepep_ll_dispatch_takes_one_launch(t, h, k, e, m, fmt, rows) == want
    if lib.deepep_ll_dispatch_is_single_launch(t, k, e, m, rows):
        assert want == 1


@pytest.mark.parametrize("tokens,a,b,want", [
    (1000, (0, 0), (0, 0), 8000),
    (1000, (1000, 160000), (0, 0), 160000),           # one report so far
    (1000, (0, 0), (1000, 160000), 160000),
    (1000, (1000, 160000), (1000, 160000), 160000),   # the same layer again
    (1000, (1000, 160000), (1000, 10000), 40000),     # a hot layer and a cold one in turn: neither sizes the other
    (1000, (1000, 10000), (1000, 160000), 40000),
    (1000, (1000, 160000), (1000, 500), 35777),       # less than balanced is balanced
    (1000, (1000, 160000), (3, 500), 160000),         # a smaller batch says nothing of a larger one
    (1000, (3, 500), (1000, 160000), 160000),
    (1000, (3, 500), (4, 50000), 20000),              # unless there is nothing else
    (4, (1000, 60000), (1000, 60000), 240),           # the decode step behind a prefill
    (4, (1000, 60000), (4, 60), 120),
])
def test_rows_expected_of_a_batch_lie_between_the_last_two(tokens, a, b, want):
    from deepep_efa_amd import _capi
    got = _capi.load().deepep_ll_expected_rows_of_two(tokens, 8, 256, 1024, a[0] << 32 | a[1], b[0] << 32 | b[1])
    assert got == want


@pytest.mark.parametrize("flag,taken", [
    (True, True), (False, True), (None, True), (1, True), (np.bool_(False), True), (0.0, True),
    ("False", False), ([], False), ((1,), False), ({}, False)])
def test_truth_values_are_taken_by_pybind11s_rules(flag, taken):
    from deepep_efa_amd import deep_ep_cpp
    x = torch.zeros((1, 128), dtype=torch.bfloat16)  # not on a GPU: what takes the flag refuses the tensor
    with pytest.raises(RuntimeError if taken else TypeError, match="is_cuda" if taken else "incompatible"):
        deep_ep_cpp.per_token_cast_to_fp8(x, flag, False)


@pytest.mark.parametrize("number,taken", [
    (3, True), (True, True), (np.int64(3), True), (decimal.Decimal(3), True), (torch.tensor(3), True),
    (3.0, False), ("3", False), (None, False), (2 ** 31, False), (-2 ** 40, False)])
def test_numbers_are_taken_by_pybind11s_rules(number, taken):
    from deepep_efa_amd import deep_ep_cpp
    member = torch.zeros((1, 8), dtype=torch.bool)
    with pytest.raises(RuntimeError if taken else TypeError, match="is_cuda" if taken else "incompatible"):
        deep_ep_cpp.channel_prefix_matrix(member, number)


def test_calls_refuse_what_is_not_their_object():
    from deepep_efa_amd import deep_ep_cpp
    x, idx = torch.zeros((1, 128), dtype=torch.bfloat16), torch.zeros((1, 2), dtype=torch.int64)
    for other in (None, 3, deep_ep_cpp.AllToAllCalls(2, 0, 2, 1, 128, 2, 0)):  # what a destroyed Buffer's runtime is
        with pytest.raises(TypeError, match="incompatible"):
            deep_ep_cpp.low_latency_dispatch(other, x, idx, None, None, 1, 2, True, False, False, False, False)
        with pytest.raises(TypeError, match="incompatible"):
            deep_ep_cpp.get_dispatch_layout(other, idx, 2, None, False, False)
    with pytest.raises(TypeError, match="incompatible"):
        deep_ep_cpp.a2a_dispatch_send(None, {}, x, idx)


def test_plain_calls_raise_the_modules_exception():
    from deepep_efa_amd import deep_ep_cpp
    with pytest.raises(deep_ep_cpp.EPException, match=r"^Failed: Assertion error deep_ep_cpp.cpp:\d+ 'x.dim\(\) == 2"):
        deep_ep_cpp.per_token_cast_to_fp8(torch.zeros(128, dtype=torch.bfloat16), False, False)
    with pytest.raises(TypeError, match="wrong number of arguments"):
        deep_ep_cpp.moe_routing_sort()
    if not torch.cuda.is_available():  # PyTorch's own kinds come through
        calls = deep_ep_cpp.AllToAllCalls(2, 0, 2, 1, 128, 2, 0)
        state = dict.fromkeys(("send_rows", "send_count", "send_expert_prefix", "send_counts", "send_cumsum", "pair_slot",
                               "workspace"), torch.zeros(1))
        with pytest.raises(torch.AcceleratorError):
            deep_ep_cpp.a2a_dispatch_send(calls, dict(state, send_capacity=8), torch.zeros((1, 128), dtype=torch.bfloat16),
                                          torch.zeros((1, 2), dtype=torch.int64))


def test_a_reduce_without_a_buffer_to_reduce_from_is_refused():
    """recv_flat may be given up by a caller who always passes the transport's own buffer."""
    from deepep_efa_amd import deep_ep_cpp
    calls, t = deep_ep_cpp.AllToAllCalls(2, 0, 2, 1, 128, 2, 0), torch.zeros((1, 2))
    state = dict(recv_flat=None, send_expert_prefix=t, pair_slot=t)
    with pytest.raises(TypeError, match="recv_flat"):
        deep_ep_cpp.a2a_combine_recv(calls, state, t.long(), t, t.bfloat16(), None, 0, False)


def test_combine_reduce_takes_its_arguments_by_position_and_by_name():
    from deepep_efa_amd import deep_ep_cpp
    x = torch.zeros((1, 128), dtype=torch.bfloat16)  # refused for not being on a GPU once the arguments are sorted out
    ids, cumsum, member = torch.zeros(1, dtype=torch.int64), torch.zeros(9, dtype=torch.int64), torch.zeros((1, 8), dtype=torch.bool)
    by_position = (x, None, ids, cumsum, member)
    names = ("recv_x", "recv_topk_weights", "sorted_token_ids", "send_cumsum", "is_token_in_rank")
    for args, kwargs in ((by_position, {}), (by_position, dict(row_of_pair=None)), (by_position + (None,) * 3, {}),
                         ((), dict(zip(names, by_position))), (by_position[:3], dict(zip(names[3:], by_position[3:])))):
        with pytest.raises(RuntimeError, match="is_cuda"):
            deep_ep_cpp.combine_reduce(*args, **kwargs)
    for args, kwargs in ((by_position[:4], {}), (by_position + (None,) * 4, {}), (by_position, dict(recv_x=x)),
                         (by_position, dict(bias=None)), (by_position, dict(bias_0=3)), ((3,) + by_position[1:], {})):
        with pytest.raises(TypeError):
            deep_ep_cpp.combine_reduce(*args, **kwargs)


def test_exchange_metadata_wants_a_matrix():
    from deepep_efa_amd import ll_runtime
    for shape in ((8,), (2, 2, 4)):
        with pytest.raises(ValueError):
            ll_runtime.exchange_metadata(torch.zeros(shape, dtype=torch.int32), 0, 8, 16)


def test_config_follows_reference_rules():
    import deep_ep
    cfg = deep_ep.Config(20, 6, 256, 6, 250)
    assert cfg.num_max_rdma_chunked_recv_tokens == 252  # rounded up to a multiple of the send chunk
    assert cfg.num_sms == 20 and cfg.num_max_nvl_chunked_send_tokens == 6
    # csrc/config.hpp:52-74 by hand for 8 ranks, bf16 hidden 7168: see the arithmetic in the test body
    ch, nvl, recv, hb = 10, 8, 256, 14336
    want = ch * nvl * 5 * 4 + ch * nvl * recv * (hb + 8 + 128 * 8 + 128 * 4 + 128 * 4)
    assert cfg.get_nvl_buffer_size_hint(hb, 8) == (want + 127) // 128 * 128
    assert cfg.get_rdma_buffer_size_hint(hb, 8) == 0
    with pytest.raises(RuntimeError, match=r"Failed: Assertion error deep_ep_cpp.cpp:\d+ 'nvl_send < nvl_recv'"):
        deep_ep.Config(20, 300, 256, 6, 128)
    for n in (2, 8, 32, 160):
        assert deep_ep.Buffer.get_dispatch_config(n).num_sms == deep_ep.Buffer.num_sms
        assert deep_ep.Buffer.get_combine_config(n).num_max_rdma_chunked_recv_tokens >= 128
    assert str(deep_ep.topk_idx_t) == "torch.int64"


def test_buffer_needs_a_world():
    import deep_ep
    with pytest.raises(ValueError, match="Either 'group' or 'comm' must be provided"):
        deep_ep.Buffer(None)


def test_c_abi_library_needs_no_torch():
    """The boundary is plain C over device pointers: the library links the HIP runtime and the C/C++
    runtime, nothing from PyTorch, and exports no C++-mangled entry point a caller would have to use."""
    import subprocess
    so = os.path.join(ROOT, "deepep_efa_amd", "libdeepep_hip.so")
    needed = subprocess.run(["readelf", "-d", so], capture_output=True, text=True, check=True).stdout
    libs = re.findall(r"Shared library: \[([^\]]+)\]", needed)
    assert any(lib.startswith("libamdhip64") for lib in libs)
    assert not [lib for lib in libs if "torch" in lib or "c10" in lib or "python" in lib], libs
    header = open(os.path.join(ROOT, "include", "deepep_hip.h")).read()
    code = re.sub(r"/\*.*?\*/", "", header, flags=re.S)  # declarations only, comments cite the reference
    assert 'extern "C"' in code and "torch" not in code and "at::" not in code and "#include <hip" not in code


def test_streams_of_another_device_wait_behind_the_system_scope_fence(tmp_path):
    """An event recorded without the fence is not what they wait for.  Host code against a runtime that keeps a record."""
    torch_dir = os.path.dirname(torch.__file__)
    program = tmp_path / "events"
    build = subprocess.run(
        ["g++", "-O0", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
         f"-I{torch_dir}/include", "-I/opt/rocm/include", os.path.join(ROOT, "tests", "event_of_another_device.cpp"), "-o", str(program),
         f"-L{torch_dir}/lib", "-lc10", f"-Wl,-rpath,{torch_dir}/lib"], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert build.returncode == 0, build.stdout
    ran = subprocess.run([str(program)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert ran.returncode == 0, ran.stdout
