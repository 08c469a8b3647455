"""CPU-only checks of the drop-in boundary: the C ABI library loads and exports every symbol that
include/mam_hip.h declares, the torch operator schemas equal the reference's strings, fake
kernels propagate shapes, the module's host logic follows the reference, and nothing falls
back to a CPU implementation."""
import ctypes
import os
import re

import numpy as np
import pytest
import torch

import mamtorch_amd as mt
from mamtorch_amd import capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "mam_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mam_[a-z_0-9]+)\s*\(", text)))


def test_c_abi_exports_every_declared_symbol():
    names = _declared_symbols()
    assert len(names) >= 12
    assert set(names) == set(capi.EXPORTS)
    lib = ctypes.CDLL(mt._native.HIP_LIB_PATH)
    for n in names:
        assert hasattr(lib, n), "libmam_hip.so does not export %s" % n
    assert lib.mam_version() >= 100
    capi.lib()
    assert capi.lib().mam_error_string(-3).decode() == "workspace missing or too small"


@pytest.mark.parametrize("N, K, M", [(2 ** 24, 128, 64), (2 ** 24 - 64, 128, 64), (128 * 224 * 224 * 4, 160, 32)])
def test_calls_of_more_rows_than_a_list_launch_holds_stay_on_the_dense_tilings(N, K, M):
    # the lists are built by a workgroup of 256 threads per row, and a launch holds less than 2^32 threads
    l = capi.lib()
    assert l.mam_fc_forward_workspace_for(N, K, M, capi.W_MK, 1) == l.mam_fc_forward_workspace(N, K, M)
    below = 2 ** 22
    assert l.mam_fc_forward_workspace_for(below, K, M, capi.W_MK, 1) > l.mam_fc_forward_workspace(below, K, M)


def test_a_km_call_asks_for_the_lists_of_its_inputs_alone():
    l, (N, K, M) = capi.lib(), (16384, 4096, 4096)
    dense = l.mam_fc_forward_workspace(N, K, M)
    km, mk = (l.mam_fc_forward_workspace_for(N, K, M, layout, 1) - dense for layout in (capi.W_KM, capi.W_MK))
    entries = K // 4 + 64
    lists = lambda rows: rows * (8 * entries + 4 * (entries // 8 + 1))
    assert 4 * K * M + lists(N) <= km < 4 * K * M + lists(N) + 16384      # a copy of the weight, lists, samples
    assert 4 * N * K + lists(N + M) <= mk < 4 * N * K + lists(N + M) + 16384      # the searched operand transposed, lists of both


@pytest.mark.parametrize("N, K, M, mk, lists", [
    (256, 4096, 4096, 1, True), (128, 4096, 4096, 1, False), (16384, 4096, 1024, 0, True), (16384, 4001, 1024, 1, True),
    (16384, 16384, 1024, 1, False), (24, 65536, 65536, 1, False)])
def test_describe_names_every_route_that_a_call_can_take(N, K, M, mk, lists):
    l = capi.lib()
    text = ctypes.create_string_buffer(640)
    one = ctypes.c_void_p(256)
    layout = capi.W_MK if mk else capi.W_KM
    describe = lambda: l.mam_fc_forward_describe(one, K, one, K if mk else M, layout, N, K, M, 1, text, 640)
    assert describe() == 0
    with_lists = text.value
    assert (b"magnitude-ordered lists" in with_lists) == lists, with_lists
    capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_DENSE)
    try:
        assert describe() == 0
    finally:
        capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_AUTO)
    dense = text.value
    assert b"lists" not in dense and with_lists.endswith(dense) and (with_lists == dense) == (not lists)
    if lists:
        # what it says the lists need is no more than what the workspace query asks for
        need = int(with_lists.split(b"with ")[1].split()[0])
        assert need <= l.mam_fc_forward_workspace_for(N, K, M, layout, 1)
    assert l.mam_fc_forward_describe(one, K, one, K if mk else M, layout, N, K, M, 1, text, 40) == 0      # cut off, not overrun
    assert len(text.value) < 40


@pytest.mark.parametrize("N, K, M, neurons", [
    (21632, 288, 64, 64), (12608, 768, 192, 64), (2048, 2048, 320, 64), (256, 4096, 192, 64), (1024, 512, 320, 64),
    (2048, 2048, 192, 128), (2048, 2048, 180, 128), (256, 4096, 320, 128), (12608, 768, 256, 128), (12608, 768, 448, 128)])
def test_neurons_per_tile_follow_the_rounds_of_workgroups(N, K, M, neurons):
    # 64 neurons per tile only where they end sooner than 128 (on 256 compute units)
    text = ctypes.create_string_buffer(400)
    one = ctypes.c_void_p(256)
    assert capi.lib().mam_fc_forward_describe(one, K, one, K, capi.W_MK, N, K, M, 1, text, 400) == 0
    assert b"tiles of 32 x %d" % neurons in text.value, text.value


@pytest.mark.parametrize("N, K, M, with_indices, mk, copied", [
    (250, 1001, 517, 1, 1, True), (250, 1001, 517, 0, 1, True), (250, 1001, 517, 0, 0, True), (500, 17, 500, 1, 1, True),
    (4, 63, 10, 1, 1, False), (16, 24, 64, 1, 0, False), (16, 33, 64, 1, 0, True), (30000, 31, 60, 0, 1, False),
    (30000, 31, 60, 1, 1, True), (4000, 130, 1000, 0, 1, False), (4000, 130, 1000, 0, 0, False), (64, 100, 100, 0, 1, True)])
def test_ragged_rows_are_lengthened_where_the_copy_pays(N, K, M, with_indices, mk, copied):
    l = capi.lib()
    text = ctypes.create_string_buffer(400)
    one = ctypes.c_void_p(256)
    layout = capi.W_MK if mk else capi.W_KM
    assert l.mam_fc_forward_describe(one, K, one, K if mk else M, layout, N, K, M, with_indices, text, 400) == 0
    assert (b"lengthen_rows_kernel" in text.value) == copied, text.value
    # the workspace query asks for the copies of the operands exactly where they are made
    need = (l.mam_fc_forward_workspace if with_indices else l.mam_fc_forward_values_workspace)(N, K, M)
    copies = l.mam_fc_forward_workspace_for(N, K, M, layout, with_indices) - need
    assert copies == (_bytes_of_copies(text.value) if copied else 0)


def _bytes_of_copies(text):
    # what mam_fc_forward_describe names for a call on copies, less its partials
    staged = text.split(b"; with less: ")[0]
    partials = re.search(rb"\((\d+) bytes of partials\)", staged)
    return int(re.match(rb"with (\d+) workspace bytes: ", staged).group(1)) - (int(partials.group(1)) if partials else 0)


@pytest.mark.parametrize("N, K, M", [(43120, 1300, 42), (10233, 3316, 78), (250, 1001, 517), (8000, 4095, 256), (70000, 300, 64)])
def test_a_call_that_takes_x_as_it_is_asks_for_no_copy_of_it(N, K, M):
    l = capi.lib()
    text = ctypes.create_string_buffer(640)
    one = ctypes.c_void_p(256)
    assert l.mam_fc_forward_describe(one, K, one, K, capi.W_MK, N, K, M, 1, text, 640) == 0
    lists_first, _, dense = text.value.rpartition(b"otherwise ")
    assert b"last k tile at the end of K" in dense, text.value
    with_lists = l.mam_fc_forward_workspace_for(N, K, M, capi.W_MK, 1)
    capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_DENSE)
    try:
        asked = l.mam_fc_forward_workspace_for(N, K, M, capi.W_MK, 1)
    finally:
        capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_AUTO)
    assert asked - l.mam_fc_forward_workspace(N, K, M) == _bytes_of_copies(dense) < 4 * M * (K + 64) + 256
    assert (asked < with_lists) == (lists_first != b"")


@pytest.mark.parametrize("N, K, M, with_indices", [(70000, 512, 64, 1), (70000, 512, 64, 0), (65535, 1024, 16, 1), (64, 512, 65536, 1),
                                                   (64, 1001, 65536, 1)])
def test_a_transposed_weight_of_any_number_of_rows(N, K, M, with_indices):
    # no row of x (but of a ragged K) and none of w is lengthened: the grid of that copy does not limit the call
    l = capi.lib()
    text = ctypes.create_string_buffer(640)
    one = ctypes.c_void_p(256)
    ldx = (K + 3) // 4 * 4
    assert l.mam_fc_forward_describe(one, ldx, one, M, capi.W_KM, N, K, M, with_indices, text, 640) == 0
    assert b"transpose_kernel + mam_fwd_sx_kernel" in text.value, text.value
    assert l.mam_fc_forward_workspace_for(N, K, M, capi.W_KM, with_indices) >= int(text.value.split(b"with ")[1].split()[0]) > 0


# what an operand's rows are: at 16-byte addresses, begun off them, of a stride off them
ROWS = {"aligned": (256, 0), "shifted": (260, 0), "strided": (256, 1)}


@pytest.mark.parametrize("rows_x", sorted(ROWS))
@pytest.mark.parametrize("rows_w", sorted(ROWS))
@pytest.mark.parametrize("with_indices", [0, 1])
@pytest.mark.parametrize("N, K, M, mk", [(2000, 300, 2000, 1), (1, 4092, 16000, 1), (200, 260, 300, 1), (250, 1001, 517, 1), (31, 1300, 42, 1),
                                         (64, 768, 256, 1), (16384, 4092, 1024, 1), (128, 2048, 4096, 0), (33, 63, 64, 0), (4, 63, 10, 1)])
def test_the_workspace_of_a_call_holds_what_the_call_makes_use_of(N, K, M, mk, with_indices, rows_x, rows_w):
    l = capi.lib()
    text = ctypes.create_string_buffer(900)
    layout = capi.W_MK if mk else capi.W_KM
    (px, dx), (pw, dw) = ROWS[rows_x], ROWS[rows_w]
    whole = (K + 3) // 4 * 4
    row = (M + 3) // 4 * 4 if not mk else whole
    call = (ctypes.c_void_p(px), whole + dx, ctypes.c_void_p(pw), row + dw, layout, N, K, M, with_indices)
    assert l.mam_fc_forward_describe(*call, text, 900) == 0
    lists_first, _, dense = text.value.rpartition(b"otherwise ")
    named = re.match(rb"with (\d+) workspace bytes: ", dense)
    asked, any_rows = l.mam_fc_forward_workspace_at(*call), l.mam_fc_forward_workspace_for(N, K, M, layout, with_indices)
    assert asked <= any_rows or (K % 16 == 0 and named)
    if lists_first:
        assert asked > int(named.group(1)) if named else asked > 0
    else:
        # copies, where the call makes them, and partials, and nothing else
        partials = re.search(rb"\((\d+) bytes of partials\)", dense)
        assert asked == (int(named.group(1)) if named else int(partials.group(1)) if partials else 0)


@pytest.mark.parametrize("N, K, M, range_len", [(16384, 4096, 4096, 1024), (256, 4096, 4096, 1024), (300, 208, 90, 128), (40, 128, 64, 64)])
@pytest.mark.parametrize("with_indices", [0, 1])
def test_whole_ranges_ask_for_their_partials_alone(N, K, M, range_len, with_indices):
    # ranges of whole tiles run on the operands as they are, as they do by any (K, M) weight
    l = capi.lib()
    one, ranges = ctypes.c_void_p(256), -(-K // range_len)
    partials = ranges * N * M * (12 if with_indices else 8)
    assert l.mam_fc_forward_ranges_workspace(N, K, M, range_len, with_indices) == partials
    assert l.mam_fc_forward_ranges_workspace_at(one, K, one, K, capi.W_MK, N, K, M, range_len, with_indices) == partials
    odd = range_len - 3
    assert l.mam_fc_forward_ranges_workspace_at(one, K, one, (M + 3) // 4 * 4, capi.W_KM, N, K, M, odd, with_indices) == -(-K // odd) * partials // ranges


@pytest.mark.parametrize("N, K, M, range_len, turned", [(256, 4096, 4096, 1024, True), (16, 208, 90, 128, True), (15, 4096, 64, 1024, False),
                                                        (64, 208, 90, 104, False), (64, 200, 90, 128, False)])
@pytest.mark.parametrize("with_indices", [0, 1])
def test_whole_ranges_of_a_km_weight_run_on_its_transposed_copy(N, K, M, range_len, turned, with_indices):
    l = capi.lib()
    x, w = ctypes.c_void_p(256), ctypes.c_void_p(260)
    partials = -(-K // range_len) * N * M * (12 if with_indices else 8)
    copy = -(-4 * M * K // 256) * 256 if turned else 0
    assert l.mam_fc_forward_ranges_workspace_at(x, K, w, M, capi.W_KM, N, K, M, range_len, with_indices) == partials + copy


@pytest.mark.parametrize("range_len, lengthened", [(96, False), (160, False), (92, False), (97, True), (100, True), (161, True), (224, True)])
def test_values_of_whole_32_k_tiles_stay_on_them(range_len, lengthened):
    # (a weight at 16-byte addresses is copied for values only where its ranges begin off them)
    l = capi.lib()
    N, K, M = 6300, 4 * range_len, 1536
    x, w, off = ctypes.c_void_p(256), ctypes.c_void_p(256), ctypes.c_void_p(260)
    text = ctypes.create_string_buffer(640)
    assert l.mam_fc_forward_ranges_describe(x, K, w, K, capi.W_MK, N, K, M, range_len, 0, text, 640) == 0
    assert (b"mam_fwd_sx_kernel" in text.value) == lengthened, text.value
    partials = 4 * N * M * 8
    assert (l.mam_fc_forward_ranges_workspace_at(x, K, w, K, capi.W_MK, N, K, M, range_len, 0) > partials) == (range_len % 4 != 0)
    assert (l.mam_fc_forward_ranges_workspace_at(x, K, off, K, capi.W_MK, N, K, M, range_len, 0) > partials) == (range_len >= 96)


@pytest.mark.parametrize("rows_x", sorted(ROWS))
@pytest.mark.parametrize("rows_w", sorted(ROWS))
@pytest.mark.parametrize("with_indices", [0, 1])
@pytest.mark.parametrize("N, K, M, range_len", [(33, 130, 70, 65), (496, 691, 105, 173), (4000, 531, 3712, 133), (160, 3200, 512, 800), (64, 1000, 64, 250),
                                                (40, 8, 5, 2), (9536, 2809, 1432, 703)])
def test_the_workspace_of_ranges_holds_their_copies(N, K, M, range_len, with_indices, rows_x, rows_w):
    l = capi.lib()
    (px, dx), (pw, dw) = ROWS[rows_x], ROWS[rows_w]
    whole = (K + 3) // 4 * 4
    asked = l.mam_fc_forward_ranges_workspace_at(ctypes.c_void_p(px), whole + dx, ctypes.c_void_p(pw), whole + dw, capi.W_MK, N, K, M, range_len,
                                                 with_indices)
    partials = -(-K // range_len) * N * M * (12 if with_indices else 8)
    # never more than the query by sizes, and no copy of x of as many neurons as these
    assert partials <= asked <= l.mam_fc_forward_ranges_workspace(N, K, M, range_len, with_indices)
    if range_len < 32:
        assert asked == partials
    elif with_indices:
        copy = 4 * M * -(-K // range_len) * -(-range_len // 64) * 64
        assert asked == partials + -(-copy // 256) * 256 if M <= 1536 else asked > partials + copy


def test_workspace_queries_are_pure_host_calls():
    l = capi.lib()
    assert l.mam_fc_forward_workspace(12608, 768, 3072) == 0          # enough tiles: no split-K
    ws = l.mam_fc_forward_workspace(256, 4096, 4096)
    assert ws > 0 and ws % (256 * 4096 * 12) == 0                     # splits x (max, min, packed groups) x N*M x 4 B
    assert l.mam_fc_forward_values_workspace(256, 4096, 4096) * 3 == ws * 2
    assert l.mam_fc_forward_workspace(0, 5, 5) == 0


def test_argument_validation_without_a_gpu():
    l = capi.lib()
    # invalid arguments are rejected on the host before anything is launched
    assert l.mam_fc_forward(None, 4, None, 4, 7, None, None, None, None, None, None, 2, 4, 2, None, 0, None) == -1
    assert b"w_layout" in l.mam_last_error()
    assert l.mam_fc_forward(None, 4, None, 4, 0, None, None, None, None, None, None, -1, 4, 2, None, 0, None) == -1
    assert l.mam_fc_forward(None, 4, None, 4, 0, None, None, None, None, None, None, 2, 4, 2, None, 0, None) == -1
    assert b"null" in l.mam_last_error()
    assert l.mam_selection_count(None, None, None, None, 2, 2, 2, 9, None) == -1
    # sizes beyond what the kernels index are refused, not truncated (pointers never dereferenced)
    one = ctypes.c_void_p(16)
    big = 2 ** 30 + 1
    assert l.mam_fc_forward(one, big, one, big, 0, None, one, one, one, None, None, 2, big, 2, None, 0, None) == -2
    assert b"2^30" in l.mam_last_error()
    assert l.mam_fc_backward(one, 4, one, 4, 1, one, one, one, None, None, one, one, big, 4, 2, None) == -2
    assert l.mam_selection_count(one, one, one, one, 2, big, 2, 1, None) == -2
    assert l.mam_fc_forward(one, 2, one, 4, 0, None, one, one, one, None, None, 2, 4, 2, None, 0, None) == -1
    assert b"leading dimension" in l.mam_last_error()
    # empty problems are a no-op
    assert l.mam_fc_forward(None, 4, None, 4, 0, None, None, None, None, None, None, 0, 4, 2, None, 0, None) == 0
    assert l.mam_selection_count(None, None, None, None, 0, 2, 2, 0, None) == 0


REFERENCE_SCHEMAS = {
    # mamtorch/kernel/v1/csrc/register_functions.cpp:21-24
    ("mamtorch_kernel_v1", "fullyconnected"): "mamtorch_kernel_v1::fullyconnected(Tensor a, Tensor b) -> Tensor[]",
    ("mamtorch_kernel_v1", "fullyconnected_backward"):
        "mamtorch_kernel_v1::fullyconnected_backward(Tensor a, Tensor b, Tensor grad, Tensor argmax, Tensor argmin) -> Tensor[]",
    # mamtorch/kernel/v4/csrc/register_functions.cpp:10-14
    ("mamtorch_kernel_v4", "fullyconnected"): "mamtorch_kernel_v4::fullyconnected(Tensor a, Tensor b) -> Tensor[]",
    ("mamtorch_kernel_v4", "fullyconnected_fast"): "mamtorch_kernel_v4::fullyconnected_fast(Tensor a, Tensor b) -> Tensor",
    ("mamtorch_kernel_v4", "fullyconnected_backward"):
        "mamtorch_kernel_v4::fullyconnected_backward(Tensor a, Tensor b, Tensor grad, Tensor argmax, Tensor argmin) -> Tensor[]",
}


@pytest.mark.parametrize("key", sorted(REFERENCE_SCHEMAS))
def test_operator_schemas_match_the_reference(key):
    ns, name = key
    op = getattr(getattr(torch.ops, ns), name).default
    assert str(op._schema) == REFERENCE_SCHEMAS[key]


def test_python_surface_matches_reference_layout():
    assert callable(mt.kernel.v1.fullyconnected)
    assert callable(mt.kernel.v4.fullyconnected)
    assert callable(mt.kernel.v4.fullyconnected_fast)
    assert mt.nn.FullyConnected.__name__ == "FullyConnected"
    assert callable(mt.sparse.fullyconnected)


def test_no_cpu_fallback():
    a, b = torch.randn(3, 4), torch.randn(4, 5)
    with pytest.raises(NotImplementedError):
        mt.kernel.v1.fullyconnected(a, b)
    with pytest.raises(NotImplementedError):
        mt.kernel.v4.fullyconnected_fast(a, b)
    layer = mt.nn.FullyConnected(4, 5)
    with pytest.raises(NotImplementedError):
        layer(a)


def test_fake_kernels_propagate_shapes():
    a = torch.empty(7, 11, device="meta")
    b = torch.empty(11, 5, device="meta")
    w = torch.empty(5, 11, device="meta")
    c, amax, amin = torch.ops.mamtorch_kernel_v4.fullyconnected(a, b)
    assert c.shape == (7, 5) and c.dtype == torch.float32
    assert amax.dtype == torch.int32 and amin.shape == (7, 5)
    assert torch.ops.mamtorch_kernel_v4.fullyconnected_fast(a, b).shape == (7, 5)
    c, amax, amin = torch.ops.mamtorch_kernel_v1.fullyconnected(a, b)
    assert c.shape == (7, 5)
    c, amax, amin, sel = torch.ops.mamtorch_kernel_v4.fullyconnected_wt(a, w, None, False)
    assert sel.shape == (0, 7, 5)
    c, amax, amin, sel = torch.ops.mamtorch_kernel_v4.fullyconnected_wt(a, w, None, True)
    assert c.shape == (7, 5) and sel.shape == (4, 7, 5)
    g = torch.empty(7, 5, device="meta")
    ag, bg = torch.ops.mamtorch_kernel_v4.fullyconnected_backward(a, b, g, amax, amin)
    assert ag.shape == (7, 11) and bg.shape == (11, 5)
    ag, wg = torch.ops.mamtorch_kernel_v4.fullyconnected_wt_backward(a, w, g, amax, amin, sel)
    assert ag.shape == (7, 11) and wg.shape == (5, 11)
    with pytest.raises(RuntimeError):
        torch.ops.mamtorch_kernel_v4.fullyconnected(a, torch.empty(12, 5, device="meta"))


def test_module_constructor_and_repr():
    torch.manual_seed(0)
    layer = mt.nn.FullyConnected(784, 256)
    assert layer.weight.shape == (256, 784) and layer.bias.shape == (256,)
    # the draws are fp32: the largest one can round up to the fp32 value of the bound
    bound = float(np.float32(1 / 784 ** 0.5))
    assert float(layer.weight.detach().abs().max()) <= bound and float(layer.bias.detach().abs().max()) <= bound
    assert (layer.beta, layer.alpha) == (0.0, 1.0)
    assert repr(layer) == "MAM@FullyConnected(in_features=784, out_features=256, bias=True)"
    layer = mt.nn.FullyConnected(8, 4, bias=False, splits=3, relu_in=True, vcon_steps=10, vcon_expand=True)
    assert layer.bias is None
    assert (layer.in_subfeatures, layer.in_subfeatures_last) == (3, 2)
    assert repr(layer) == ("MAM@FullyConnected(in_features=8, out_features=4, bias=False, vcon_steps=10, "
                           "vcon_type=linear, splits=3, vcon_expand=True, relu_in=True)")
    assert sorted(n for n, _ in mt.nn.FullyConnected(3, 2).state_dict().items()) == ["bias", "weight"]


def test_vanishing_contribution_schedule():
    layer = mt.nn.FullyConnected(8, 4, vcon_steps=4)
    assert (layer.beta, layer.alpha) == (1.0, 0.0)
    betas = []
    for _ in range(5):
        layer.vcon_step()
        betas.append(layer.beta)
    assert betas[:3] == [0.75, 0.5, 0.25] and betas[3] == 0 and betas[4] == 0
    assert layer.alpha == 1.0
    layer = mt.nn.FullyConnected(8, 4, vcon_steps=3, vcon_type="exponential", vcon_eps=1e-3)
    layer.vcon_step()
    assert abs(layer.beta - 0.1) < 1e-12 and abs(layer.alpha - 0.9) < 1e-12
    layer.vcon_step(); layer.vcon_step()
    assert layer.beta == 0 or abs(layer.beta - 1e-3) < 1e-15   # gamma**3 lands on eps up to rounding
    layer.vcon_step()
    assert layer.beta == 0
    layer = mt.nn.FullyConnected(8, 4, vcon_steps=2, vcon_expand=True, splits=2)
    layer.vcon_step()
    assert layer.alpha == 0.5 * 8 / 4
    layer = mt.nn.FullyConnected(8, 4, vcon_steps=2, vcon_type="cosine")
    with pytest.raises(Exception, match="vcon_type 'cosine' is not supported"):
        layer.vcon_step()
    layer = mt.nn.FullyConnected(8, 4, vcon_steps=-1)
    with pytest.raises(Exception, match="Invalid value for vcon_steps"):
        layer.vcon_step()


def test_selection_count_requires_store_args():
    layer = mt.nn.FullyConnected(8, 4)
    with pytest.raises(Exception, match="store_args is False"):
        layer.reset_selection_count()
    with pytest.raises(Exception, match="store_args is False"):
        layer.update_selection_count()
    layer = mt.nn.FullyConnected(8, 4, store_args=True)
    with pytest.raises(Exception, match="No argmax or argmin"):
        layer.update_selection_count()
    layer.reset_selection_count()
    assert layer.max_selection_count.dtype == torch.int32 and layer.max_selection_count.shape == (4, 8)
    assert int(layer.min_selection_count.sum()) == 0


def test_bench_refuses_more_than_one_gpu():
    """The benchmark measures one GPU: any other --gpus value exits with a message before touching torch."""
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert r.returncode == 2 and "one GPU" in r.stderr and r.stdout.strip() == ""
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--workload", "nonsense"], capture_output=True,
                       text=True)
    assert r.returncode != 0


def test_legacy_layers_constructors_schedules_and_names():
    """mamtorch.nn.v1.FullyConnected, mamtorch.nn.v4.FullyConnected and mamtorch.MAMDense under their
    reference names (mamtorch/nn/__init__.py:1-6, mamtorch/__init__.py:7)."""
    assert mt.nn.v4.FullyConnected is mt.nn.FullyConnected
    layer = mt.nn.v1.FullyConnected(12, 6, vcon_steps=4, init_mode="normal")
    assert repr(layer) == "MAM@FullyConnected(in_features=12, out_features=6, bias=True, vcon_steps=4, vcon_type=linear)"
    assert layer.weight.shape == (6, 12) and bool((layer.bias == 0).all()) and layer.beta == 1.0
    for want in (0.75, 0.5, 0.25, 0):
        layer.vcon_step()
        assert layer.beta == want
    bound = float(np.float32((6 / (2 + 6)) ** 0.5))
    torch.manual_seed(0)
    uniform = mt.nn.v1.FullyConnected(50, 6)
    assert float(uniform.weight.abs().max()) <= bound and uniform.beta == 0.0
    with pytest.raises(Exception, match="not supported"):
        mt.nn.v1.FullyConnected(4, 4, vcon_steps=2, vcon_type="cubic").vcon_step()
    with pytest.raises(Exception, match="No argmax"):
        uniform.update_selection_count()
    dense = mt.MAMDense(10, 3, beta=True, beta_decay="descending-parabola", beta_epochs=4)
    assert dense.input_features == 10 and dense.state_size == 3 and dense.beta == 1.0
    dense.adjust_beta(2)
    assert dense.beta == 0.75
    dense.adjust_beta(4)
    assert dense.beta == 0
    asc = mt.MAMDense(10, 3, beta=True, beta_decay="ascending-parabola", beta_epochs=4)
    asc.adjust_beta(1)
    assert abs(asc.beta - 0.5625) < 1e-12


def test_resolve_row_offsets_at_a_weight_beyond_4_gib(tmp_path):
    """The 32-bit weight-row offsets of the index-resolving code (mamtorch_amd/csrc/mam_offsets.h), checked
    by a host-only C++ program at M = 262150, ldw = 4096, where (M - 1) * ldw * 4 wraps in 32 bits."""
    import subprocess

    exe = str(tmp_path / "offsets_host")
    subprocess.run(["g++", "-O1", "-std=c++17", os.path.join(ROOT, "tests", "offsets_host.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout[-2000:]


def test_static_forward_limit_is_checked_on_the_host():
    l = capi.lib()
    N, K, M = 224, 4096, 4224      # 3 ranges of K x 3 planes x N*M words = 34 MB of partials
    assert l.mam_fc_forward_workspace(N, K, M) > l.mam_fc_forward_static_limit() >= 24 * 2 ** 20
    one = ctypes.c_void_p(16)       # never dereferenced: the size check precedes every launch
    assert l.mam_fc_forward_static(one, K, one, K, capi.W_MK, None, one, one, one, None, None, N, K, M, None) == -2
    assert b"scratch" in l.mam_last_error()
    assert l.mam_set_option(99, 0) == -1
    # a value outside the option's range is refused and leaves the option as it was
    assert l.mam_set_option(capi.OPT_BACKWARD_ONE_LAUNCH, 3) == -1
    assert l.mam_set_option(capi.OPT_FORWARD_TILING, -1) == -1
    assert l.mam_set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_AUTO) == 0


def test_the_reference_import_name():
    import mamtorch
    import mamtorch.kernel.v4.fullyconnected_fast  # noqa: F401
    import mamtorch.nn.compat
    import mamtorch.nn.v1.fullyconnected
    import mamtorch.nn.v4.fullyconnected
    import mamtorch.sparse.kernel.v1.cusparsemm  # noqa: F401

    assert mamtorch.nn.FullyConnected is mt.nn.FullyConnected is mamtorch.nn.v4.fullyconnected.FullyConnected
    assert mamtorch.nn.v1.fullyconnected.FullyConnected is mt.nn.FullyConnectedV1
    assert mamtorch.MAMDense is mamtorch.nn.compat.MAMDense
    assert mamtorch.kernel.v4.fullyconnected is mt.kernel.v4.fullyconnected
