"""Operands staged in the workspace (csrc/mam_forward.hip, Staging): ragged K, unaligned rows and (K, M) weights run on
lengthened or transposed copies; values, indices and hand-over equal the C oracle's bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from helpers import assert_bits_equal, assert_index_equal

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("N,K,M", [(1, 15, 5), (2, 17, 129), (33, 63, 64), (31, 65, 130), (16, 1001, 127), (40, 4003, 33), (70, 33, 300)])
@pytest.mark.parametrize("layout_mk", [True, False])
@pytest.mark.parametrize("pad", [0, 5])
def test_ragged_rows(N, K, M, layout_mk, pad):
    from mamtorch_amd import capi

    g = torch.Generator().manual_seed(N + K)
    x, w, bias = torch.randn(N, K, generator=g), torch.randn(M, K, generator=g), torch.randn(M, generator=g)
    x[0] = -x[0].abs()                       # all products of this row share a sign: the last element is an extreme
    w[0] = w[0].abs()
    x[0, -1], w[0, -1] = -1e-3, 1e-3
    layout = capi.W_MK if layout_mk else capi.W_KM
    xs = torch.full((N, K + pad), float("nan"), device=DEV)
    xs[:, :K] = x.to(DEV)
    wl = w if layout_mk else w.T.contiguous()
    ws = torch.full((wl.size(0), wl.size(1) + pad), float("nan"), device=DEV)
    ws[:, :wl.size(1)] = wl.to(DEV)
    xd, wd = xs[:, :K], ws[:, :wl.size(1)]
    w_sel, x_sel = torch.zeros(2, N, M, device=DEV), torch.zeros(2, N, M, device=DEV)
    c, amax, amin = capi.fc_forward(xd, wd, layout, bias.to(DEV), w_sel=w_sel, x_sel=x_sel)
    values = capi.fc_forward_values(xd, wd, layout, bias.to(DEV))
    want = oracle.forward(x.numpy(), w.numpy(), oracle.W_MK, bias.numpy())
    tag = "N %d K %d M %d" % (N, K, M)
    assert_bits_equal(c.cpu().numpy(), want[0], tag + " c")
    assert_bits_equal(values.cpu().numpy(), want[0], tag + " values-only c")
    rows, cols = np.arange(N)[:, None], np.arange(M)[None, :]
    for plane, (got, index) in enumerate(zip((amax, amin), want[1:3])):
        assert_index_equal(got.cpu().numpy(), index, tag + " index")
        assert_bits_equal(x_sel[plane].cpu().numpy(), x.numpy()[rows, index], tag + " x_sel")
        assert_bits_equal(w_sel[plane].cpu().numpy(), w.numpy()[cols, index], tag + " w_sel")


@pytest.mark.parametrize("N,K,M", [(33, 64, 1), (5, 80, 63), (64, 288, 64), (31, 272, 65), (70, 2048, 129), (40, 4096, 192),
                                   (65, 528, 257), (33, 64, 320), (200, 2064, 64)])
def test_tiles_of_64_neurons(N, K, M):
    """Aligned (M, K) weights around odd multiples of 64 neurons: one, two and four k tiles, a partial last one, split and
    unsplit K."""
    from mamtorch_amd import capi

    g = torch.Generator().manual_seed(N + K + M)
    x, w, bias = torch.randn(N, K, generator=g), torch.randn(M, K, generator=g), torch.randn(M, generator=g)
    xd, wd = x.to(DEV), w.to(DEV)
    w_sel, x_sel = torch.zeros(2, N, M, device=DEV), torch.zeros(2, N, M, device=DEV)
    c, amax, amin = capi.fc_forward(xd, wd, capi.W_MK, bias.to(DEV), w_sel=w_sel, x_sel=x_sel)
    values = capi.fc_forward_values(xd, wd, capi.W_MK, bias.to(DEV))
    want = oracle.forward(x.numpy(), w.numpy(), oracle.W_MK, bias.numpy())
    tag = "N %d K %d M %d" % (N, K, M)
    assert_bits_equal(c.cpu().numpy(), want[0], tag + " c")
    assert_bits_equal(values.cpu().numpy(), want[0], tag + " values-only c")
    rows, cols = np.arange(N)[:, None], np.arange(M)[None, :]
    for plane, (got, index) in enumerate(zip((amax, amin), want[1:3])):
        assert_index_equal(got.cpu().numpy(), index, tag + " index")
        assert_bits_equal(x_sel[plane].cpu().numpy(), x.numpy()[rows, index], tag + " x_sel")
        assert_bits_equal(w_sel[plane].cpu().numpy(), w.numpy()[cols, index], tag + " w_sel")


def _planted(N, K, M, seed):
    """Ties across the whole row and at its end, zeros of both signs, rows without a product."""
    g = torch.Generator().manual_seed(seed)
    x, w = torch.randn(N, K, generator=g), torch.randn(M, K, generator=g)
    x[0] = -x[0].abs()                               # one sign throughout, the extreme at the last element
    w[0] = w[0].abs()
    x[0, -1], w[0, -1] = -1e-3, 1e-3
    x[1], x[2] = torch.randint(-2, 3, (K,), generator=g).float(), 0.25
    w[1:3] = torch.randint(-2, 3, (2, K), generator=g).float()
    x[3, : K - 20], x[4, K - 70:] = -0.0, float("nan")
    w[3], w[4, K - 64:] = 0.5, 7.0
    return x, w


def _runs_as(x, w, with_indices, route, range_len=None):
    """The route that the call is described by, which the workspace that it brings has room for."""
    from mamtorch_amd import capi

    l = capi.lib()
    (N, K), M = x.shape, w.shape[0]
    call = (capi._p(x), capi._ld(x), capi._p(w), capi._ld(w), capi.W_MK, N, K, M)
    if range_len is None:
        text = capi.fc_forward_describe(x, w, capi.W_MK, with_indices)
        room = l.mam_fc_forward_workspace_at(*call, int(with_indices))
    else:
        text = capi.fc_forward_ranges_describe(x, w, range_len, capi.W_MK, with_indices)
        room = l.mam_fc_forward_ranges_workspace_at(*call, range_len, int(with_indices))
    first = text.split("; with less: ")[0]
    assert route in first, text
    if first.startswith("with "):
        assert room >= int(first.split()[1]), text


# operand rows: aligned, 16 bytes apart but begun off them, of odd stride
@pytest.mark.parametrize("pad,shift", [(0, 0), (4, 1), (3, 2)])
@pytest.mark.parametrize("N,K,M", [(33, 128, 64), (37, 129, 130), (33, 191, 70), (64, 192, 129), (200, 260, 300), (31, 1300, 42), (40, 2050, 192),
                                   (5, 4092, 65)])
def test_last_tile_at_the_end_of_the_row(N, K, M, pad, shift):
    """Rows of any length and alignment without a copy of x: all of K in one range and in several, tails of one to 63 columns."""
    from mamtorch_amd import capi

    x, w = _planted(N, K, M, N + K)
    bias = torch.randn(M, generator=torch.Generator().manual_seed(1))

    def padded(t):      # infinities all round: a column too many would win
        buf = torch.full((t.size(0) * (K + pad) + 8,), float("inf"), device=DEV)
        view = buf[shift: shift + t.size(0) * (K + pad)].view(t.size(0), K + pad)[:, :K]
        view.copy_(t)
        return view

    want = oracle.forward(x.numpy(), w.numpy(), oracle.W_MK, bias.numpy())
    for xd, wd in ((padded(x), w.to(DEV)), (padded(x), padded(w)), (x.to(DEV), padded(w))):
        w_sel, x_sel = torch.zeros(2, N, M, device=DEV), torch.zeros(2, N, M, device=DEV)
        _runs_as(xd, wd, True, "last k tile at the end of K" if K % 16 or pad or shift else "mam_fwd_sx_kernel")
        _runs_as(xd, wd, False, "last k tile at the end of K" if K % 16 or pad or shift else "mam_fwd_sx_kernel")
        c, amax, amin = capi.fc_forward(xd, wd, capi.W_MK, bias.to(DEV), w_sel=w_sel, x_sel=x_sel)
        values = capi.fc_forward_values(xd, wd, capi.W_MK, bias.to(DEV))
        tag = "N %d K %d M %d" % (N, K, M)
        assert_bits_equal(c.cpu().numpy(), want[0], tag + " c")
        assert_bits_equal(values.cpu().numpy(), want[0], tag + " values-only c")
        rows, cols = np.arange(N)[:, None], np.arange(M)[None, :]
        for plane, (got, index) in enumerate(zip((amax, amin), want[1:3])):
            assert_index_equal(got.cpu().numpy(), index, tag + " index")
            assert_bits_equal(x_sel[plane].cpu().numpy(), x.numpy()[rows, index], tag + " x_sel")
            assert_bits_equal(w_sel[plane].cpu().numpy(), w.numpy()[cols, index], tag + " w_sel")


@pytest.mark.parametrize("pad", [0, 3])
@pytest.mark.parametrize("N,K,M,range_len", [(33, 128, 70, 64), (33, 130, 70, 65), (40, 264, 129, 100), (5, 448, 65, 128), (70, 1000, 300, 250),
                                             (64, 1001, 64, 333), (130, 999, 64, 201)])
def test_last_tile_at_the_end_of_each_range(N, K, M, range_len, pad):
    from mamtorch_amd import capi

    x, w = _planted(N, K, M, N + K)
    xd = torch.full((N, K + pad), float("inf"), device=DEV)[:, :K].copy_(x)
    wd = torch.full((M, K + pad), float("inf"), device=DEV)[:, :K].copy_(w)
    route = "mam_fwd_sx_kernel" if (K % 16 == 0 and range_len % 64 == 0 and pad == 0) else "last k tile at the end of K"
    if K - K // range_len * range_len in range(1, 64):
        route = "lengthen_rows_kernel"      # a last range too short for a tile of its own
    for with_indices in (True, False):
        _runs_as(xd, wd, with_indices, route, range_len)
    c, amax, amin = capi.fc_forward_ranges(xd, wd, range_len, capi.W_MK)
    values, _, _ = capi.fc_forward_ranges(xd, wd, range_len, capi.W_MK, with_indices=False)
    total = None
    for s, k in enumerate(range(0, K, range_len)):
        part = oracle.forward(x[:, k:k + range_len].contiguous().numpy(), w[:, k:k + range_len].contiguous().numpy(), oracle.W_MK)
        total = part[0] if total is None else total + part[0]
        tag = "N %d K %d M %d range %d" % (N, K, M, s)
        assert_index_equal(amax[s].cpu().numpy(), part[1] + k, tag + " argmax")
        assert_index_equal(amin[s].cpu().numpy(), part[2] + k, tag + " argmin")
    assert_bits_equal(c.cpu().numpy(), total, tag + " c")
    assert_bits_equal(values.cpu().numpy(), total, tag + " values")


# x of 16 MiB and more, few neurons: a part of the last row tile, whole tiles, a partial last one, one that ends with the row
@pytest.mark.parametrize("N,K,M", [(16390, 256, 33), (8193, 528, 70), (4101, 1027, 200), (2053, 2048, 65), (1033, 4093, 129)])
def test_rows_fetched_ahead(N, K, M):
    from mamtorch_amd import capi

    x, w = _planted(N, K, M, N + K)
    xd, wd = x.to(DEV), w.to(DEV)
    for with_indices in (True, False):
        _runs_as(xd, wd, with_indices, "x fetched ahead")
    c, amax, amin = capi.fc_forward(xd, wd, capi.W_MK)
    values = capi.fc_forward_values(xd, wd, capi.W_MK)
    want = oracle.forward(x.numpy(), w.numpy(), oracle.W_MK, None)
    tag = "N %d K %d M %d" % (N, K, M)
    assert_bits_equal(c.cpu().numpy(), want[0], tag + " c")
    assert_bits_equal(values.cpu().numpy(), want[0], tag + " values-only c")
    assert_index_equal(amax.cpu().numpy(), want[1], tag + " argmax")
    assert_index_equal(amin.cpu().numpy(), want[2], tag + " argmin")


@pytest.mark.parametrize("N,K,M", [(65600, 80, 33), (65535, 64, 65), (40, 130, 65600)])
def test_a_transposed_weight_of_any_number_of_rows(N, K, M):
    """More rows together than one launch of lengthen_rows holds, against the tiling that takes a (K, M) weight as it is."""
    from mamtorch_amd import capi

    g = torch.Generator(device=DEV).manual_seed(N)
    x, w = torch.randint(-9, 10, (N, K), generator=g, device=DEV).float(), torch.randn(K, M, generator=g, device=DEV)
    assert "transpose_kernel + mam_fwd_sx_kernel" in capi.fc_forward_describe(x, w, capi.W_KM)
    outs = []
    for tiling in (capi.FORWARD_TILING_AUTO, capi.FORWARD_TILING_WIDE):
        capi.set_option(capi.OPT_FORWARD_TILING, tiling)
        try:
            outs.append(capi.fc_forward(x, w, capi.W_KM) + (capi.fc_forward_values(x, w, capi.W_KM),))
        finally:
            capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_AUTO)
    for got, want in zip(*outs):
        assert torch.equal(got, want)
