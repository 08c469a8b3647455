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
