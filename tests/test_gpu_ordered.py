"""The forward over magnitude-ordered lists (csrc/mam_ordered.hip) against the C oracle, bit for bit: sizes on both
sides of every tile width, list operands on either side, and data that the lists do not finish (ties, zeros,
NaN / infinities, one sign, sparse rows, denormal and overflowing products)."""
import numpy as np
import pytest
import torch

import oracle
from helpers import assert_bits_equal, assert_index_equal

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _data(kind, rows, k, g):
    t = torch.randn(rows, k, generator=g)
    r = torch.rand(rows, k, generator=g)
    if kind == "uniform":
        t = r * 2 - 1
    elif kind == "relu":
        t = t.relu()
    elif kind == "ties":
        t = (t * 4).round() / 4
    elif kind == "levels":                  # as the lists like it, and many equal products
        t = (t * 8).round() / 8
    elif kind == "bounded levels":
        t = ((r * 2 - 1) * 8).round() / 8
    elif kind == "positive":
        t = r + 0.1
    elif kind == "zero rows":
        t[torch.rand(rows, generator=g) < 0.3] = 0
        t[0] = -0.0
    elif kind == "nan and inf":
        t[r < 1e-3] = float("nan")
        t[(r > 0.5) & (r < 0.501)] = float("inf")
        t[(r > 0.6) & (r < 0.601)] = -float("inf")
        t[(r > 0.7) & (r < 0.8)] = -0.0
    elif kind == "sparse":
        t[r < 0.97] = 0
    elif kind == "denormal":
        t = t * 1e-24
    elif kind == "overflow":
        t = t * 1e25
    return t


def _check(N, K, M, kind_x, kind_w, layout_mk=True, pad=0, seed=0):
    from mamtorch_amd import capi

    g = torch.Generator().manual_seed(seed)
    x = _data(kind_x, N, K + pad, g)[:, :K]
    w = _data(kind_w, M, K, g)
    bias = torch.randn(M, generator=g)
    want = oracle.forward(x.contiguous().numpy(), w.numpy(), oracle.W_MK, bias.numpy())
    xd = _strided(x, pad)
    wd = (w if layout_mk else w.T.contiguous()).to(DEV)
    layout = capi.W_MK if layout_mk else capi.W_KM
    w_sel, x_sel = torch.zeros(2, N, M, device=DEV), torch.zeros(2, N, M, device=DEV)
    (c, amax, amin), decision = _by_lists(xd, wd, layout, bias.to(DEV), w_sel=w_sel, x_sel=x_sel)
    (values,), _ = _by_lists(xd, wd, layout, bias.to(DEV), indices=False)
    tag = "%s x %s, N %d K %d M %d" % (kind_x, kind_w, N, K, M)
    assert_bits_equal(c.cpu().numpy(), want[0], tag + " c")
    assert_bits_equal(values.cpu().numpy(), want[0], tag + " values-only c")
    assert_index_equal(amax.cpu().numpy(), want[1], tag + " argmax")
    assert_index_equal(amin.cpu().numpy(), want[2], tag + " argmin")
    rows, cols = np.arange(N)[:, None], np.arange(M)[None, :]
    for plane, index in enumerate(want[1:3]):
        assert_bits_equal(x_sel[plane].cpu().numpy(), x.numpy()[rows, index], tag + " x_sel")
        assert_bits_equal(w_sel[plane].cpu().numpy(), w.numpy()[cols, index], tag + " w_sel")
    return decision


def _by_lists(xd, wd, layout, bias=None, indices=True, w_sel=None, x_sel=None, tiling="LISTS"):
    """A call with the lists allowed at every size (or as ``tiling`` says): its outputs, and what the device decided -- (side, leading entries, entries
    per list), side 0: the dense kernels, 1: rows of x are searched, 2: rows of w -- which lies at the start of the workspace."""
    from mamtorch_amd import capi

    N, K = xd.shape
    M = wd.shape[0] if layout == capi.W_MK else wd.shape[1]
    capi.set_option(capi.OPT_FORWARD_TILING, getattr(capi, "FORWARD_TILING_" + tiling))
    try:
        need = capi.lib().mam_fc_forward_workspace_for(N, K, M, layout, int(indices))
        ws = torch.full((need,), 255, dtype=torch.uint8, device=DEV)
        if indices:
            out = capi.fc_forward(xd, wd, layout, bias, workspace=ws, w_sel=w_sel, x_sel=x_sel)
        else:
            out = (capi.fc_forward_values(xd, wd, layout, bias, workspace=ws),)
        torch.cuda.synchronize()
    finally:
        capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_AUTO)
    return out, ws[:12].view(torch.int32).tolist()


def _strided(x, pad):
    N, K = x.shape
    out = torch.zeros(N, K + pad, device=DEV)[:, :K]
    out.copy_(x.to(DEV))
    return out


@pytest.mark.parametrize("N,K,M", [
    (64, 1216, 70), (65, 1217, 33), (64, 2432, 34), (33, 2433, 64), (130, 4864, 40), (40, 4865, 36), (34, 9728, 33),
    (33, 9729, 32), (5, 200, 7), (1, 130, 300), (300, 131, 1), (257, 96, 129), (520, 768, 96)])
@pytest.mark.parametrize("kinds", [("normal", "uniform"), ("uniform", "normal"), ("normal", "normal")])
@pytest.mark.parametrize("layout_mk", [True, False])
def test_sizes_on_both_sides_of_every_tile_width(N, K, M, kinds, layout_mk):
    side, lead, _ = _check(N, K, M, *kinds, layout_mk=layout_mk, pad=3 if layout_mk else 0)
    if 768 <= K <= 9728 and "uniform" in kinds:
        # the rows of the normal operand are searched; a (K, M) weight's are not listed
        assert (side, lead) == ((1 if kinds[0] == "normal" else 2 if layout_mk else 0), 0)


@pytest.mark.parametrize("N, K, M", [(8, 800, 32), (9, 800, 33), (65, 900, 97), (33, 2000, 41), (32, 3000, 9), (129, 3000, 66),
                                     (64, 5000, 6)])       # 32, 16, 8, 4 tile rows; blocks of one row to all
@pytest.mark.parametrize("kinds", [("levels", "bounded levels"), ("bounded levels", "levels"), ("levels", "levels")])
def test_equal_products_met_by_different_lanes(N, K, M, kinds):
    """A wave's last outputs are finished by lanes of their own: the first index wins wherever an equal product was met."""
    _check(N, K, M, *kinds, seed=N)


@pytest.mark.parametrize("K", [800, 3000, 5000])                      # 32, 8 and 4 tile rows
@pytest.mark.parametrize("M", [32, 48, 64, 96, 100, 101, 112])
@pytest.mark.parametrize("kinds", [("normal", "uniform"), ("uniform", "normal")])
def test_outputs_that_are_lines_and_parts_of_lines(K, M, kinds):
    _check(70, K, M, *kinds, seed=M)


@pytest.mark.parametrize("kind", ["ties", "positive", "zero rows", "nan and inf", "sparse", "denormal", "overflow"])
@pytest.mark.parametrize("other", ["uniform", "normal", "same"])
def test_data_the_lists_do_not_finish(kind, other):
    """With the lists allowed: most of these the device hands to the dense kernels, which are behind the same guard."""
    for K in (300, 2500):
        _check(70, K, 68, kind, kind if other == "same" else other, seed=1)
        _check(70, K, 68, kind if other == "same" else other, kind, seed=2)


def test_a_few_bad_rows_among_good_ones():
    """Rows of zeros, of NaN and of constants inside an otherwise ordinary batch: most of the call goes by lists."""
    from mamtorch_amd import capi

    g = torch.Generator().manual_seed(5)
    N, K, M = 640, 768, 96
    x, w = torch.randn(N, K, generator=g), torch.rand(M, K, generator=g) * 2 - 1
    x[7] = 0.0
    x[100, 3] = float("nan")
    x[200] = 1.5
    x[300, 5] = float("inf")
    x[400].abs_()
    w[11] = 0.0
    w[12] = -0.25
    w[13, 700] = float("nan")
    want = oracle.forward(x.numpy(), w.numpy(), oracle.W_MK)
    capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_LISTS)
    try:
        c, amax, amin = capi.fc_forward(x.to(DEV), w.to(DEV), capi.W_MK)
        values = capi.fc_forward_values(x.to(DEV), w.to(DEV), capi.W_MK)
    finally:
        capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_AUTO)
    assert_bits_equal(c.cpu().numpy(), want[0], "c")
    assert_bits_equal(values.cpu().numpy(), want[0], "values-only c")
    assert_index_equal(amax.cpu().numpy(), want[1], "argmax")
    assert_index_equal(amin.cpu().numpy(), want[2], "argmin")


@pytest.mark.parametrize("N, K", [(2047, 640), (2048, 700), (2049, 1023), (2051, 1024), (2050, 1025)])
@pytest.mark.parametrize("listed", ["x", "w"])
def test_lists_of_many_short_rows(N, K, listed):
    """A wave per row from 2048 rows on, up to K = 1024; among the rows some of zeros, of one magnitude, with a NaN or an infinity, and
    of fewer entries than a list holds, the last row too."""
    from mamtorch_amd import capi

    g = torch.Generator().manual_seed(N)
    many = torch.randn(N, K, generator=g)
    many[3], many[4], many[9, 17], many[10, K - 1], many[N - 1, 5:] = 0.0, 0.5, float("nan"), float("inf"), 0.0
    few = torch.rand(40, K, generator=g) * 2 - 1
    x, w = (many, few) if listed == "x" else (few, many)
    want = oracle.forward(x.numpy(), w.numpy(), oracle.W_MK)
    (c, amax, amin), (side, lead, _) = _by_lists(x.to(DEV), w.to(DEV), capi.W_MK)
    assert (side, lead) == (1 if listed == "x" else 2, 0)
    assert_bits_equal(c.cpu().numpy(), want[0], "c")
    assert_index_equal(amax.cpu().numpy(), want[1], "argmax")
    assert_index_equal(amin.cpu().numpy(), want[2], "argmin")


@pytest.mark.parametrize("N, K, M", [(640, 768, 640), (700, 1024, 701), (1000, 2432, 300), (300, 2432, 1000), (512, 4864, 513),
                                     (400, 4095, 402), (1200, 520, 333), (333, 520, 1201)])
@pytest.mark.parametrize("kinds", [("normal", "normal"), ("relu", "normal")])
def test_two_sided_searches(N, K, M, kinds):
    """Normal weights: the leading entries of one operand first, then a search bounded by what they leave."""
    side, lead, _ = _check(N, K, M, *kinds, seed=3)
    assert lead > 0 and side == (2 if N > 2 * M and (kinds[0] == "normal" or K > 1000) else 1)


@pytest.mark.parametrize("N, K, M", [(640, 768, 640), (300, 2432, 1000), (1000, 2432, 300), (400, 4095, 402)])
def test_two_sided_searches_over_special_rows(N, K, M):
    """Rows of zeros, of one magnitude, of few entries, ties, NaN and infinities on either operand of a two-sided search."""
    from mamtorch_amd import capi

    g = torch.Generator().manual_seed(K + N)
    x, w = torch.randn(N, K, generator=g), torch.randn(M, K, generator=g)
    for t, free in zip((x, w), _unsampled(N, M)):
        t[free[0]] = 0.0
        t[free[5]] = -0.75
        t[free[6]] = torch.randint(0, 2, (K,), generator=g).float() * 2 - 1
        t[free[10], 4:] = 0.0
        t[free[20]] = (t[free[20]] * 2).round() / 2
        t[free[30], K // 2] = float("nan")
        t[free[31], K - 1] = float("inf")
        t[free[32], 0] = -float("inf")
        t[free[-1]].abs_()
    bias = torch.randn(M, generator=g)
    want = oracle.forward(x.numpy(), w.numpy(), oracle.W_MK, bias.numpy())
    sel = torch.zeros(4, N, M, device=DEV)
    out, d = _by_lists(x.to(DEV), w.to(DEV), capi.W_MK, bias.to(DEV), w_sel=sel[:2], x_sel=sel[2:])
    values, dv = _by_lists(x.to(DEV), w.to(DEV), capi.W_MK, bias.to(DEV), indices=False)
    assert d == dv and d[0] != 0 and d[1] > 0
    assert_bits_equal(out[0].cpu().numpy(), want[0], "c")
    assert_bits_equal(values[0].cpu().numpy(), want[0], "values-only c")
    for plane in range(2):
        assert_index_equal(out[1 + plane].cpu().numpy(), want[1 + plane], "index")
        index = want[1 + plane]
        assert_bits_equal(sel[plane].cpu().numpy(), w.numpy()[np.arange(M)[None, :], index], "w_sel")
        assert_bits_equal(sel[2 + plane].cpu().numpy(), x.numpy()[np.arange(N)[:, None], index], "x_sel")


@pytest.mark.parametrize("N, K, M", [(256, 4096, 4096), (12608, 768, 3072), (12608, 3072, 768), (16384, 4096, 1024)])
@pytest.mark.parametrize("kinds", [("normal", "uniform"), ("uniform", "normal"), ("normal", "normal")])
def test_lists_and_dense_tilings_agree_on_full_size_calls(N, K, M, kinds):
    """The layers that training and inference run: every output of both routes, bit for bit."""
    from mamtorch_amd import capi

    g = torch.Generator(device=DEV).manual_seed(12)
    make = {"normal": lambda r: torch.randn(r, K, generator=g, device=DEV),
            "uniform": lambda r: torch.rand(r, K, generator=g, device=DEV) * 2 - 1}
    x, w, bias = make[kinds[0]](N), make[kinds[1]](M) * 0.02, torch.randn(M, generator=g, device=DEV)
    got = {}
    for tiling in ("LISTS", "DENSE"):
        sel = torch.zeros(4, N, M, device=DEV)
        out, d = _by_lists(x, w, capi.W_MK, bias, w_sel=sel[:2], x_sel=sel[2:], tiling=tiling)
        values, _ = _by_lists(x, w, capi.W_MK, bias, indices=False, tiling=tiling)
        got[tiling] = (*out, sel, *values)
        if tiling == "LISTS":
            assert d[0] != 0 and (d[1] > 0) == (kinds == ("normal", "normal"))
    for one, other in zip(got["LISTS"], got["DENSE"]):
        assert torch.equal(one.view(torch.int32), other.view(torch.int32))
    if N == 256:
        want = oracle.forward(x.cpu().numpy(), w.cpu().numpy(), oracle.W_MK, bias.cpu().numpy())
        assert_bits_equal(got["DENSE"][0].cpu().numpy(), want[0], "c")
        assert_index_equal(got["DENSE"][1].cpu().numpy(), want[1], "argmax")
        assert_index_equal(got["DENSE"][2].cpu().numpy(), want[2], "argmin")


def test_every_replay_of_a_graph_decides_anew():
    """A captured call on data that suits the lists, then data that does not (dense kernels), then lists again."""
    from mamtorch_amd import capi

    N, K, M = 66, 520, 70
    g = torch.Generator().manual_seed(6)
    x, w = torch.zeros(N, K, device=DEV), torch.zeros(M, K, device=DEV)
    capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_LISTS)
    try:
        capi.fc_forward(x, w, capi.W_MK)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = capi.fc_forward(x, w, capi.W_MK)
    finally:
        capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_AUTO)
    for kinds in [("uniform", "uniform"), ("positive", "positive"), ("normal", "normal"), ("ties", "positive")]:
        xs, ws = _data(kinds[0], N, K, g), _data(kinds[1], M, K, g)
        x.copy_(xs)
        w.copy_(ws)
        graph.replay()
        torch.cuda.synchronize()
        want = oracle.forward(xs.numpy(), ws.numpy(), oracle.W_MK)
        assert_bits_equal(out[0].cpu().numpy(), want[0], "%s x %s c" % kinds)
        assert_index_equal(out[1].cpu().numpy(), want[1], "%s x %s argmax" % kinds)
        assert_index_equal(out[2].cpu().numpy(), want[2], "%s x %s argmin" % kinds)


@pytest.mark.parametrize("side", ["normal", "uniform"])      # of x: its rows are searched, the rows of w are searched
@pytest.mark.parametrize("keep", ["w_sel", "x_sel"])
def test_either_hand_over_array_alone(side, keep):
    from mamtorch_amd import capi

    g = torch.Generator().manual_seed(7)
    N, K, M = 640, 768, 616
    x, w = _data(side, N, K, g), _data("uniform" if side == "normal" else "normal", M, K, g)
    want = oracle.forward(x.numpy(), w.numpy(), oracle.W_MK)
    sel = torch.full((2, N, M), float("nan"), device=DEV)
    capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_LISTS)
    try:
        c, amax, amin = capi.fc_forward(x.to(DEV), w.to(DEV), capi.W_MK, **{keep: sel})
        torch.cuda.synchronize()
    finally:
        capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_AUTO)
    assert_bits_equal(c.cpu().numpy(), want[0], "c")
    assert_index_equal(amax.cpu().numpy(), want[1], "argmax")
    assert_index_equal(amin.cpu().numpy(), want[2], "argmin")
    for plane, index in enumerate(want[1:3]):
        operand, rows = (x, np.arange(N)[:, None]) if keep == "x_sel" else (w, np.arange(M)[None, :])
        assert_bits_equal(sel[plane].cpu().numpy(), operand.numpy()[rows, index], keep)


@pytest.mark.parametrize("indices", [True, False])
@pytest.mark.parametrize("pad, offset", [(3, 0), (4, 1)])
def test_rows_that_are_not_aligned_go_by_lists(indices, pad, offset):
    """The copies that the dense tiling would make of such operands do not take the lists' room."""
    from mamtorch_amd import capi

    g = torch.Generator().manual_seed(8)
    N, K, M = 640, 768, 616
    x, w = torch.randn(N, K + pad, generator=g), torch.rand(M, K, generator=g) * 2 - 1
    want = oracle.forward(x[:, offset:offset + K].contiguous().numpy(), w.numpy(), oracle.W_MK)
    out, (side, lead, _) = _by_lists(x.to(DEV)[:, offset:offset + K], w.to(DEV), capi.W_MK, indices=indices)
    assert (side, lead) == (1, 0)
    assert_bits_equal(out[0].cpu().numpy(), want[0], "c")
    for got, expected in zip(out[1:], want[1:]):
        assert_index_equal(got.cpu().numpy(), expected, "index")


def _unsampled(N, M):
    """Rows of x and of w that no sampled output of the device's decision belongs to."""
    x_rows = {(2 * i + 1) * N // 128 for i in range(64)}
    w_rows = {((i * 2654435769 & 0xffffffff) * M) >> 32 for i in range(64)}
    return [r for r in range(N) if r not in x_rows], [r for r in range(M) if r not in w_rows]


@pytest.mark.parametrize("N, K, M", [(640, 768, 300), (330, 1300, 202), (330, 2500, 202), (323, 4900, 101)])     # 32, 16, 8, 4 tile rows
@pytest.mark.parametrize("searched", ["x", "w"])
@pytest.mark.parametrize("indices", [True, False])
def test_rows_that_no_list_finishes(N, K, M, searched, indices):
    """Rows of one magnitude, of one sign, of few entries, NaN and infinities on the searched side and on the other one, next to each
    other and alone, at the ends too, inside a call that goes by lists."""
    from mamtorch_amd import capi

    g = torch.Generator().manual_seed(K)
    if searched == "w":
        N, M = M, N
    x, w = torch.randn(N, K, generator=g), torch.rand(M, K, generator=g) * 2 - 1
    if searched == "w":
        x, w = torch.rand(N, K, generator=g) * 2 - 1, torch.randn(M, K, generator=g)
    a, b = (x, w) if searched == "x" else (w, x)
    free_a, free_b = _unsampled(N, M) if searched == "x" else _unsampled(N, M)[::-1]
    ones = torch.randint(0, 2, (4, K), generator=g).float() * 2 - 1
    near = next(r for r in free_a[10:] if r + 1 in free_a and r + 2 in free_a)
    a[free_a[0]] = ones[0]
    a[near:near + 3] = ones[1:]
    a[free_a[40], 5:] = 0.0
    a[free_a[41]].abs_()
    a[free_a[-1]] = -0.5
    b[free_b[0]] = 0.25 * ones[0]
    b[free_b[20]].abs_()
    b[free_b[21], 1:] = 0.0
    b[free_b[22], K - 1] = float("nan")
    b[free_b[-1], 2] = -float("inf")
    bias = torch.randn(M, generator=g)
    want = oracle.forward(x.numpy(), w.numpy(), oracle.W_MK, bias.numpy())
    out, (side, lead, _) = _by_lists(x.to(DEV), w.to(DEV), capi.W_MK, bias.to(DEV), indices)
    assert (side, lead) == (1 if searched == "x" else 2, 0)
    assert_bits_equal(out[0].cpu().numpy(), want[0], "c")
    for got, expected in zip(out[1:], want[1:]):
        assert_index_equal(got.cpu().numpy(), expected, "index")


@pytest.mark.parametrize("scattered", [True, False])
def test_rows_that_no_list_finishes_do_not_hold_up_the_call(scattered):
    """4 % of the rows of x all +-1, which the lists take (0.55 and 0.50 of the dense tilings' time): within 0.9 of it.  One output
    of such a row at a time took 1.1 and 3.6 times the dense tilings' time."""
    from mamtorch_amd import capi

    g = torch.Generator(device=DEV).manual_seed(9)
    N, K, M = 16384, 4096, 1024
    x, w = torch.randn(N, K, generator=g, device=DEV), torch.rand(M, K, generator=g, device=DEV) * 2 - 1
    rows = torch.randperm(N, generator=g, device=DEV)[:N // 25] if scattered else torch.arange(N // 25, device=DEV)
    x[rows] = torch.randint(0, 2, (N // 25, K), generator=g, device=DEV).float() * 2 - 1
    times = {}
    for tiling in ("DENSE", "AUTO"):
        capi.set_option(capi.OPT_FORWARD_TILING, getattr(capi, "FORWARD_TILING_" + tiling))
        try:
            for _ in range(3):
                out = capi.fc_forward(x, w, capi.W_MK)
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(5):
                out = capi.fc_forward(x, w, capi.W_MK)
            end.record()
            end.synchronize()
        finally:
            capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_AUTO)
        times[tiling] = (start.elapsed_time(end), out)
    assert times["AUTO"][0] < 0.9 * times["DENSE"][0], (times["AUTO"][0], times["DENSE"][0])
    for got, dense in zip(times["AUTO"][1], times["DENSE"][1]):
        assert torch.equal(got, dense)


@pytest.mark.parametrize("indices", [True, False])
def test_a_call_without_room_for_its_lists_still_runs(indices):
    """A device with too little memory left for the lists: the operator asks for what the dense tilings need instead."""
    import mamtorch_amd as mt

    g = torch.Generator(device=DEV).manual_seed(10)
    N, K, M = 8192, 4096, 1024
    x, w = torch.randn(N, K, generator=g, device=DEV), torch.rand(M, K, generator=g, device=DEV) * 2 - 1
    forward = (lambda: mt.kernel.v4.fullyconnected_wt(x, w)) if indices else (
        lambda: [mt.kernel.v4.fullyconnected_fast_wt(x, w)])
    want = forward()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    from mamtorch_amd import capi
    least = 3 * N * M * 4
    assert capi.lib().mam_fc_forward_workspace_for(N, K, M, capi.W_MK, int(indices)) > least + (64 << 20)
    total = torch.cuda.get_device_properties(DEV).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(DEV) + least + (48 << 20)) / total, DEV)
    try:
        got = forward()
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, DEV)
    for one, other in zip(got, want):
        assert torch.equal(one, other)


@pytest.mark.parametrize("N, K, M", [(64, 4096, 16384), (16384, 4096, 64), (40, 8000, 16384), (64, 4096, 32768)])
@pytest.mark.parametrize("indices", [True, False])
def test_calls_of_few_rows_go_by_lists_only_where_the_search_is_short(N, K, M, indices):
    """Too few rows for the waves of a workgroup: the dense tilings, unless one side is uniform; the results are the same."""
    from mamtorch_amd import capi

    g = torch.Generator(device=DEV).manual_seed(11)
    x, w = torch.randn(N, K, generator=g, device=DEV), torch.randn(M, K, generator=g, device=DEV)
    for uniform in (False, True):
        if uniform:
            x = torch.rand(N, K, generator=g, device=DEV) * 2 - 1
        out, (side, _, _) = _by_lists(x, w, capi.W_MK, indices=indices, tiling="AUTO")
        assert (side != 0) == uniform, side
        capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_DENSE)
        try:
            dense = capi.fc_forward(x, w, capi.W_MK) if indices else (capi.fc_forward_values(x, w, capi.W_MK),)
        finally:
            capi.set_option(capi.OPT_FORWARD_TILING, capi.FORWARD_TILING_AUTO)
        for one, other in zip(out, dense):
            assert torch.equal(one, other)
