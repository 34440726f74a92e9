"""GPU parity of the Linear for 17-128 tokens (linear_mid.hip), and the cases of 9-16 beside
it (the 16-token MFMA decode).

Raw and tiled weights (the same bits: same products, same order) against the CPU oracle
(cpu_kernels.cpp:208-218), against the general paths that the tuning hook forces (the
16-token MFMA decode below 64 tokens, the bf16 GEMM from 64), and against themselves.
Shapes: token tiles and their remainders, single rows, ragged row groups, one block, an
odd number of blocks, phases of 1-4 blocks, 1 / 2 / 4 / 8 K splits.  Bars: 1e-5 (fp32
sums) below 64 tokens and 1e-6 against the decode (the same exact block products grouped
differently); 1e-2 from 64 tokens (both operands rounded once to bf16).
"""
import numpy as np
import pytest

from helpers import assert_bitexact, empty_f32, note, rel_l2, slower_by, to_dev, to_host
from llmengine_amd import capi
from llmengine_amd import synthetic as S

pytestmark = pytest.mark.gpu


def weight(seed, N, K):
    return S.q8_0_weight(seed, N, K)[0]


def tiled_dev(dw, N, K, dev):
    import torch
    t = torch.empty(capi.tiled_bytes(N, K), dtype=torch.uint8, device=dev)
    capi.tile(dw, t, N, K)
    return t


def tol(M):
    return 1e-5 if M < 64 else 1e-2


@pytest.mark.parametrize("M,N,K,bias", [
    (9, 100, 32, "f32"), (16, 65, 1024, None), (12, 300, 992, None),
    (17, 1, 96, "bf16"), (31, 63, 256, None), (32, 64, 288, "f32"), (33, 257, 512, "bf16"),
    (48, 129, 544, None), (49, 1000, 4096, "f32"), (63, 640, 4128, None),
    (63, 16384 + 5, 256, None), (40, 50000, 96, None),
    (64, 100, 32, "bf16"), (65, 513, 1056, None), (80, 300, 4160, "f32"), (81, 77, 288, None),
    (96, 4864, 224, "bf16"), (97, 1024, 2048, None), (128, 4096, 160, "f32"),
    (128, 96, 8192, None)])
def test_mid_linear(dev, orc, M, N, K, bias):
    import torch
    note(f"mid linear M={M} N={N} K={K} bias={bias}")
    raw = weight(900 + N % 97, N, K)
    x = S.activations(901 + M, (M, K))
    b32 = S.activations(902, (N,), tag=S.TAG_BIAS)
    b16 = (b32.view(np.uint32) >> 16).astype(np.uint16)
    if bias == "bf16":
        b32 = (b16.astype(np.uint32) << 16).view(np.float32)
    dx, dw = to_dev(x, dev), to_dev(raw, dev)
    dt = tiled_dev(dw, N, K, dev)
    db = {None: None, "f32": to_dev(b32, dev), "bf16": to_dev(b16.view(np.int16), dev)}[bias]
    y = [empty_f32((M, N), dev) for _ in range(4)]
    for out, w, tiled in ((y[0], dw, False), (y[1], dt, True), (y[2], dt, True)):
        if bias == "bf16":
            capi.linear_bias_bf16(dx, w, db, out, M, N, K, tiled=tiled)
        else:
            (capi.linear_tiled if tiled else capi.linear)(dx, w, db, out, M, N, K)
    general = to_dev(b32, dev) if bias else None
    capi.linear_ex(dx, dw, general, y[3], M, N, K, path=3 if M < 64 else 2)
    torch.cuda.synchronize()
    got = to_host(y[0])
    assert_bitexact(to_host(y[1]), got, "tiled vs raw")
    assert torch.equal(y[1], y[2])
    assert rel_l2(got, to_host(y[3])) <= (1e-6 if M < 64 else 1e-2)
    rows = np.unique(np.linspace(0, N - 1, min(N, 200)).astype(int))
    w_rows = np.ascontiguousarray(raw.reshape(N, -1)[rows]).reshape(-1)
    want = orc.linear(x, w_rows, b32[rows] if bias else None, M, rows.size, K)
    assert rel_l2(got[:, rows], want) <= tol(M)


@pytest.mark.parametrize("M,Ns,K", [(20, (70, 33, 1), 512), (63, (4096, 128, 128), 896),
                                    (13, (500, 20, 20), 736), (77, (1024, 40, 300), 2080)])
def test_mid_multi(dev, orc, M, Ns, K):
    """Segment boundaries inside a wave's row groups; below 64 tokens each output has the
    single Linear's bits."""
    note(f"mid multi M={M} Ns={Ns} K={K}")
    ws = [weight(910 + i, n, K) for i, n in enumerate(Ns)]
    bs = [S.activations(911, (Ns[0],), tag=S.TAG_BIAS), None,
          S.activations(912, (Ns[2],), tag=S.TAG_BIAS)]
    x = S.activations(913, (M, K))
    dx, dws = to_dev(x, dev), [to_dev(w, dev) for w in ws]
    dbs = [None if b is None else to_dev(b, dev) for b in bs]
    dts = [tiled_dev(w, n, K, dev) for w, n in zip(dws, Ns)]
    yr, yt = ([empty_f32((M, n), dev) for n in Ns] for _ in range(2))
    capi.linear_multi(dx, dws, dbs, yr, Ns, M, K)
    capi.linear_multi_tiled(dx, dts, dbs, yt, Ns, M, K)
    for i, n in enumerate(Ns):
        got = to_host(yr[i])
        assert_bitexact(to_host(yt[i]), got, f"tiled vs raw {i}")
        assert rel_l2(got, orc.linear(x, ws[i], bs[i], M, n, K)) <= tol(M)
        if M < 64:
            single = empty_f32((M, n), dev)
            capi.linear(dx, dws[i], dbs[i], single, M, n, K)
            assert_bitexact(to_host(single), got, f"single vs fused {i}")


@pytest.mark.parametrize("M,N,K", [(17, 50, 64), (40, 1111, 4096), (63, 8000, 544),
                                   (48, 11008, 1056), (10, 300, 992)])
def test_mid_swiglu(dev, orc, M, N, K):
    note(f"mid swiglu M={M} N={N} K={K}")
    wg, wu = weight(920, N, K), weight(921, N, K)
    x = S.activations(922, (M, K))
    dx, dg, du = to_dev(x, dev), to_dev(wg, dev), to_dev(wu, dev)
    yr, yt = empty_f32((M, N), dev), empty_f32((M, N), dev)
    capi.linear_swiglu(dx, dg, du, yr, M, N, K)
    capi.linear_swiglu_tiled(dx, tiled_dev(dg, N, K, dev), tiled_dev(du, N, K, dev), yt, M, N, K)
    got = to_host(yr)
    assert_bitexact(to_host(yt), got, "tiled vs raw")
    rows = np.unique(np.linspace(0, N - 1, min(N, 200)).astype(int))
    cut = [np.ascontiguousarray(w.reshape(N, -1)[rows]).reshape(-1) for w in (wg, wu)]
    g, u = (orc.sgemm_nt(x, w, M, rows.size, K).astype(np.float64) for w in cut)
    assert rel_l2(got[:, rows], g / (1.0 + np.exp(-g)) * u) <= tol(M)


@pytest.mark.parametrize("M", [24, 70])
def test_mid_special_values(dev, M):
    """Inf, NaN, zero rows and the largest magnitudes give the general path's non-finite
    entries and its finite values, on both layouts; other tokens are untouched."""
    N, K = 96, 1056
    raw = weight(930, N, K)
    x = S.activations(931, (M, K))
    x[1, 5], x[2, 100], x[3, 7], x[4, :], x[5, 3] = np.inf, -np.inf, np.nan, 0.0, 3.0e38
    note(f"mid special values M={M}")
    dx, dw = to_dev(x, dev), to_dev(raw, dev)
    y, yt, yg = (empty_f32((M, N), dev) for _ in range(3))
    capi.linear(dx, dw, None, y, M, N, K)
    capi.linear_tiled(dx, tiled_dev(dw, N, K, dev), None, yt, M, N, K)
    capi.linear_ex(dx, dw, None, yg, M, N, K, path=3 if M < 64 else 2)
    got, want = to_host(y), to_host(yg)
    assert_bitexact(to_host(yt), got, "tiled vs raw")
    fin = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fin) and not fin[1:4].all() and fin[6:].all()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])
    ok = fin.copy()
    ok[5] = False  # 3e38 products: the sum's order decides what overflows
    assert rel_l2(got[ok], want[ok]) <= (1e-6 if M < 64 else 1e-2)


def test_mid_split_counters_and_noalloc(dev):
    """Launches of different split counts back to back on one stream leave the counters
    clean, and the no-allocation entry point gives the same bits."""
    import torch
    note("mid split counters")
    x = to_dev(S.activations(940, (63, 8256)), dev)
    for N, K in ((200, 8256), (700, 512), (64, 4096), (200, 8256)):
        dw = to_dev(weight(941, N, K), dev)
        y, y2 = empty_f32((63, N), dev), empty_f32((63, N), dev)
        capi.linear(x, dw, None, y, 63, N, K)
        capi.linear_noalloc(x, dw, None, y2, 63, N, K)
        torch.cuda.synchronize()
        assert torch.equal(y, y2) and bool(torch.isfinite(y).all())


def test_mid_capture_on_a_smaller_reservation(dev):
    """A stream whose graph workspace was reserved for 16 tokens still captures 40: the
    row tiles share it in several launches, with the eager call's bits."""
    import torch
    M, N, K = 40, 4096, 8192  # 5.5 MB of partials; a reservation holds at least 4 MiB
    note("mid capture on a smaller reservation")
    x, dw = to_dev(S.activations(950, (M, K)), dev), to_dev(weight(951, N, K), dev)
    y, eager = empty_f32((M, N), dev), empty_f32((M, N), dev)
    st = torch.cuda.Stream()
    capi.workspace_reserve(1, 1, stream=st)
    capi.linear(x, dw, None, eager, M, N, K, stream=st)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        capi.linear(x, dw, None, y, M, N, K, stream=st)
    for _ in range(3):
        y.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert_bitexact(to_host(y), to_host(eager), "replay vs eager")


def test_mid_noalloc_scratch_limit(dev):
    """K splits whose partials outgrow the no-allocation scratch (33.6 MB at 16400 rows)
    give mle_q8_0_linear's bits there too."""
    M, N, K = 63, 16400, 4128
    note("mid noalloc scratch limit")
    x, dw = to_dev(S.activations(960, (M, K)), dev), to_dev(weight(961, N, K), dev)
    y, y2 = empty_f32((M, N), dev), empty_f32((M, N), dev)
    capi.linear(x, dw, None, y, M, N, K)
    capi.linear_noalloc(x, dw, None, y2, M, N, K)
    assert_bitexact(to_host(y2), to_host(y), "noalloc vs linear")


def test_mid_multi_past_the_split_bound(dev):
    """Three outputs of 49152 rows together, each below the bound from which a launch
    takes no K splits, keep their single Linears' bits."""
    M, N, K = 20, 16384, 544
    note("mid multi past the split bound")
    x = to_dev(S.activations(970, (M, K)), dev)
    ws = [to_dev(weight(971 + i, N, K), dev) for i in range(3)]
    ys, one = [empty_f32((M, N), dev) for _ in ws], empty_f32((M, N), dev)
    capi.linear_multi(x, ws, [None] * 3, ys, [N] * 3, M, K)
    for w, y in zip(ws, ys):
        capi.linear(x, w, None, one, M, N, K)
        assert_bitexact(to_host(y), to_host(one), "fused vs single")


@pytest.mark.parametrize("M,N,K", [(9, 100, 32), (12, 6000, 896), (16, 1024, 1024)])
def test_up_to_16_tokens_take_the_decode(dev, M, N, K):
    """9-16 tokens on rows of any length run the 16-token decode: its bits, on both layouts
    and in a fused launch."""
    note(f"16-token decode M={M} N={N} K={K}")
    x, dw = to_dev(S.activations(980, (M, K)), dev), to_dev(weight(981, N, K), dev)
    y, yt, yd, y0, y1 = (empty_f32((M, N), dev) for _ in range(5))
    capi.linear(x, dw, None, y, M, N, K)
    capi.linear_tiled(x, tiled_dev(dw, N, K, dev), None, yt, M, N, K)
    capi.linear_ex(x, dw, None, yd, M, N, K, path=3)
    capi.linear_multi(x, [dw, dw], [None] * 2, [y0, y1], [N] * 2, M, K)
    want = to_host(yd)
    for got in (y, yt, y0, y1):
        assert_bitexact(to_host(got), want, "decode bits")


@pytest.mark.parametrize("M,N,K,tiled", [
    (17, 9216, 5120, False), (20, 6400, 5120, True), (17, 13824, 1024, False),
    (20, 49136, 768, False), (17, 50880, 4096, False)])
def test_mid_is_no_slower_than_chunks(dev, M, N, K, tiled):
    """Row groups that leave a partly filled round of workgroups: the launch agrees with the
    16-token chunks of the decode, which the tuning hook forces, and takes no longer (the
    best of nine runs each, in turn; these took 1.15-1.25 times as long)."""
    note(f"mid vs chunks M={M} N={N} K={K} tiled={tiled}")
    x, w = to_dev(S.activations(990, (M, K)), dev), to_dev(weight(991, N, K), dev)
    if tiled:
        w = tiled_dev(w, N, K, dev)
    y, yd = empty_f32((M, N), dev), empty_f32((M, N), dev)
    auto = capi.linear_tiled if tiled else capi.linear
    ratio = slower_by(lambda: auto(x, w, None, y, M, N, K),
                      lambda: capi.linear_ex(x, w, None, yd, M, N, K, path=3, tiled=tiled))
    assert rel_l2(to_host(y), to_host(yd)) <= 1e-6
    assert ratio <= 1.05, ratio


@pytest.mark.parametrize("M,N,K", [(70, 7952, 6656), (80, 7168, 11008), (95, 4224, 15872),
                                   (96, 4864, 8192), (81, 4608, 11008)])
def test_mid_is_no_slower_than_the_gemm(dev, M, N, K):
    """64-96 tokens on rows past 4096 elements and more row groups than the batch kernel's
    K splits have room for: no slower than the GEMM, which the tuning hook forces (the best
    of nine runs each, in turn; these took 1.35-1.5 times as long, now the same kernel)."""
    note(f"mid vs gemm M={M} N={N} K={K}")
    x, w = to_dev(S.activations(992, (M, K)), dev), to_dev(weight(993, N, K), dev)
    y, yg = empty_f32((M, N), dev), empty_f32((M, N), dev)
    ratio = slower_by(lambda: capi.linear(x, w, None, y, M, N, K),
                      lambda: capi.linear_ex(x, w, None, yg, M, N, K, path=2))
    assert rel_l2(to_host(y), to_host(yg)) <= 1e-2
    assert ratio <= 1.15, ratio


@pytest.mark.parametrize("M,N,K,tiled", [(18, 24, 60000, False), (38, 100, 48000, True),
                                         (20, 300, 27008, False), (34, 40, 58464, False)])
def test_mid_long_rows_are_no_slower_than_chunks(dev, M, N, K, tiled):
    """Few outputs of very long rows: K splits enough to occupy the GPU, so the launch takes
    no longer than the 16-token chunks (these took 1.2-2.2 times as long with 8 splits)."""
    note(f"mid long rows M={M} N={N} K={K} tiled={tiled}")
    x, w = to_dev(S.activations(994, (M, K)), dev), to_dev(weight(995, N, K), dev)
    if tiled:
        w = tiled_dev(w, N, K, dev)
    y, yd = empty_f32((M, N), dev), empty_f32((M, N), dev)
    auto = capi.linear_tiled if tiled else capi.linear
    ratio = slower_by(lambda: auto(x, w, None, y, M, N, K),
                      lambda: capi.linear_ex(x, w, None, yd, M, N, K, path=3, tiled=tiled))
    assert rel_l2(to_host(y), to_host(yd)) <= 1e-6
    assert ratio <= 1.05, ratio


@pytest.mark.parametrize("M,N,K", [(24, 640, 54336), (20, 200, 19680), (32, 400, 8192)])
def test_mid_swiglu_long_rows_are_no_slower_than_chunks(dev, M, N, K):
    """The same for a gate/up pair, against its calls for 16 tokens and for the rest."""
    note(f"mid swiglu long rows M={M} N={N} K={K}")
    x = to_dev(S.activations(996, (M, K)), dev)
    g, u = to_dev(weight(997, N, K), dev), to_dev(weight(998, N, K), dev)
    y, yc = empty_f32((M, N), dev), empty_f32((M, N), dev)

    def chunks():
        capi.linear_swiglu(x[:16], g, u, yc[:16], 16, N, K)
        capi.linear_swiglu(x[16:], g, u, yc[16:], M - 16, N, K)

    ratio = slower_by(lambda: capi.linear_swiglu(x, g, u, y, M, N, K), chunks)
    assert rel_l2(to_host(y), to_host(yc)) <= 2e-6
    assert ratio <= 1.05, ratio


@pytest.mark.parametrize("Ns,K", [((4096, 512, 80), 12288), ((1000, 1000, 1000), 12288),
                                  ((32, 2048, 32), 22528), ((16384, 16384, 16384), 1024),
                                  ((49200, 64, 96), 544)])
def test_mid_multi_of_different_splits(dev, Ns, K):
    """Outputs that split K differently alone keep their single Linears' bits in one fused
    call, and outputs that split alike share a launch."""
    M = 21
    note(f"mid multi of different splits Ns={Ns} K={K}")
    x = to_dev(S.activations(975, (M, K)), dev)
    ws = [to_dev(weight(976 + i, n, K), dev) for i, n in enumerate(Ns)]
    ys = [empty_f32((M, n), dev) for n in Ns]
    yt = [empty_f32((M, n), dev) for n in Ns]
    capi.linear_multi(x, ws, [None] * 3, ys, Ns, M, K)
    capi.linear_multi_tiled(x, [tiled_dev(w, n, K, dev) for w, n in zip(ws, Ns)], [None] * 3, yt,
                            Ns, M, K)
    for w, n, y, t in zip(ws, Ns, ys, yt):
        one = empty_f32((M, n), dev)
        capi.linear(x, w, None, one, M, n, K)
        assert_bitexact(to_host(y), to_host(one), "fused vs single")
        assert_bitexact(to_host(t), to_host(one), "tiled vs raw")
