"""GPU parity of the fused Linear entry points against the CPU oracle.

* ``mle_q8_0_linear_swiglu``: y = silu(x . Wg^T) * (x . Wu^T), silu(g) = g / (1 + e^-g)
  (reference cpu_kernels.cpp:848-858 applied to two Linears, cpu_kernels.cpp:208-218).
  The oracle side is the oracle's own two Linears followed by silu * up in float64.
* ``mle_q8_0_linear_multi``: up to three Linears on one input in one launch; each output
  against the oracle Linear (+ bias), and bit for bit against the single Linear entry
  point for M < 64 (same kernels, same arithmetic).

Bars: relative L2 <= 1e-5 for M < 64 (FP32-exact MFMA decode) and <= 1e-2 for M >= 64
(bf16 MFMA GEMM), as for the plain Linear.
"""
import functools

import numpy as np
import pytest

from helpers import empty_f32, note, own_stream, rel_l2, to_dev, to_host
from llmengine_amd import capi
from llmengine_amd import synthetic as S

pytestmark = pytest.mark.gpu


def tol(M):
    return 1e-5 if M < 64 else 1e-2


@functools.lru_cache(maxsize=None)
def weight(seed, rows, cols):
    return S.q8_0_weight(seed, rows, cols)[0]


def silu_mul(g, u):
    g = g.astype(np.float64)
    return g / (1.0 + np.exp(-g)) * u.astype(np.float64)


@pytest.mark.parametrize("M,N,K", [(1, 300, 512), (3, 333, 1024), (8, 1000, 4096),
                                   (16, 256, 256), (17, 96, 992), (40, 130, 64),
                                   (64, 192, 256), (100, 320, 1024), (129, 64, 512)])
def test_swiglu_matches_oracle(dev, orc, M, N, K):
    note(f"swiglu M={M} N={N} K={K}")
    wg, wu = weight(60 + N, N, K), weight(61 + N, N, K)
    x = S.activations(62 + K, (M, K))
    want = silu_mul(orc.linear(x, wg, None, M, N, K), orc.linear(x, wu, None, M, N, K))
    y = empty_f32((M, N), dev)
    capi.linear_swiglu(to_dev(x, dev), to_dev(wg, dev), to_dev(wu, dev), y, M, N, K)
    err = rel_l2(to_host(y), want)
    assert err <= tol(M), err


@pytest.mark.parametrize("M", [1, 8, 512])
def test_swiglu_llama_ffn_full(dev, orc, M):
    """Llama-7B gate/up [11008, 4096] at decode and prefill sizes: the whole output
    against the separate Linears of the same entry points (silu * up in float64),
    sampled rows against the oracle, and repeats bitwise equal."""
    import torch
    N, K = 11008, 4096
    note(f"swiglu llama M={M}")
    wg, wu = to_dev(weight(23, N, K), dev), to_dev(weight(24, N, K), dev)
    xh = S.activations(25, (M, K))
    x = to_dev(xh, dev)
    y, y2 = empty_f32((M, N), dev), empty_f32((M, N), dev)
    g, u = empty_f32((M, N), dev), empty_f32((M, N), dev)
    capi.linear_swiglu(x, wg, wu, y, M, N, K)
    capi.linear_swiglu(x, wg, wu, y2, M, N, K)
    capi.linear(x, wg, None, g, M, N, K)
    capi.linear(x, wu, None, u, M, N, K)
    torch.cuda.synchronize()
    assert torch.equal(y, y2)
    got = to_host(y)
    assert rel_l2(got, silu_mul(to_host(g), to_host(u))) <= tol(M)
    rows = np.array([0, M // 2, M - 1])
    wgh, wuh = weight(23, N, K), weight(24, N, K)
    want_rows = silu_mul(orc.sgemm_nt(xh[rows], wgh, rows.size, N, K),
                         orc.sgemm_nt(xh[rows], wuh, rows.size, N, K))
    assert rel_l2(got[rows], want_rows) <= tol(M)


@pytest.mark.parametrize("M", [1, 2, 5, 16, 40, 70])
def test_multi_output_matches_oracle_and_single(dev, orc, M):
    import torch
    K = 512
    Ns = (160, 96, 32)
    ws = [weight(70 + i, n, K) for i, n in enumerate(Ns)]
    biases = [S.activations(80, (Ns[0],), tag=S.TAG_BIAS), None,
              S.activations(82, (Ns[2],), tag=S.TAG_BIAS)]
    x = S.activations(83, (M, K))
    note(f"multi M={M} Ns={Ns}")
    dx = to_dev(x, dev)
    dws = [to_dev(w, dev) for w in ws]
    dbs = [to_dev(b, dev) if b is not None else None for b in biases]
    ys = [empty_f32((M, n), dev) for n in Ns]
    capi.linear_multi(dx, dws, dbs, ys, Ns, M, K)
    torch.cuda.synchronize()
    for i, n in enumerate(Ns):
        want = orc.linear(x, ws[i], biases[i], M, n, K)
        got = to_host(ys[i])
        assert rel_l2(got, want) <= tol(M), i
        if M < 64:
            single = empty_f32((M, n), dev)
            capi.linear(dx, dws[i], dbs[i], single, M, n, K)
            torch.cuda.synchronize()
            assert torch.equal(single, ys[i]), i


@pytest.mark.parametrize("M,Ns", [(1, (4096, 1024, 1024)), (2, (4096, 1024, 1024)),
                                  (2, (4096, 4096, 4096)), (4, (4096, 1024, 1024)),
                                  (4, (4096, 4096, 4096)), (8, (4096, 4096, 4096))])
def test_multi_output_llama_qkv(dev, orc, M, Ns):
    """q/k/v of a grouped-query ([4096, 4096], [1024, 4096] x 2) and a multi-head
    ([4096, 4096] x 3) layer: one launch equals three single Linears bit for bit
    (at M=8 the fused multi-head launch uses 8-wave workgroups, the single ones
    4-wave), except where the fused launch alone takes the row-range decode (4 tokens
    on 512-1024 row groups: the multi-head layer's 768), within 1e-6 there; each
    output is within 1e-5 relative L2 of the oracle."""
    import torch
    K = 4096
    hws = [weight(90 + i, n, K) for i, n in enumerate(Ns)]
    hx = S.activations(93, (M, K))
    dws = [to_dev(w, dev) for w in hws]
    dx = to_dev(hx, dev)
    ys = [empty_f32((M, n), dev) for n in Ns]
    for rep in range(3):  # repeated launches reuse the workspace: same bits every time
        capi.linear_multi(dx, dws, None, ys, Ns, M, K)
        torch.cuda.synchronize()
        if rep == 0:
            first = [y.clone() for y in ys]
        else:
            assert all(torch.equal(a, b) for a, b in zip(first, ys))
    G = sum((n + 15) // 16 for n in Ns)
    fused_rows = M in (3, 4) and 512 <= G <= 1024
    for i, n in enumerate(Ns):
        single = empty_f32((M, n), dev)
        capi.linear(dx, dws[i], None, single, M, n, K)
        torch.cuda.synchronize()
        if fused_rows:
            assert rel_l2(to_host(ys[i]), to_host(single)) <= 1e-6, i
        else:
            assert torch.equal(single, ys[i]), i
        assert rel_l2(to_host(ys[i]), orc.sgemm_nt(hx, hws[i], M, n, K)) <= 1e-5, i


# ----------------------------------------------------------------------------- argmax

def first_argmax(x):
    """Greedy pick of the reference (first maximum; NaN ignored; all-NaN -> 0)."""
    out = []
    for row in x:
        ok = ~np.isnan(row)
        if not ok.any():
            out.append(0)
            continue
        best = np.max(row[ok])
        out.append(int(np.flatnonzero(ok & (row == best))[0]))
    return np.array(out, dtype=np.int32)


@pytest.mark.parametrize("rows,n", [(1, 1), (1, 7), (3, 2048), (2, 2049), (8, 151936),
                                    (1, 151936), (5, 100_000)])
def test_argmax_matches_first_maximum(dev, rows, n):
    import torch
    note(f"argmax rows={rows} n={n}")
    x = S.activations(200 + n, (rows, n))
    idx = torch.empty(rows, dtype=torch.int32, device=dev)
    val = empty_f32((rows,), dev)
    capi.argmax(to_dev(x, dev), rows, n, idx, val)
    torch.cuda.synchronize()
    want = first_argmax(x)
    assert np.array_equal(idx.cpu().numpy(), want)
    assert np.array_equal(val.cpu().numpy(), x[np.arange(rows), want])


@pytest.mark.parametrize("rows,n", [(1, 1), (3, 2047), (2, 2048), (2, 2049), (5, 4097),
                                    (128, 2050), (129, 2050), (1, 524289), (2, 600001)])
def test_argmax_chunk_edges(dev, rows, n):
    """The maximum at the ends of chunks and rows, rows of any 4-byte alignment, on both
    sides of the one-launch bound; back-to-back calls and replays of a capture leave the
    shared counters clean."""
    import torch
    note(f"argmax chunk edges rows={rows} n={n}")
    x = S.activations(700, (rows, n))
    places = [0, n - 1, min(n - 1, 2047), min(n - 1, 2048), n // 2]
    wants, devs = [], []
    for k in range(3):
        for r in range(rows):
            x[r, places[(r + k) % 5]] = 20.0 + k
        wants.append(first_argmax(x))
        devs.append(to_dev(x, dev))
    idx, val = torch.empty(rows, dtype=torch.int32, device=dev), empty_f32((rows,), dev)
    for k in (0, 1, 2, 0):
        capi.argmax(devs[k], rows, n, idx, val)
        assert idx.cpu().numpy().tolist() == wants[k].tolist()
        assert to_host(val).tolist() == [20.0 + k] * rows
    for counters in (0, rows * 32):  # bytes alone are enough
        st = own_stream() if counters else torch.cuda.Stream()
        capi.workspace_reserve(16 * rows * 256, counters, stream=st)
        g = torch.cuda.CUDAGraph()
        y = devs[0].clone()
        idx2, val2 = torch.empty_like(idx), torch.empty_like(val)
        with torch.cuda.graph(g, stream=st):
            capi.argmax(y, rows, n, idx, val, stream=st)
        for k in (1, 2, 0):
            y.copy_(devs[k])
            for _ in range(2):
                idx.fill_(-1)
                val.fill_(float("nan"))
                g.replay()
                assert idx.cpu().numpy().tolist() == wants[k].tolist()
                assert to_host(val).tolist() == [20.0 + k] * rows
                capi.argmax(devs[(k + 1) % 3], rows, n, idx2, val2)


@pytest.mark.parametrize("rows,n", [(1, 196608), (3, 196609), (2, 300001), (1, 393216),
                                    (2, 393217), (1, 524288)])
def test_argmax_long_rows(dev, rows, n):
    """Rows of more pieces than meet at a counter: two pieces a chunk, then (counted as the
    nodes of a capture) two launches; the maximum in any piece, the first of ties."""
    import ctypes
    import torch
    note(f"argmax long rows rows={rows} n={n}")
    x = np.zeros((rows, n), np.float32)
    x[:, ::3] = -1.0
    idx, val = torch.empty(rows, dtype=torch.int32, device=dev), empty_f32((rows,), dev)
    for at in (0, 1, 2047, 2048, 4096, 196607, n - 2, n - 1):
        y = x.copy()
        y[:, min(at, n - 1):] = np.where(y[:, min(at, n - 1):] < 0, 2.0, 1.0)
        capi.argmax(to_dev(y, dev), rows, n, idx, val)
        want = first_argmax(y)
        assert np.array_equal(idx.cpu().numpy(), want)
        assert np.array_equal(to_host(val), y[np.arange(rows), want])
    st = own_stream()
    capi.workspace_reserve(16 * rows * 256, rows * 32, stream=st)
    g = torch.cuda.CUDAGraph(keep_graph=True)
    d = to_dev(x, dev)
    with torch.cuda.graph(g, stream=st):
        capi.argmax(d, rows, n, idx, val, stream=st)
    nodes = ctypes.c_size_t(0)
    rc = capi.load().hipGraphGetNodes(ctypes.c_void_p(g.raw_cuda_graph()), None,
                                      ctypes.byref(nodes))
    assert rc == 0 and nodes.value == (1 if n <= 393216 else 2)


def test_argmax_on_a_reservation_of_bytes_allocates_nothing(dev):
    """A loop that reserved bytes alone for its greedy picks: eager calls allocate nothing
    (the pick's counters included), and captured ones are accepted."""
    import torch
    note("argmax on a reservation of bytes")
    rows, n = 128, 5000
    x = S.activations(710, (rows, n))
    d, want = to_dev(x, dev), first_argmax(x)
    idx, val = torch.empty(rows, dtype=torch.int32, device=dev), empty_f32((rows,), dev)
    st = own_stream()
    capi.workspace_reserve(16 * rows * 256, 0, stream=st)
    gen = capi.workspace_info(st)[2]
    torch.cuda.synchronize()
    for _ in range(3):
        capi.argmax(d, rows, n, idx, val, stream=st)
    st.synchronize()
    assert np.array_equal(idx.cpu().numpy(), want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        capi.argmax(d, rows, n, idx, val, stream=st)
    for _ in range(3):
        idx.fill_(-1)
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(idx.cpu().numpy(), want)
    assert capi.workspace_info(st)[2] == gen


def test_argmax_ties_signed_zero_and_nan(dev):
    import torch
    n = 10_000
    x = np.full((6, n), -1.0, dtype=np.float32)
    x[0, [4000, 17, 9000]] = 3.0                    # tie -> lowest index 17
    x[1, :] = 0.0
    x[1, 5] = -0.0                                  # -0 == +0: index 0 wins
    x[1, 0] = -0.0
    x[2, :] = np.nan
    x[2, 7777] = -5.0                               # only non-NaN value
    x[3, :] = np.nan                                # NaN only -> 0
    x[4, :] = -np.inf
    x[4, 123] = np.float32(-3.4e38)                 # finite beats -inf
    x[5, :] = np.inf                                # all +inf -> 0
    idx = torch.empty(6, dtype=torch.int32, device=dev)
    val = empty_f32((6,), dev)
    capi.argmax(to_dev(x, dev), 6, n, idx, val)
    torch.cuda.synchronize()
    got = idx.cpu().numpy()
    assert got.tolist() == [17, 0, 7777, 0, 123, 0]
    v = val.cpu().numpy()
    assert v[0] == 3.0 and v[2] == -5.0 and np.isnan(v[3]) and v[5] == np.inf
    assert first_argmax(x).tolist() == got.tolist()


def test_lm_head_then_argmax(dev, orc):
    """Tied lm_head [151936, 896] Linear at M=1 and M=8 followed by the device argmax:
    the picked token equals the first maximum of the oracle's logits wherever the
    top two oracle logits are not within the Linear's error of each other."""
    import torch
    V, H = 151936, 896
    w = weight(300, V, H)
    dw = to_dev(w, dev)
    for M in (1, 8):
        x = S.activations(301 + M, (M, H))
        logits = empty_f32((M, V), dev)
        capi.linear(to_dev(x, dev), dw, None, logits, M, V, H)
        idx = torch.empty(M, dtype=torch.int32, device=dev)
        capi.argmax(logits, M, V, idx)
        torch.cuda.synchronize()
        assert np.array_equal(idx.cpu().numpy(), first_argmax(to_host(logits)))
        want = orc.linear(x, w, None, M, V, H)
        top2 = np.sort(want, axis=1)[:, -2:]
        clear = (top2[:, 1] - top2[:, 0]) > 1e-4 * np.abs(top2[:, 1])
        assert np.array_equal(idx.cpu().numpy()[clear], first_argmax(want)[clear])
