"""The fp32 GEMMs and convolutions on fp16 split products (at the op level launches
of at least 512 rows, K >= 128 and 1.25e9 multiply-adds): edges of the tiles, of the K split and of
the range that two fp16 terms cover, against 64-bit products.

Bound per element: every product term is exact in the fp32 accumulation, which
takes at most 3 K / 16 + 32 roundings (each of at most 2^-23 of a partial sum, and
those are at most S = sum |x w|), and the dropped parts of the operands are below
2^-21 S together: |error| <= (3 K / 16 + 32) 2^-23 S + 2^-21 S. What small values lose
beside large ones is below 1.5 2^-21 S where the sums certify it, and such elements
are computed in fp32 where they do not."""
import numpy as np
import pytest
import torch

import gsplat_hip as G
from gpu_util import KEEP, case, dev, empty, host, stream

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(11)


def rnd(*s, scale=1.0):
    return (RNG.standard_normal(s) * scale).astype(np.float32)


def linear(x, w, b=None, res=None, epi=0):
    M, K = x.shape
    N = w.shape[0]
    y = empty(M, N)
    xd, wd = dev(x), dev(w)
    bd = None if b is None else dev(b)
    rd = None if res is None else dev(res)
    G.check(G.lib().gs_hip_linear(G.ptr(xd), G.ptr(wd), G.ptr(bd), G.ptr(y), M, K, N, 0,
                                  epi | (G.EPI_RESIDUAL if res is not None else 0), G.ptr(rd), stream()))
    return host(y)


def assert_bound(got, x, w, extra=0.0):
    K = x.shape[1]
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    ref, S = x64 @ w64.T, np.abs(x64) @ np.abs(w64).T
    bound = ((3 * K / 16 + 32) * 2.0 ** -23 + 2.0 ** -21) * S + extra
    err = np.abs(got - ref)
    assert (err <= bound).all(), f"worst {np.max(err / np.maximum(bound, 1e-300)):.3g} of the bound"
    return np.sqrt(np.mean(err ** 2)) / max(np.sqrt(np.mean(ref ** 2)), 1e-300)


@pytest.mark.parametrize("M,K,N", [(272001, 128, 36), (61000, 160, 132), (4100, 128, 2404),
                                   (2049, 4096, 164), (1000, 992, 1284), (9000, 224, 1540),
                                   (12290, 768, 516), (513, 4096, 644), (12800, 100, 1000),
                                   (10000, 131, 1000)])
def test_linear_split_products(M, K, N):
    """Ragged tiles in M and N, few and many K steps, split and unsplit K,
    zero-padded K (100 -> 128, 131 -> 160)."""
    case(f"split linear M={M} K={K} N={N}")
    x, w = rnd(M, K), rnd(N, K, scale=0.02)
    rel = assert_bound(linear(x, w), x, w)
    print(f"M={M} K={K} N={N}: rms error {rel:.2e} of the result's")


@pytest.mark.parametrize("epi", ["gelu", "relu", "residual"])
@pytest.mark.parametrize("M,K,N", [(768, 1600, 1028), (12300, 256, 1024)])
def test_linear_split_epilogues(epi, M, K, N):
    case(f"split linear {epi} M={M}")
    x, w, b, r = rnd(M, K), rnd(N, K, scale=0.05), rnd(N, scale=0.1), rnd(M, N)
    v = x.astype(np.float64) @ w.astype(np.float64).T + b
    S = np.abs(x.astype(np.float64)) @ np.abs(w.astype(np.float64)).T
    bound = ((3 * K / 16 + 32) * 2.0 ** -23 + 2.0 ** -21) * S + 1e-6 * (1 + np.abs(v))
    if epi == "gelu":  # slope at most 1.13
        ref = 0.5 * v * (1 + np.tanh(np.sqrt(2 / np.pi) * (v + 0.044715 * v ** 3)))
        got = linear(x, w, b, epi=G.EPI_GELU)
    elif epi == "relu":
        ref, got = np.maximum(v, 0), linear(x, w, b, epi=G.EPI_RELU)
    else:
        ref, got = v + r, linear(x, w, b, res=r)
        bound = bound + 2.0 ** -22 * np.abs(ref)
    assert (np.abs(got - ref) <= 1.2 * bound).all()


def test_linear_split_row_and_column_magnitudes():
    """Rows of x and of W from 1e-30 to 1e18 and rows of zeros: every row
    outside the unscaled range takes its own power of two."""
    case("split linear magnitudes")
    M, K, N = 2560, 512, 1024
    xs = np.array([1.0, 1e-30, 1e-12, 3e-5, 3e-3, 40.0, 7e4, 1e9, 1e18, 0.0])
    ws = np.array([0.02, 1e-18, 1e-9, 30.0, 1e12, 0.0])
    x = (rnd(M, K) * xs[np.arange(M) % len(xs)][:, None].astype(np.float32))
    w = (rnd(N, K) * ws[np.arange(N) % len(ws)][:, None].astype(np.float32))
    # results below the normal range are rounded to multiples of 2^-149
    assert_bound(linear(x, w), x, w, extra=2.0 ** -140)


@pytest.mark.parametrize("xs,ws", [(1e-36, 1e35), (1e-20, 1e33), (1e-30, 1e35), (1e-4, 1e34), (1e30, 1e-36)])
def test_linear_split_magnitudes_that_cancel(xs, ws):
    """Rows of x and of W that only together are in range."""
    case(f"split linear magnitudes {xs} {ws}")
    M, K, N = 2560, 1024, 512
    x, w = rnd(M, K) * np.float32(xs), rnd(N, K) * np.float32(ws)
    assert_bound(linear(x, w), x, w, extra=2.0 ** -140)


def test_linear_split_wide_rows():
    """One element 2^26 times the others, met by a zero weight: the others keep
    full precision (their products are all the result)."""
    case("split linear wide rows")
    M, K, N = 2560, 512, 1024
    x, w = rnd(M, K), rnd(N, K)
    x[:, 7] = 2.0 ** 26
    w[:, 7] = 0.0
    assert_bound(linear(x, w), x, w)


def assert_wide(got, x, w):
    """assert_bound, and the errors of all elements together within 1.5e-6 of S
    (three roundings of 2^-24 per 512 of K and the kernel's 1.5 2^-21)."""
    assert_bound(got, x, w)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    S = np.abs(x64) @ np.abs(w64).T
    assert np.sqrt(np.mean(((got - x64 @ w64.T) / S) ** 2)) < 1.5e-6


@pytest.mark.parametrize("M,K,N", [(2560, 512, 1024), (1100, 2048, 644)])
@pytest.mark.parametrize("loud,rest", [(2.0 ** -7, -22), (2.0 ** -7, -45), (1.0, -20), (1.0, -26), (1.0, -37),
                                       (32.0, -30), (2.0 ** 26, -5), (2.0 ** 26, -30)])
def test_linear_split_one_loud_value(loud, rest, M, K, N):
    """A loud value that meets zeros: the others' products are all the result,
    whatever the two magnitudes; in x, in W, and behind the sampled values."""
    case(f"split linear loud {loud} rest 2^{rest} M={M}")
    for at in (7, K - 3):
        x, w = rnd(M, K, scale=2.0 ** rest), rnd(N, K)
        x[:, at], w[:, at] = loud, 0.0
        assert_wide(linear(x, w), x, w)
    x, w = rnd(M, K), rnd(N, K, scale=2.0 ** rest)
    x[:, 7], w[:, 7] = 0.0, loud
    assert_wide(linear(x, w), x, w)


def test_linear_split_values_of_all_magnitudes():
    """Rows whose values spread over 2^-60 .. 1, and rows of zeros."""
    case("split linear spread")
    M, K, N = 2560, 512, 1024
    x = rnd(M, K) * np.exp2(RNG.uniform(-60, 0, (M, K))).astype(np.float32)
    w = rnd(N, K) * np.exp2(RNG.uniform(-60, 0, (N, K))).astype(np.float32)
    x[5::7, :] = 0.0
    w[3::11, :] = 0.0
    x[2, :300] = 0.0
    got = linear(x, w)
    assert_bound(got, x, w)
    assert not got[5::7].any() and not got[:, 3::11].any()


def test_conv_split_one_loud_channel():
    """A loud input channel with zero weights, the others far below it, also where
    the window's first taps are outside the image."""
    case("split conv loud channel")
    B, H, W, Ci, Co = 2, 40, 64, 96, 256
    x, w = rnd(B, H, W, Ci, scale=1e-9), rnd(Co, 3, 3, Ci, scale=0.05)
    x[..., 50], w[..., 50] = 3.0, 0.0
    conv = lambda a, f: torch.nn.functional.conv2d(
        torch.from_numpy(a.astype(np.float64)).permute(0, 3, 1, 2),
        torch.from_numpy(f.astype(np.float64)).permute(0, 3, 1, 2), padding=1).permute(0, 2, 3, 1).numpy()
    for relu in (False, True):
        xi = np.maximum(x, 0) if relu else x
        ref, S = conv(xi, w), conv(np.abs(xi), np.abs(w))
        y = empty(B, H, W, Co)
        xd, wd = dev(x), dev(w)
        G.check(G.lib().gs_hip_conv2d(G.ptr(xd), B, H, W, Ci, G.ptr(wd), None, G.ptr(y), Co, 3, 1, 1, 1,
                                      G.CONV_RELU_IN if relu else 0, None, stream()))
        K = 9 * Ci
        assert (np.abs(host(y) - ref) <= ((3 * K / 16 + 32) * 2.0 ** -23 + 2.0 ** -21) * S).all()


def test_linear_split_rows_do_not_depend_on_their_tile():
    """A row's bits are the same beside ordinary rows, rows that need a power
    of two and rows with infinities and NaN."""
    case("split linear neighbours")
    M, K, N = 2560, 512, 1024
    x, w = rnd(M, K), rnd(N, K, scale=0.02)
    base = linear(x, w)
    z = x.copy()
    z[5::64] *= 1e-9
    z[9::64, 3] = np.inf
    z[17::64, 100] = np.nan
    got = linear(z, w)
    same = np.ones(M, bool)
    for o in (5, 9, 17):
        same[o::64] = False
    np.testing.assert_array_equal(got[same], base[same])


@pytest.mark.parametrize("M,N,K", [(640, 512, 4096), (3000, 1024, 640)])
def test_linear_split_infinities_and_nan(M, N, K):
    """Infinities, NaN and finite values beyond fp16's and bf16's range in x and
    in W propagate as in IEEE arithmetic."""
    case(f"split linear non-finite M={M}")
    x, w = rnd(M, K), rnd(N, K, scale=0.02)
    x[3, 5], x[70, 0], x[130, 17], x[200, 9] = np.inf, -np.inf, np.nan, 3.3e38
    w[2, 5], w[40, 9], w[100, 11] = 0.0, np.inf, np.nan
    with np.errstate(invalid="ignore", over="ignore"):
        ref = (x.astype(np.float64) @ w.astype(np.float64).T).astype(np.float32)
    got = linear(x, w)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    np.testing.assert_array_equal(got[inf], ref[inf])
    ok = np.isfinite(ref)
    assert np.isfinite(got[ok]).all()
    S = np.abs(np.where(np.isfinite(x), x, 0).astype(np.float64)) @ np.abs(
        np.where(np.isfinite(w), w, 0).astype(np.float64)).T
    assert (np.abs(got.astype(np.float64) - ref)[ok] <= 1e-5 * S[ok] + 1e-30).all()


@pytest.mark.parametrize("B,H,W,Ci,Co,k,s,relu,res", [
    (2, 96, 130, 32, 256, 3, 1, True, True), (2, 83, 89, 96, 132, 3, 1, False, True),
    (4, 93, 97, 64, 256, 3, 2, False, False), (1, 200, 200, 160, 256, 1, 1, False, False),
    (2, 100, 131, 32, 256, 3, 1, True, False), (2, 31, 37, 256, 128, 5, 1, False, False)])
def test_conv_split_products(B, H, W, Ci, Co, k, s, relu, res):
    """Implicit-GEMM convolutions: padding, ragged rows, strides, the ReLU
    prologue and the residual, some pixels tiny and some huge."""
    case(f"split conv {B}x{H}x{W} {Ci}->{Co} k={k} s={s}")
    p = k // 2
    x, w, b = rnd(B, H, W, Ci), rnd(Co, k, k, Ci, scale=0.05), rnd(Co, scale=0.1)
    x[:, 3, 5] *= 1e-6
    x[:, -2, 7] *= 3e5
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    r = rnd(B, Ho, Wo, Co) if res else None
    xi = np.maximum(x, 0) if relu else x
    conv = lambda a, f: torch.nn.functional.conv2d(
        torch.from_numpy(a.astype(np.float64)).permute(0, 3, 1, 2),
        torch.from_numpy(f.astype(np.float64)).permute(0, 3, 1, 2), stride=s, padding=p).permute(0, 2, 3, 1).numpy()
    ref, S = conv(xi, w) + b, conv(np.abs(xi), np.abs(w))
    if res:
        ref = ref + r
    K = k * k * Ci
    bound = ((3 * K / 16 + 32) * 2.0 ** -23 + 2.0 ** -21) * S + 2.0 ** -22 * (np.abs(ref) + 1)
    y = empty(B, Ho, Wo, Co)
    xd, wd, bd, rd = dev(x), dev(w), dev(b), None if r is None else dev(r)
    G.check(G.lib().gs_hip_conv2d(G.ptr(xd), B, H, W, Ci, G.ptr(wd), G.ptr(bd), G.ptr(y), Co, k, s, p, 1,
                                  G.CONV_RELU_IN if relu else 0, G.ptr(rd), stream()))
    assert (np.abs(host(y) - ref) <= bound).all()


def test_context_weights_follow_set_weight(tiny_cfg):
    """The split planes are those of the weight set last, also under a replayed
    graph."""
    case("split planes after set_weight")
    cfg = G.default_config(**tiny_cfg)
    n = 3 * cfg.img_h * cfg.img_w
    imgs = [dev(G.seed_uniform(3, f"view{v}", n).reshape(1, 3, cfg.img_h, cfg.img_w)) for v in (1, 2)]
    outs = [empty(1, cfg.img_h, cfg.img_w, c) for c in (3, 1, cfg.desc_dim) * 2]
    KEEP.extend(imgs)
    s = torch.cuda.Stream()
    m = G.Mastr(cfg, 1)

    def run():
        m.pair(*imgs, 1, *outs, s.cuda_stream)
        torch.cuda.synchronize()
        return [host(o).copy() for o in outs]

    m.set_graph(True)
    m.init_seeded(0, 0.02, 0.1)
    first = run()
    m.init_seeded(1, 0.02, 0.1)
    second = run()
    m.init_seeded(0, 0.02, 0.1)
    again = run()
    m.close()
    for a, b, c in zip(first, second, again):
        assert not np.array_equal(a, b)
        np.testing.assert_array_equal(a, c)


# ---- attention on fp16 split products --------------------------------------------
def attention(q, k, v, prec=0):
    B, Nq, D = q.shape
    Nkv, H = k.shape[1], D // 64
    o = empty(B, Nq, D)
    qd, kd, vd = dev(q), dev(k), dev(v)
    sq, sk = (Nq * D, 64, D), (Nkv * D, 64, D)
    G.check(G.lib().gs_hip_attention_prec(G.ptr(qd), G.ptr(kd), G.ptr(vd), G.ptr(o), B, H, Nq, Nkv, 64, 0.125,
                                          *sq, *sk, *sk, *sq, prec, stream()))
    return host(o)


def attention64(q, k, v):
    B, Nq, D = q.shape
    h = lambda t: t.astype(np.float64).reshape(B, -1, D // 64, 64).transpose(0, 2, 1, 3)
    with np.errstate(invalid="ignore", over="ignore"):
        s = h(q) @ h(k).transpose(0, 1, 3, 2) * 0.125
        e = np.exp(s - s.max(-1, keepdims=True))
        p = e / e.sum(-1, keepdims=True)
        o = p @ h(v)
    # |error| <= |o|'s rounding + the score error times |v|: per score a few 2^-22 of
    # sum |q k| / 8, and the exponentials turn it into that share of P |v|
    ds = (np.abs(h(q)) @ np.abs(h(k)).transpose(0, 1, 3, 2)).max(-1, keepdims=True) * 0.125
    bound = (p @ np.abs(h(v))) * (2.0 ** -19 + ds * 2.0 ** -20)
    back = lambda t: t.transpose(0, 2, 1, 3).reshape(B, Nq, D)
    return back(o), back(bound)


@pytest.mark.parametrize("B,H,Nq,Nkv", [(1, 1, 1, 1), (1, 2, 31, 33), (2, 3, 129, 63), (1, 12, 768, 1000),
                                        (1, 16, 768, 768), (9, 16, 256, 65), (12, 16, 640, 130)])
def test_attention_split_products(B, H, Nq, Nkv):
    """Ragged queries and keys, one key, split and unsplit key ranges."""
    case(f"split attention B={B} H={H} Nq={Nq} Nkv={Nkv}")
    q, k, v = rnd(B, Nq, 64 * H), rnd(B, Nkv, 64 * H), rnd(B, Nkv, 64 * H)
    ref, bound = attention64(q, k, v)
    assert (np.abs(attention(q, k, v) - ref) <= bound).all()


@pytest.mark.parametrize("qs,ks,vs", [(1e-20, 1.0, 1.0), (1e4, 1e-3, 1.0), (30.0, 1.0, 1.0), (1.0, 1.0, 1e-9),
                                      (1.0, 1e-12, 1e-3), (1e-4, 3e4, 2e4), (1.0, 1.0, 3e5), (1e-6, 1e6, 1.0),
                                      (1.0, 1.0, 0.0)])
@pytest.mark.parametrize("B,Nkv", [(1, 700), (20, 200)])
def test_attention_split_magnitudes(qs, ks, vs, B, Nkv):
    case(f"split attention scales {qs} {ks} {vs} B={B}")
    q, k, v = rnd(B, 200, 768, scale=qs), rnd(B, Nkv, 768, scale=ks), rnd(B, Nkv, 768, scale=vs)
    ref, bound = attention64(q, k, v)
    assert (np.abs(attention(q, k, v) - ref) <= bound + 1e-44).all()


def check_attention(q, k, v, factor=1.0, prec=0):
    """Against 64 bits with attention64's bound, and with small inputs together within
    1.5e-6 of sum p |v| (factor: what large scores allow besides)."""
    ref, bound = attention64(q, k, v)
    err = np.abs(attention(q, k, v, prec) - ref)
    assert (err <= bound).all()
    B, Nq, D = q.shape
    h = lambda t: t.astype(np.float64).reshape(B, -1, D // 64, 64).transpose(0, 2, 1, 3)
    s = h(q) @ h(k).transpose(0, 1, 3, 2) * 0.125
    p = np.exp(s - s.max(-1, keepdims=True))
    S = ((p / p.sum(-1, keepdims=True)) @ np.abs(h(v))).transpose(0, 2, 1, 3).reshape(B, Nq, D)
    S = np.where(S > 0, S, 1.0)
    assert np.sqrt(np.mean((err / S) ** 2)) < 1.5e-6 * factor


@pytest.mark.parametrize("prec", [0, 2])
@pytest.mark.parametrize("qs,ks,vs", [(4e5, 1e-5, 1.0), (1e8, 1e-8, 1.0), (1e12, 1e-12, 1.0), (1e-12, 1e12, 1.0),
                                      (1e-30, 1e30, 1e-30), (1.0, 1.0, 1e30)])
@pytest.mark.parametrize("B,Nkv", [(1, 700), (20, 200)])
def test_attention_split_magnitudes_that_cancel(qs, ks, vs, B, Nkv, prec):
    """Large queries with small keys and the reverse: scores of order 1."""
    case(f"split attention scales {qs} {ks} {vs} B={B} precision {prec}")
    q, k, v = rnd(B, 200, 768, scale=qs), rnd(B, Nkv, 768, scale=ks), rnd(B, Nkv, 768, scale=vs)
    check_attention(q, k, v, prec=prec)


@pytest.mark.parametrize("loud", [30.0, 1e6, 1e12])
@pytest.mark.parametrize("B,Nkv", [(1, 700), (20, 200)])
def test_attention_split_loud_values(loud, B, Nkv):
    """Loud values beside small ones that are all the result: a head dimension of Q
    that meets zeros in K (and the reverse), one dimension of V, one key of V
    without probability."""
    case(f"split attention loud {loud} B={B}")
    q, k, v = rnd(B, 200, 768), rnd(B, Nkv, 768), rnd(B, Nkv, 768)
    for t, z in ((q, k), (k, q)):
        a, b = t.copy(), z.copy()
        a[..., 9::64], b[..., 9::64] = loud, 0.0
        check_attention(*((a, b, v) if t is q else (b, a, v)))
    small = v / np.float32(loud)
    small[..., 5::64] = rnd(B, Nkv, 12)  # the other dimensions are small beside it
    check_attention(q, k, small)
    small = v / np.float32(loud)
    small[:, 33] *= np.float32(loud)
    k2, q2 = k.copy(), q.copy()
    q2[..., 2::64] = 40.0
    k2[..., 2::64] = 0.0
    k2[:, 33, 2::64] = -60.0  # a score of -300: its large V does not count
    check_attention(q2, k2, small, 4.0)


@pytest.mark.parametrize("B,Nkv", [(1, 700), (20, 200)])
def test_attention_split_zero_dimensions(B, Nkv):
    """Heads narrower than 64, padded with zeros, and a head of zeros."""
    case(f"split attention zero dimensions B={B}")
    q, k, v = rnd(B, 200, 768), rnd(B, Nkv, 768), rnd(B, Nkv, 768)
    for t in (q, k, v):
        t.reshape(B, -1, 12, 64)[..., 40:] = 0.0
    v[..., 64:128] = 0.0
    check_attention(q, k, v)
    got = attention(q, k, v).reshape(B, 200, 12, 64)
    assert not got[..., 40:].any() and not got[:, :, 1].any()


@pytest.mark.parametrize("below", [10, 17, 24, 30, 40, 60])
@pytest.mark.parametrize("B,Nkv", [(1, 700), (20, 200)])
def test_attention_split_sink(below, B, Nkv):
    """One key takes nearly all weight and has a V of zeros: the result is that of
    the others, 2^-below of its weight each."""
    case(f"split attention sink 2^-{below} B={B}")
    q, k, v = rnd(B, 200, 768, scale=0.3), rnd(B, Nkv, 768, scale=0.3), rnd(B, Nkv, 768)
    q[..., 2::64], k[..., 2::64] = 4.0, 0.0
    k[:, Nkv // 2, 2::64] = below * np.log(2) * 8 / 4.0
    v[:, Nkv // 2] = 0.0
    check_attention(q, k, v, 4.0)


@pytest.mark.parametrize("B,Nkv", [(1, 700), (20, 200)])
def test_attention_split_infinities_and_nan(B, Nkv):
    """A head whose V, K or Q holds an infinity or NaN: the other heads are
    untouched, in that head infinities of V reach every query and a score of
    -inf drops its key."""
    case(f"split attention non-finite B={B}")
    q, k, v = np.abs(rnd(B, 200, 768)), rnd(B, Nkv, 768), rnd(B, Nkv, 768)
    base = attention(q, k, v)
    k2, v2 = k.copy(), v.copy()
    v2[0, 40, 3] = np.inf          # head 0, dim 3
    v2[0, 41, 64 * 2 + 5] = np.nan  # head 2, dim 5
    k2[0, 7, 64 * 4:64 * 5] = -np.inf  # head 4: scores of -inf
    got = attention(q, k2, v2)
    clean = np.ones(768, bool)
    for hd in (0, 2, 4):
        clean[64 * hd:64 * hd + 64] = False
    np.testing.assert_array_equal(got[:, :, clean], base[:, :, clean])
    assert (got[0, :, 3] == np.inf).all() and np.isnan(got[0, :, 133]).all()
    keep = np.arange(Nkv) != 7
    ref, bound = attention64(q[:1], k[:1, keep], v[:1, keep])
    h4 = slice(256, 320)
    assert (np.abs(got[:1, :, h4] - ref[:, :, h4]) <= bound[:, :, h4]).all()
    for hd in (0, 2):
        fin = np.isfinite(got[0, :, 64 * hd:64 * hd + 64])
        assert fin.sum() == 200 * 63
