"""The candidate ranges of the pixel-driven and slant-stacking kernels, which are formed in
float32 with a margin for their rounding, checked by brute force up to 32766 pixels a side.

Pixel-driven forward (csrc/pd.hip, pd_fwd_bin): the rows of a bin (in double) and the columns
of each row (in float) have to hold every pixel with a sample that the kernel counts for the
bin.  Slant-stacking back projection (csrc/ss.hip, ss_back_kernel): the three bins from
ceil(tc - hw), the third only up to tc + hw, have to hold every bin whose line reaches the
pixel, and for a pixel two or more pixels inside the image each such bin's stepped range has
to hold the pixel's step (the kernel does not look at it there).

Samples and lines in float32 as the kernels compute them, in both arithmetic forms.
"""
import numpy as np
import pytest

f32, f64 = np.float32, np.float64
SIDES = [3, 64, 511, 4096, 16385, 32766]
DEG = [0.0, 0.001, 0.3, 7.0, 30.0, 44.99, 45.0, 45.01, 60.0, 89.5, 89.999, 90.0, 90.001, 91.0, 120.0, 135.0,
       150.3, 179.7, 179.999, 180.0]


def fma(a, b, c):
    return (a.astype(f64) * np.asarray(b, f64) + np.asarray(c, f64)).astype(f32)


def trig(theta, arith):
    if arith == "fast":
        return np.sin(f32(theta)), np.cos(f32(theta))
    return f32(np.sin(f64(theta))), f32(np.cos(f64(theta)))


# ---- pixel-driven ----------------------------------------------------------------------

def pd_hits(theta, s, c, arith, nh, x0, y0, e, method):
    """Whether pixel centres (x0, y0) have a sample that counts for bin e."""
    hit = np.zeros(np.broadcast(x0, y0).shape, bool)
    for d in (f32(-0.25), f32(0.25)):
        x, y = (x0 + d).astype(f32), (y0 + d).astype(f32)
        xs = (x * s).astype(f32)
        with np.errstate(divide="ignore", invalid="ignore"):
            if arith == "fast":
                t, q = np.abs(fma(y, -c, xs)), (xs * (f32(1) / c)).astype(f32)
            else:
                t, q = np.abs((xs - (y * c).astype(f32)).astype(f32)), (xs / c).astype(f32)
            keep = np.zeros(hit.shape, bool)
            if f64(theta) != np.pi / 2:
                keep |= y > q
        if theta == 0:
            keep |= np.broadcast_to(y > 0, hit.shape)
        t = np.where(keep, t, -t).astype(f32)
        if method == 0:
            v = nh - 0.5 - t.astype(f64)
            l = np.trunc(v + np.copysign(0.49999999999999994, v)) if arith == "fast" \
                else np.sign(v) * np.floor(np.abs(v) + 0.5)
            hit |= l == e
        else:
            t1 = (f32(nh) - t).astype(f32)
            hit |= np.minimum((f32(e + 1) - t1).astype(f32), (t1 - f32(e - 1)).astype(f32)) > 0
    return hit


@pytest.mark.parametrize("arith", ["fast", "ieee"])
@pytest.mark.parametrize("npix", SIDES)
def test_pixel_driven_ranges_hold_every_sample(npix, arith):
    nh = npix // 2
    rng = np.random.default_rng(npix)
    found = 0
    for deg in DEG:
        theta = f32(deg * np.pi / 180)
        s, c = trig(theta, arith)
        C, S = abs(f64(c)), (-f64(s) if c < 0 else f64(s))
        rs = 1.0 / S if S != 0 else 0.0
        dshift = 0.25 * abs(C - S)
        bins = np.unique(np.concatenate([[1, 2, npix - 1], rng.integers(1, max(2, npix), 6)]))
        for e in bins[bins < npix]:
            half = 1.0 + dshift + 0.01 + npix * 2.0 ** -18
            tl, th = nh - e - half, nh - e + half
            xa, xb = 0.5 - nh, npix - 1 - nh + 0.5
            i0, i1 = 0, npix - 1
            if C > 0:
                i0 = int(min(max(0.0, np.ceil((tl + min(xa * S, xb * S)) / C + nh - 0.5)), npix))
                i1 = int(max(-1.0, min(npix - 1.0, np.floor((th + max(xa * S, xb * S)) / C + nh - 0.5))))
            # rows just outside the range hold nothing
            col = ((np.arange(npix) - nh).astype(f32) + f32(0.5))
            for i in {i0 - 1, i0 - 3, i1 + 1, i1 + 3} & set(range(npix)):
                y0 = f32(i - nh) + f32(0.5)
                for m in (0, 1):
                    assert not pd_hits(theta, s, c, arith, nh, col, y0, e, m).any(), (deg, e, i)
            if i1 < i0 or rs == 0.0:
                continue
            i = np.unique(np.concatenate([[i0, i0 + 1, i1 - 1, i1], rng.integers(i0, i1 + 1, 40)]))
            i = i[(i >= i0) & (i <= i1)]
            y0 = ((i - nh).astype(f32) + f32(0.5))
            a = f32(C * rs)
            lo = f32((-th if rs > 0 else -tl) * rs + nh - 0.5)
            hi = f32((-tl if rs > 0 else -th) * rs + nh - 0.5)
            j0 = np.minimum(np.maximum(0, np.ceil(fma(y0, a, lo))), npix).astype(np.int64)
            j1 = np.maximum(-1, np.minimum(npix - 1, np.floor(fma(y0, a, hi)))).astype(np.int64)
            k = np.arange(1, 9)
            j = np.concatenate([j0[:, None] - k, j1[:, None] + k], 1)       # just outside
            x0 = ((j - nh).astype(f32) + f32(0.5))
            ok = (j >= 0) & (j < npix)
            inside = np.clip((j0 + j1) // 2, 0, npix - 1)
            for m in (0, 1):
                out = pd_hits(theta, s, c, arith, nh, x0, y0[:, None], e, m) & ok
                assert not out.any(), (deg, e, m, i[out.any(1)])
                found += pd_hits(theta, s, c, arith, nh, (inside - nh).astype(f32) + f32(0.5), y0, e, m).sum()
    assert found > 50 or npix < 10


# ---- slant-stacking --------------------------------------------------------------------

def ss_round(v, arith):
    if arith == "fast":
        return np.trunc((v + np.copysign(f32(0.49999997), v)).astype(f32)).astype(np.int64)
    v = v.astype(f64)
    return (np.sign(v) * np.floor(np.abs(v) + 0.5)).astype(np.int64)


def ss_ranges(s, c, ybranch, arith, npix):
    """Stepped range of every bin (plan.hip, ss_view_ranges)."""
    nh = npix // 2
    tf = (np.arange(npix) - nh).astype(f32)
    one = np.ones(npix, f32)
    mnh, nh1 = f32(-nh), f32(nh - 1)

    def middle(p, q):
        mn, mx = np.minimum(p, q), np.maximum(p, q)
        m1, m2 = np.maximum(mn, mnh), np.minimum(mx, nh1)
        return np.minimum(m1, m2), np.maximum(m1, m2)

    if abs(f64(s)) < 1e-5:
        lim = [0 * one, 0 * one, mnh * one, nh1 * one]
    elif abs(f64(c)) < 1e-5:
        lim = [mnh * one, nh1 * one, 0 * one, 0 * one]
    else:
        if arith == "fast":
            nhv, nhm = f32(nh) * one, nh1 * one
            x1, x2 = (fma(nhv, s, tf) / c).astype(f32), (fma(nhm, -s, tf) / c).astype(f32)
            y1, y2 = (fma(nhv, c, tf) / s).astype(f32), (fma(nhm, -c, tf) / s).astype(f32)
        else:
            def q(v, d):
                return (v / d).astype(f32)
            x1 = (q(tf, c) + q(f32(nh) * s * one, c)).astype(f32)
            x2 = (q(tf, c) - q(nh1 * s * one, c)).astype(f32)
            y1 = (q(tf, s) + q(f32(nh) * c * one, s)).astype(f32)
            y2 = (q(tf, s) - q(nh1 * c * one, s)).astype(f32)
        lim = list(middle(x1, x2)) + list(middle(y1, y2))
    u0 = np.maximum(ss_round(lim[2] if ybranch else lim[0], arith), -nh)
    u1 = np.minimum(ss_round(lim[3] if ybranch else lim[1], arith), npix - nh)
    u1 = np.maximum(u0, u1)
    none = np.arange(npix) >= 2 * nh
    return np.where(none, 0, u0), np.where(none, 0, u1)


@pytest.mark.parametrize("arith", ["fast", "ieee"])
@pytest.mark.parametrize("npix", SIDES)
def test_slant_stacking_bins_hold_every_line(npix, arith):
    nh = npix // 2
    rng = np.random.default_rng(npix)
    margin = f32(f32(0.01) + f32(npix * 2.0 ** -18))
    found = 0
    for deg in DEG + [44.9999, 45.0001, 134.9999]:
        s, c = trig(f32(deg * np.pi / 180), arith)
        ybranch = not (0.70710678118654757 < abs(f64(s)))
        a, b = (s, c) if ybranch else (c, s)
        edge = np.array([-nh, 1 - nh, 2 - nh, 3 - nh, 0, nh - 5, nh - 4, nh - 3, nh - 1])
        u = np.concatenate([np.repeat(edge, edge.size), rng.integers(-nh, npix - nh, 4000)])
        P = np.concatenate([np.tile(edge, edge.size), rng.integers(-nh, npix - nh, 4000)])
        on = (u >= -nh) & (u < npix - nh) & (P >= -nh) & (P < npix - nh)
        u, P = u[on], P[on]
        uf = u.astype(f32)
        tc = fma(uf, a, (P.astype(f32) * b).astype(f32))
        hw = fma(np.abs(b) * np.ones(1, f32), f32(1) + margin, margin)
        tf = np.ceil((tc - hw).astype(f32))
        third = (tf + 2).astype(f32) <= (tc + hw).astype(f32)
        u0, u1 = ss_ranges(s, c, ybranch, arith, npix)
        inner = (u + nh >= 2) & (P + nh >= 2) & (u + nh < 2 * nh - 3) & (P + nh < 2 * nh - 3)
        for k in range(-4, 8):
            t = (tf + k).astype(f32)
            with np.errstate(over="ignore"):
                if arith == "fast":
                    q = (fma(uf, -a, t) * (f32(1) / b)).astype(f32)
                else:
                    q = ((t / b).astype(f32) - ((uf * a).astype(f32) / b).astype(f32)).astype(f32)
            fl = np.floor(q).astype(np.int64)
            hit = (fl == P) | (fl + 1 == P) | (ss_round(q, arith) == P)
            hit &= (t >= -nh) & (t < nh)
            taken = (k in (0, 1)) | ((k == 2) & third)
            assert not (hit & ~taken).any(), (deg, k, u[hit & ~taken], P[hit & ~taken])
            bin_ = np.clip(t.astype(np.int64) + nh, 0, npix - 1)
            within = (u >= u0[bin_]) & (u < u1[bin_])
            wrong = hit & inner & ~within
            assert not wrong.any(), (deg, k, u[wrong], P[wrong])
            found += int((hit & inner).sum())
    assert found > 1000 or npix < 10
