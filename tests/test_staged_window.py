"""The index bounds of the distance-driven forward's two paths, checked by brute force.

Staged (csrc/dd_device.h, fwd_staged): for a block of B bins and views with at most NC
candidate pixels per bin and line (bins narrower than NC - 1.25 pixels) the kernel copies
W = (NC-1) B pixels of each line into LDS, starting at q0 = floor(fl(D0lo + K)) + nh - 2,
clamped to [-((W-NC) & ~3), npix-1] and rounded down to a multiple of 4.  Every bin reads its
NC candidates from its first pixel x (the one-test search, clamped into the line), with no
clamp of its own: on every line of every chunk, also where the bin misses the line and on the
lines past the block's last one that fill the last chunk, x + nh - q0 has to lie in
[0, W - NC].

Diagonal (fwd_diag): lane d takes the lines L(d) .. L(d) + steps - 1.  Every line that its bin
meets has to be among them, L has to be monotonic in the bin (the wave's extremes come from its
first and last lane), and NC candidates from the first pixel have to reach the bin's end.

All keys in float32 as the kernels compute them, in both arithmetic forms.
"""
import numpy as np
import pytest

f32 = np.float32


def view(w, sign, arith):
    """Constants of a view with bins w pixels wide (column sweep for sign > 0): the functions
    D(j), K(u) and rinv, t."""
    b = f32(1.0 / w)
    a = f32(sign * np.sqrt(1.0 - 1.0 / w ** 2))
    rinv = f32(1) / b
    t = f32(a * rinv)
    if arith == "fast":
        return lambda j: (f32(j) * rinv).astype(f32), lambda u: (f32(u) * t).astype(f32), rinv, t
    return (lambda j: (f32(j) / b).astype(f32), lambda u: ((f32(u) * a).astype(f32) / b).astype(f32),
            rinv, t)


def first_pixel(Dlo, K, nh, npix, near):
    """(unclamped, clamped) index - nh of the pixel that holds Dlo on a line with offset K."""
    if near:
        fe = np.floor(((Dlo + f32(0.5)).astype(f32) + K).astype(f32))
        fe = np.where(Dlo < (fe - K).astype(f32), fe - 1, fe)
    else:
        fe = np.floor((Dlo + K).astype(f32))
        e1 = fe + 1
        fe = np.where(Dlo >= (e1 - K).astype(f32), e1, np.where(Dlo < (fe - K).astype(f32), fe - 1, fe))
    return np.clip(fe, -nh, npix - 1 - nh).astype(np.int64)


def block_lines(npix, nh, D0lo, D1hi, t):
    """The block's first and last line, as the kernel bounds them in double."""
    rt = 1.0 / float(t)
    ua, ub = sorted(((-nh - float(D1hi)) * rt, (npix - nh - float(D0lo)) * rt))
    ua, ub = (min(max(v + nh - 0.5, -4.0), npix + 4.0) for v in (ua, ub))
    return max(0, int(np.floor(ua)) - 2), min(npix - 1, int(np.ceil(ub)) + 2)


def window_violations(npix, w, sign, b, nc, width, arith, blocks=None, lines=None):
    nh = npix // 2
    D, Kf, _, t = view(w, sign, arith)
    fl = min(16 * b // width, 8)
    bad = seen = 0
    for d0 in range(0, npix, b) if blocks is None else blocks:
        d1 = min(d0 + b - 1, npix - 1)
        i_lo, i_hi = block_lines(npix, nh, D(d0 - nh), D(d1 + 1 - nh), t)
        if i_hi < i_lo:
            continue
        i = np.arange(i_lo, i_lo + -(-(i_hi - i_lo + 1) // fl) * fl)   # whole chunks
        if lines:
            i = np.unique(np.concatenate([i[:40], i[-40:], i[::max(1, i.size // lines)]]))
        K = Kf((i - nh).astype(f32) + f32(0.5))[:, None]
        q = np.floor((D(d0 - nh) + K).astype(f32)).astype(np.int64) + nh - 2
        q0 = np.minimum(np.maximum(q, -((width - nc) & ~3)), npix - 1) & ~3
        off = first_pixel(D(np.arange(d0, d1 + 1) - nh)[None, :], K, nh, npix, True) + nh - q0
        bad += int(np.count_nonzero((off < 0) | (off > width - nc)))
        seen += off.size
    assert seen
    return bad


# bins at the bottom and just below the top of each staged bracket
STAGED = [(1.0005, 3), (1.3, 3), (1.74, 3), (1.76, 4), (2.74, 4), (2.76, 6), (3.74, 6), (4.74, 6)]


@pytest.mark.parametrize("arith", ["fast", "ieee"])
@pytest.mark.parametrize("b", [64, 128, 256])
@pytest.mark.parametrize("w,nc", STAGED)
def test_window_holds_every_candidate_of_every_line(w, nc, b, arith):
    assert int(np.floor(w + 0.25)) + 2 <= nc and 16 * b // ((nc - 1) * b) >= 1
    for sign in (1, -1):
        for npix in (1, 2, 5, 63, 65, 130, 601, 1024):
            assert window_violations(npix, w, sign, b, nc, (nc - 1) * b, arith) == 0, (npix, sign)
        for npix in (2048, 8191, 32766):
            blocks = sorted({k * b for k in (0, 1, 2, 5, npix // b // 3, npix // b // 2,
                                             npix // b - 2, npix // b - 1, (npix - 1) // b)})
            assert window_violations(npix, w, sign, b, nc, (nc - 1) * b, arith, blocks, 200) == 0, \
                (npix, sign)


def test_a_narrower_window_overflows():
    for w, nc in [(1.74, 3), (2.74, 4), (4.74, 6)]:
        assert window_violations(1024, w, 1, 64, nc, (nc - 1) * 64 - 12, "fast") > 0, (w, nc)


WIDE = [1.76, 2.76, 3.8, 4.76, 6.7, 7.74, 9.7, 11.74, 14.74, 18.7, 22.74, 30.74, 31.0, 57.3, 400.0, 5729.6,
        1e6]


@pytest.mark.parametrize("arith", ["fast", "ieee"])
@pytest.mark.parametrize("w", WIDE)
def test_diagonals_take_every_line_of_every_bin(w, arith):
    nc = int(np.floor(w + 0.25)) + 2
    nc = nc if nc <= 32 else (nc + 3) // 4 * 4      # plan.hip, dd_candidates
    for sign in (1, -1):
        for npix in (1, 2, 17, 64, 65, 363, 1024, 8191, 32766):
            nh = npix // 2
            D, Kf, rinv, t = view(w, sign, arith)
            d = np.arange(npix)
            if npix > 400:
                d = np.unique(np.concatenate([d[:70], d[-70:], d[::npix // 60]]))
            rt = 1.0 / float(t)
            e0 = (-nh - D(d + 1 - nh).astype(np.float64)) * rt
            e1 = (npix - nh - D(d - nh).astype(np.float64)) * rt
            L = np.floor(np.minimum(e0, e1) + (nh - 0.5625)).astype(np.int64) + 1
            steps = int(np.floor((npix + float(rinv)) * abs(rt) + 0.14)) + 1
            assert (np.diff(L) * np.sign(np.diff(L).sum() or 1) >= 0).all()
            i = np.arange(npix)
            K = Kf((i - nh).astype(f32) + f32(0.5))[None, :]
            Dlo, Dhi = D(d - nh)[:, None], D(d + 1 - nh)[:, None]
            lo, hi = (f32(-nh) - K).astype(f32), (f32(npix - nh) - K).astype(f32)
            meets = (Dhi > lo) & (Dlo < hi)
            taken = (i[None, :] >= L[:, None]) & (i[None, :] < L[:, None] + steps)
            assert not (meets & ~taken).any(), (npix, sign)
            assert meets.any() or npix == 1
            x = first_pixel(Dlo, K, nh, npix, nc <= 32)
            short = meets & (x + nc < npix - nh) & ((f32(1) * (x + nc) - K).astype(f32) < Dhi) & (Dlo > lo)
            assert not short.any(), (npix, sign)
