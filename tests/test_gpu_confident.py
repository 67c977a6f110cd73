"""Mask costs of confident logits: planes that get small, or large, beside what
float16 operands hold (the contraction takes bf16 ones there).

The predictions match the label map's shapes, so that a query's own cost is as
small as its logits allow and nothing hides a lost plane.  Each plane's value in
float64 gets an interval from the float32 formulas' own error, which is not
relative: log2(1 + e^-|z|) rounds 1 + e^-|z| to 2^-24 of 1.  With u = 2^-22 (|z| + 4),
the relative error of e^-|z| by a float32 exponent (each of the few operations
after it adds 2^-24 more):

    p, q: u;   softplus(+-z): u times it + 2^-23;   H, p^gamma: from these;

and a plane as an operand keeps 20, 14 or 8 bits (float32, float16, bf16: at least
two fewer than its terms hold, for the sums), or is 2^-34 off where float16 operands
are taken.  Sums and costs of the interval ends bound the result.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_parity import rounded  # noqa: E402

pytestmark = pytest.mark.gpu
BITS = {"float32": 20, "float16": 14, "bfloat16": 8}


@pytest.fixture(scope="module")
def ml():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import mask_loss_amd
    return mask_loss_amd.mask_loss


def planes(z, dtype, ug, ugm, gamma, alpha):
    """(neg, pos, wp, w) of float64 logits, each as its interval's two ends."""
    az = np.abs(z)
    e = np.exp(-az)
    u = 2.0 ** -22 * (az + 4.0)
    p, q = np.where(z >= 0, 1.0, e) / (1.0 + e), np.where(z >= 0, e, 1.0) / (1.0 + e)
    cn, cp = np.log1p(e) + np.maximum(z, 0.0), np.log1p(e) + np.maximum(-z, 0.0)
    an, ap = (1.0, 1.0) if alpha < 0 else (1.0 - alpha, alpha)
    ends = []
    for sg in (-1.0, 1.0):
        r = 1.0 + sg * u
        P, Q = p * r, q * r
        N, O = np.maximum(cn * r + sg * 2.0 ** -23, 0.0), np.maximum(cp * r + sg * 2.0 ** -23, 0.0)
        w = np.ones_like(z)
        if ug:
            w = np.clip(((P * O + Q * N) / np.log(2.0)) ** ug * (1.0 + sg * 2.0 ** -18 * ug), ugm, 1.0)
        ends.append([w * an * P ** gamma * N, w * ap * Q ** gamma * O, w * P, w])
    wide = gamma != 0 or (ug != 0 and ugm < 2.0 ** -6)
    b, a = 2.0 ** -BITS[dtype], 0.0 if wide else 2.0 ** -34
    return [(np.maximum(x * (1 - b) - a, 0.0), y * (1 + b) + a) for x, y in zip(*ends)]


def case(dtype, s, H, W, G, m, spread, seed, Q=20, B=2):
    """Label blocks of 1..G (0: background), and queries 0.. that predict one
    label each with logits of magnitude about m, others that predict none."""
    rng = np.random.default_rng(seed)
    t = np.repeat(np.repeat(rng.integers(0, G + 1, size=(B, -(-H // 4), -(-W // 4))), 4, 1), 4, 2)[:, :H, :W]
    t = np.ascontiguousarray(np.repeat(np.repeat(t, s, 1), s, 2))
    low = t[:, ::s, ::s]
    want = (np.arange(Q) % (G + 1))[None, :, None, None]  # query 0 predicts background
    mag = np.maximum(m + spread * rng.normal(size=(B, Q, H, W)), 0.25 * m)
    z = np.where((low[:, None] == want) & (want > 0), mag, -mag)[None]
    return (t, *rounded(z, dtype))


def check(ml, dtype, s, H, W, G, m, spread, ug, ugm, gamma, alpha, smooth=1.0, force=None, seed=0):
    t, zt, z = case(dtype, s, H, W, G, m, spread, seed)
    if force is not None:
        zt[..., : H // 3, :] = force
        z = zt.double().numpy()
    L, B, Q = z.shape[:3]
    zc, ct = torch.zeros(L, B, Q, 3, device="cuda"), torch.zeros(B, G + 1, dtype=torch.long, device="cuda")
    got = ml.pairwise_mask_loss_forward(zt.cuda(), torch.from_numpy(t).cuda(), zc, ct, smooth, 1.0, 1.0, 1.0, 0, ug, ugm,
                                        gamma, alpha, 0.0, -1.0, True, True).cpu().numpy()
    N2 = s * s
    neg, pos, wp, w = planes(z.reshape(L, B, Q, -1), dtype, ug, ugm, gamma, alpha)
    cells = t.reshape(B, H, s, W, s).transpose(0, 1, 3, 2, 4).reshape(B, H * W, N2)
    n = np.stack([(cells == g).sum(2) for g in range(1, G + 1)], 2).astype(np.float64)  # (B, cells, G)
    sides = []
    for k, o in ((0, 1), (1, 0)):
        num = np.einsum("lbqc,bcg->lbqg", neg[k], N2 - n) + np.einsum("lbqc,bcg->lbqg", pos[k], n)
        S = np.maximum(N2 * w[o].sum(3), 1e-12)[..., None]
        I = np.einsum("lbqc,bcg->lbqg", wp[k], n)
        P, T = N2 * wp[o].sum(3)[..., None], np.einsum("lbqc,bcg->lbqg", w[o], n)
        sides.append((num / S, 1.0 - (2.0 * I + smooth) / (P + T + smooth), S))
    r = 1.0 + 2.0 ** -20  # the sums' and the quotients' float32
    there = np.broadcast_to((n.sum(1) > 0)[None, :, None], got[0].shape)
    held = sides[1][0] * sides[0][2] < 1e38  # (a sum beyond float32 may leave the costs non-finite)
    assert np.array_equal(np.isfinite(got[0])[held], there[held])
    there = there & held
    lo, hi, x = sides[0][0][there] / r, sides[1][0][there] * r, got[0][there]
    assert (x >= lo).all() and (x <= hi).all(), (x[x < lo], lo[x < lo], x[x > hi], hi[x > hi])
    lo, hi, x = sides[1][1][there] - 2.0 ** -21, sides[0][1][there] + 2.0 ** -21, got[1][there]
    assert (x >= lo).all() and (x <= hi).all(), (x[x < lo], lo[x < lo], x[x > hi], hi[x > hi])


FOCAL = [(1.0, 0.05, 2.0, -1.0), (0.0, 0.05, 2.0, 0.25), (0.0, 0.05, 1.0, -1.0), (1.0, 0.05, 3.5, 0.25)]
FLOOR = [(1.0, 0.0, 0.0, -1.0), (2.0, 0.0, 0.0, -1.0), (3.0, 1e-4, 0.0, -1.0), (1.0, 1e-4, 2.0, 0.25)]
PLAIN = [(1.0, 0.05, 0.0, -1.0), (0.0, 0.05, 0.0, -1.0), (1.0, 0.05, 0.0, 0.25), (2.0, 0.5, 0.0, -1.0),
         (0.5, 0.1, 0.0, 0.6)]
MODES = pytest.mark.parametrize("mode", FOCAL + FLOOR + PLAIN, ids=lambda v: "ug%g_min%g_gamma%g_alpha%g" % v)


DTYPES = pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])


@DTYPES
@pytest.mark.parametrize("s,G", [(1, 6), (1, 40), (2, 6), (4, 40)])
@MODES
def test_small_planes(ml, dtype, s, G, mode):
    for m, spread in ((6.0, 1.0), (8.0, 0.1), (13.0, 1.0), (20.0, 2.0), (30.0, 0.0)):
        check(ml, dtype, s, 16, 24, G, m, spread, *mode)


@DTYPES
@pytest.mark.parametrize("s,G,H,W", [(1, 3, 13, 15), (16, 3, 9, 8), (17, 40, 8, 12), (1, 130, 60, 64)])
def test_small_planes_sizes(ml, dtype, s, G, H, W):
    for mode in (FOCAL[0], FLOOR[1], PLAIN[0], PLAIN[1]):
        check(ml, dtype, s, H, W, G, 9.0, 1.0, *mode)


@DTYPES
@pytest.mark.parametrize("s,G", [(1, 6), (1, 40), (4, 6), (4, 40), (16, 6)])
def test_filled_rows(ml, dtype, s, G):
    """A third of the map at one large logit (the lowest value of the type at
    the end): the other cells' sums are as exact as without it."""
    for fill in (-20.0, -70.0, -500.0, -6e4, float(torch.finfo(getattr(torch, dtype)).min)):
        check(ml, dtype, s, 24, 64, G, 3.0, 1.0, 1.0, 0.05, 0.0, -1.0, force=fill)
