"""Targets at a multiple of the logit resolution: per-cell label counts, their
64-cell blocks and the contraction on them, against the float64 oracle.

The label maps mix one-label cells with cells of random pixels, hold labels
outside the GT range, and start on an address that is only 8-byte aligned in
some cases; sizes sit on both sides of a block (64 cells), of a workgroup (256
cells) and of the rows that the preparation keeps in LDS at once (160 of u8,
80 of u16).  Tolerances are those of test_gpu_parity.py.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import mask_oracle as O  # noqa: E402
from test_gpu_parity import RTOL, close, rounded  # noqa: E402
from test_gpu_surface import close as close_extra, dice_grad_cancellation  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ml():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import mask_loss_amd
    return mask_loss_amd.mask_loss


def label_map(rng, B, H, W, s, G, noise):
    t = np.repeat(np.repeat(rng.integers(0, G + 1, size=(B, H, W)), s, 1), s, 2)
    mixed = rng.random(t.shape) < noise
    t[mixed] = rng.integers(-1, G + 4, size=int(mixed.sum()))
    return t


def on_gpu(t, shifted):
    """A contiguous device tensor, at an odd multiple of 8 bytes if `shifted`."""
    buf = torch.empty(t.size + 1, dtype=torch.int64, device="cuda")
    v = buf[1 if shifted else 0:][:t.size].view(t.shape)
    v.copy_(torch.from_numpy(t))
    assert v.is_contiguous() and (v.data_ptr() % 16 == 8) == shifted
    return v


# (s, H, W, G, bg, shifted)
SHAPES = [
    (2, 7, 9, 5, 0, False), (2, 8, 8, 5, -1, True), (2, 16, 17, 180, 0, False), (3, 5, 13, 30, 2, True),
    (4, 16, 16, 12, 0, False), (4, 13, 20, 31, 0, True), (4, 8, 33, 32, 400, False), (4, 16, 24, 100, 3, False),
    (5, 9, 8, 161, 0, False), (15, 4, 17, 3, 0, True), (16, 4, 20, 90, 0, False),
]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda v: "s%d_%dx%d_G%d_bg%d_%d" % v)
def test_costs(ml, shape, dtype):
    s, H, W, G, bg, shifted = shape
    rng = np.random.default_rng(s * 1000 + H * W)
    L, B, Q, C = 2, 2, 37, 6
    t = label_map(rng, B, H, W, s, G, 0.3)
    t[1, :s] = 1  # one whole cell row of one label
    zt, z64 = rounded(rng.normal(0, 2.0, size=(L, B, Q, H, W)), dtype)
    zc = rng.normal(size=(L, B, Q, C)).astype(np.float32)
    ct = rng.integers(0, C, size=(B, G + 1))
    got = ml.pairwise_mask_loss_forward(zt.cuda(), on_gpu(t, shifted), torch.from_numpy(zc).cuda(),
                                        torch.from_numpy(ct).cuda(), 1.0, 1.0, 1.0, 1.0, bg, 1.0, 0.05, 0.0, -1.0,
                                        0.0, -1.0, True, True).cpu().numpy()
    ref = O.pairwise_mask_loss_forward(z64, t, zc.astype(np.float64), ct, background_index=bg, use_softmax=True)
    for k in range(2):
        close(got[k], ref[k], RTOL[dtype], 1e-2)


@pytest.mark.parametrize("saved", [True, False])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("shape", [(2, 16, 17, 18, 0, True), (4, 13, 20, 24, 0, False), (16, 4, 20, 9, 0, False)],
                         ids=lambda v: "s%d_%dx%d_G%d_bg%d_%d" % v)
def test_backward(ml, shape, dtype, saved):
    """The mask-logit gradient with the counts of the forward's saved state and
    with counts made again."""
    s, H, W, G, bg, shifted = shape
    rng = np.random.default_rng(s + H)
    L, B, Q, C = 2, 2, 30, 6
    t = label_map(rng, B, H, W, s, G, 0.3)
    zt, z64 = rounded(rng.normal(0, 2.0, size=(L, B, Q, H, W)), dtype)
    zc = rng.normal(size=(L, B, Q, C + 1)).astype(np.float32)
    ct = rng.integers(0, C, size=(B, G + 1))
    z, tt, zct, ctt = zt.cuda(), on_gpu(t, shifted), torch.from_numpy(zc).cuda(), torch.from_numpy(ct).cuda()
    head = (z, tt, zct, ctt, 1.0, 1.0, 1.0, 1.0, bg, 1.0, 0.05)
    tail = (0.0, -1.0, 0.0, -1.0, C, True, True)
    p2g, _, _, _, _, state = ml.mask_matching_fused(*head, 1e30, -1.0, True, False, 1, 0, *tail)[:6]
    one = torch.ones(L, device="cuda")
    args = (one, one, one, *head[:4], p2g, *head[4:], -1.0, True, False, *tail)
    gm, _ = ml.mask_matching_backward_fused(*args, state) if saved else ml.mask_matching_backward(*args)
    ref, _ = O.matching_backward(np.ones(L), np.ones(L), np.ones(L), z64, t, zc.astype(np.float64), ct,
                                 p2g.cpu().numpy(), background_index=bg, force_cls=True, void_class_index=C,
                                 use_softmax=True)
    close(gm.float().cpu().numpy(), ref, RTOL[dtype], 1e-2 * np.abs(ref).max())


@pytest.mark.parametrize("shape", [(2, 7, 9, 5, True), (4, 16, 17, 40, False), (4, 20, 16, 170, True), (17, 4, 6, 9, False)],
                         ids=lambda v: "s%d_%dx%d_C%d_%d" % v)
def test_dense(ml, shape):
    s, H, W, C, shifted = shape
    rng = np.random.default_rng(s * H)
    L, B = 2, 3
    t = label_map(rng, B, H, W, s, C - 1, 0.3)
    z = rng.normal(0, 2.0, size=(L, B, C, H, W)).astype(np.float32)
    zt, tt, z64 = torch.from_numpy(z).cuda(), on_gpu(t, shifted), z.astype(np.float64)
    nm = float(L * B * C)
    close(ml.forward_sigmoid_ce_loss(zt, tt, nm, 1.5, 2.0, 0.25).cpu().numpy(),
          O.sigmoid_ce_loss(z64, t, nm, 1.5, 2.0, 0.25), 1e-5, 1e-2)
    loss, I, P, T = ml.forward_dice_loss(zt, tt, 1.0, nm, 1.5)
    rl, rI, rP, rT = O.dice_loss(z64, t, 1.0, nm, 1.5)
    for a, b in ((loss, rl), (I, rI), (P, rP), (T, rT)):
        close(a.cpu().numpy(), b, 1e-5, 1e-2)
    go = torch.tensor([1.0, -0.5], device="cuda")
    ref = O.sigmoid_ce_backward(go.cpu().numpy(), z64, t, nm, 1.5, 2.0, 0.25)
    close(ml.backward_sigmoid_ce_loss(go, zt, tt, nm, 1.5, 2.0, 0.25).cpu().numpy(), ref, 1e-5,
          1e-2 * np.abs(ref).max())
    # the backward takes the forward's float32 sums; its numerator cancels for
    # partial counts (dice_grad_cancellation)
    sums = [v.cpu().numpy() for v in (I, P, T)]
    ref = O.dice_loss_backward(go.cpu().numpy(), z64, t, *sums, 1.0, nm, 1.5)
    close_extra(ml.backward_dice_loss(go, zt, tt, I, P, T, 1.0, nm, 1.5).cpu().numpy(), ref, 1e-5,
                1e-2 * np.abs(ref).max(), dice_grad_cancellation(go.cpu().numpy(), z64, t, *sums, 1.0, nm, 1.5))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("shape", [(2, 8, 8, 1, True), (3, 15, 17, 16, False), (4, 16, 20, 17, True),
                                   (4, 16, 16, 161, False), (15, 5, 13, 330, False), (15, 4, 4, 3, True)],
                         ids=lambda v: "s%d_%dx%d_C%d_%d" % v)
def test_dense_groups(ml, shape, dtype):
    """The kernels that count for themselves: 16 and 17 classes, two groups by
    LDS (161); the counts in memory below 16 classes and for 330 at s = 15."""
    s, H, W, C, shifted = shape
    rng = np.random.default_rng(s * H + C)
    L, B = 2, 2
    t = label_map(rng, B, H, W, s, C - 1, 0.3)
    zt, z64 = rounded(rng.normal(0, 2.0, size=(L, B, C, H, W)), dtype)
    zt, tt = zt.cuda(), on_gpu(t, shifted)
    nm, go = float(L * B * C), torch.tensor([1.0, -0.5], device="cuda")
    close(ml.forward_sigmoid_ce_loss(zt, tt, nm, 1.5, 2.0, 0.25).cpu().numpy(),
          O.sigmoid_ce_loss(z64, t, nm, 1.5, 2.0, 0.25), 1e-5, 1e-2)
    # half the spacing of float16 below 2^-14, where these gradients lie
    sub = 2.0 ** -25 if dtype == "float16" else 0.0
    ref = O.sigmoid_ce_backward(go.cpu().numpy(), z64, t, nm, 1.5, 2.0, 0.25)
    close_extra(ml.backward_sigmoid_ce_loss(go, zt, tt, nm, 1.5, 2.0, 0.25).float().cpu().numpy(), ref, RTOL[dtype],
                1e-2 * np.abs(ref).max(), sub)
    loss, I, P, T = ml.forward_dice_loss(zt, tt, 1.0, nm, 1.5)
    sums = [v.cpu().numpy() for v in (I, P, T)]
    ref = O.dice_loss_backward(go.cpu().numpy(), z64, t, *sums, 1.0, nm, 1.5)
    close_extra(ml.backward_dice_loss(go, zt, tt, I, P, T, 1.0, nm, 1.5).float().cpu().numpy(), ref, RTOL[dtype],
                1e-2 * np.abs(ref).max(), sub + dice_grad_cancellation(go.cpu().numpy(), z64, t, *sums, 1.0, nm, 1.5))


@pytest.mark.parametrize("shape", [(2, 40, 40, 300), (2, 24, 40, 300), (4, 24, 25, 500), (2, 64, 72, 2),
                                   (4, 128, 136, 20), (3, 40, 57, 60)], ids=lambda v: "s%d_%dx%d_L%d" % v)
def test_pair_groups(ml, shape):
    """The pair kernel on u8 counts with more 64-cell groups per wave than its two
    ring slots: with 4,096 waves resident the shapes give 7, 4, 3, 2, 6 and 3
    groups, the third and the last a tail that is no whole group.  Every layer
    holds the same logits, so one layer's oracle serves the waves of all.

    Each group has labels of its own, and the logits' size changes from group to
    group, so a group's logits or counts taken for another's show at once.  Planes
    of 11 bits and counts that are exact put each sum within 2^-12 of itself (all
    terms are non-negative), a quotient within 2^-11; the entry for |z| < 2^-9 and
    the float32 sums are far below the rest of the 2^-10 allowed."""
    s, H, W, L = shape
    rng = np.random.default_rng(s * 1000 + W)
    B, Q, C, G = 2, 37, 6, 24
    group = (np.arange(H * W) // 64).reshape(H, W)
    own = 1 + (5 * group + rng.integers(0, 2, size=(B, H, W))) % G
    t = np.repeat(np.repeat(own, s, 1), s, 2)
    mixed = rng.random(t.shape) < 0.2
    t[mixed] = rng.integers(-1, G + 2, size=int(mixed.sum()))
    size = 0.25 + (7 * group) % 11 * 0.5
    zt, z64 = rounded(rng.normal(size=(1, B, Q, H, W)) * size, "bfloat16")
    zc = rng.normal(size=(1, B, Q, C)).astype(np.float32)
    ct = rng.integers(0, C, size=(B, G + 1))
    zg, zcg = zt.cuda().expand(L, -1, -1, -1, -1).contiguous(), torch.from_numpy(zc).cuda().expand(L, -1, -1, -1).contiguous()
    got = ml.pairwise_mask_loss_forward(zg, on_gpu(t, False), zcg, torch.from_numpy(ct).cuda(), 1.0, 1.0, 1.0, 1.0, 0,
                                        1.0, 0.05, 0.0, -1.0, 0.0, -1.0, True, True)
    ref = O.pairwise_mask_loss_forward(z64, t, zc.astype(np.float64), ct, background_index=0, use_softmax=True)
    for k in range(2):
        want = torch.from_numpy(np.asarray(ref[k])).cuda().expand(L, -1, -1, -1)
        there = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got[k]), there)
        assert (got[k].double() - want)[there].abs().max().item() <= 2.0 ** -10 * max(1.0, want[there].abs().max().item())
