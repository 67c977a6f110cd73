"""The cost contraction's operand forms at their edges, against the float64 oracle.

Planes beyond float16 (|z| > 127, or > 2558 at the smallest weight) make a wave redo
its range with bf16 operands; rows of odd sizes start off 16-byte (and 4-byte)
boundaries; label codes use the whole byte (256 GT slots); counts above 2047
(s >= 46) split into two float16 parts; the wide classes (32 and more, 112 and
more non-empty GTs) sum per slot.  Tolerances are those of test_gpu_parity.py.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import mask_oracle as O  # noqa: E402
from test_gpu_parity import RTOL, close, rounded  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ml():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import mask_loss_amd
    return mask_loss_amd.mask_loss


def check(ml, dtype, s, H, W, labels, bg, big=(), Q=21, ug=1.0, gamma=0.0, alpha=-1.0, seed=0):
    """labels: the GT slots that occur (others stay empty); big: logits put
    into a few cells of some rows."""
    rng = np.random.default_rng(seed)
    B, C, GT = 2, 5, max(labels) + 1
    t = rng.choice(np.asarray(labels), size=(B, H * s, W * s))
    z = rng.normal(0, 2.0, size=(1, B, Q, H, W)).astype(np.float32)
    for q in range(0, Q, 4):
        for v in big:
            z[0, :, q, rng.integers(H), rng.integers(W)] = v
    zt, z64 = rounded(z, dtype)
    zc = rng.normal(size=(1, B, Q, C)).astype(np.float32)
    ct = rng.integers(0, C, size=(B, GT))
    got = ml.pairwise_mask_loss_forward(zt.cuda(), torch.from_numpy(t).cuda(), torch.from_numpy(zc).cuda(),
                                        torch.from_numpy(ct).cuda(), 1.0, 1.0, 1.0, 1.0, bg, ug, 0.05, gamma, alpha,
                                        0.0, -1.0, True, True).cpu().numpy()
    ref = O.pairwise_mask_loss_forward(z64, t, zc.astype(np.float64), ct, background_index=bg, ug=ug,
                                       mask_gamma=gamma, mask_alpha=alpha, use_softmax=True)
    for k in range(2):
        close(got[k], ref[k], RTOL[dtype], 1e-2)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("s", [1, 2])
@pytest.mark.parametrize("G", [9, 40, 130])
@pytest.mark.parametrize("size", [(16, 16), (13, 15), (9, 10)], ids=lambda v: "%dx%d" % v)
def test_sizes_and_classes(ml, dtype, s, G, size):
    check(ml, dtype, s, *size, range(G + 1), 0)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("G", [9, 40])
@pytest.mark.parametrize("s", [1, 4])
@pytest.mark.parametrize("big", [(126.0, -126.0), (200.0, -130.0), (-2600.0, 3000.0), (6.0e4, -5.0e4)],
                         ids=lambda v: "%g" % v[0])
@pytest.mark.parametrize("ug", [0.0, 1.0])
def test_planes_beyond_float16(ml, dtype, G, s, big, ug):
    check(ml, dtype, s, 16, 17, range(G + 1), 0, big=big, ug=ug)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("labels,bg", [(range(256), 7), (range(256), 255), (range(1, 255), 400), ((0, 3, 255), 1),
                                       ((0, 3, 254), -1)], ids=["256_bg7", "256_bg255", "255_nobg", "few_255", "few_254"])
def test_label_codes(ml, dtype, labels, bg):
    check(ml, dtype, 1, 24, 24, labels, bg, Q=17)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("s,G", [(45, 3), (46, 3), (64, 40), (255, 2)])
def test_large_counts(ml, dtype, s, G):
    check(ml, dtype, s, 3, 5, range(G + 1), 0)


@pytest.mark.parametrize("gamma,alpha,ug", [(0.0, -1.0, 0.0), (2.0, 0.25, 0.0), (2.0, 0.25, 1.0), (2.0, -1.0, 2.0),
                                            (1.0, 0.6, 1.0), (0.0, 0.3, 1.0)])
def test_formula_modes(ml, gamma, alpha, ug):
    check(ml, "float32", 1, 16, 20, range(12), 0, ug=ug, gamma=gamma, alpha=alpha)
