"""Forms of the matching step beside those of test_gpu_parity.py: upstream
gradients at other strides, and the strategies with more columns than lanes."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import assign as OA  # noqa: E402
from oracle import points_oracle as PO  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ml():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import mask_loss_amd
    return mask_loss_amd.mask_loss


def inputs(seed, L, B, Q, H, W, G, C, dtype=torch.float32):
    rng = np.random.default_rng(seed)
    z = torch.from_numpy(rng.normal(0, 2, size=(L, B, Q, H, W)).astype(np.float32)).to(dtype).cuda()
    t = torch.from_numpy(rng.integers(0, G + 1, size=(B, H, W))).cuda()
    zc = torch.from_numpy(rng.normal(size=(L, B, Q, C)).astype(np.float32)).cuda()
    ct = torch.from_numpy(rng.integers(0, C - 1, size=(B, G + 1))).cuda()
    return z, t, zc, ct


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", ["broadcast", "every_other", "column"])
def test_upstream_gradient_strides(ml, dtype, form):
    L = 3
    z, t, zc, ct = inputs(1, L, 2, 12, 9, 16, 5, 4, dtype)
    head, tail = (1.0, 1.0, 1.0, 1.0, 0, 1.0, 0.05), (0.0, -1.0, 0.0, -1.0, 3, True, True)
    out = ml.mask_matching_fused(z, t, zc, ct, *head, 1e30, -1.0, True, False, 1, 0, *tail)
    if form == "broadcast":
        g = [torch.tensor(v, device="cuda").expand(L) for v in (1.0, 0.5, -2.0)]
    elif form == "every_other":
        g = [torch.arange(2 * L, device="cuda", dtype=torch.float32).add_(k)[::2] for k in range(3)]
    else:
        g = list(torch.randn(L, 3, device="cuda").unbind(1))
    args = (z, t, zc, ct, out[0], *head, -1.0, True, False, *tail, out[5])
    got = ml.mask_matching_backward_fused(*g, *args)
    ref = ml.mask_matching_backward_fused(*[x.contiguous() for x in g], *args)
    assert all(x.stride(0) != 1 for x in g)
    assert torch.equal(got[0], ref[0]) and torch.equal(got[1], ref[1])
    assert got[0].abs().sum() > 0


@pytest.mark.parametrize("strategy", [0, 1, 2, 3])
@pytest.mark.parametrize("K,G,Q", [(1, 7, 5), (1, 70, 5), (2, 130, 33), (4, 100, 64), (2, 250, 17), (1, 31, 1)])
def test_strategies_with_more_columns_than_queries(ml, strategy, K, G, Q):
    """Only the first Q open columns are rows of an assignment; the lists in LDS
    hold no more."""
    test_strategies_with_many_columns(ml, strategy, K, G, Q)


@pytest.mark.parametrize("strategy", [0, 1, 2, 3])
@pytest.mark.parametrize("K,G,Q", [(1, 70, 200), (2, 70, 100), (3, 130, 150), (2, 3, 40)])
def test_strategies_with_many_columns(ml, strategy, K, G, Q):
    z, t, zc, ct = inputs(2, 1, 2, Q, 24, 24, G, 6)
    head, tail = (1.0, 1.0, 1.0, 1.0, 0, 1.0, 0.05), (0.0, -1.0, 0.0, -1.0, 5, True, True)
    out = ml.mask_matching(z, t, zc, ct, *head, 1e30, -1.0, True, False, K, strategy, *tail)
    sep = ml.pairwise_mask_loss_forward(z, t, zc, ct, *head, 0.0, -1.0, 0.0, -1.0, True, True)
    total = ((sep[0] + sep[1]) + sep[2]).double().cpu().numpy().reshape(2, Q, G)
    p2g, rounds = OA.assign_batch(total, 1e30, K, strategy)
    assert np.array_equal(out[0].cpu().numpy().reshape(2, Q), p2g)
    assert np.array_equal(out[1].cpu().numpy().reshape(2, Q), rounds)


@pytest.mark.parametrize("one_cell", [False, True])
@pytest.mark.parametrize("H,W,P", [(1, 1, 50), (2, 1, 1025), (4, 8, 16384), (64, 128, 16384), (128, 128, 12544)])
def test_point_gradient_buckets(ml, H, W, P, one_cell):
    """The points' buckets split over workgroups: planes of fewer buckets than
    workgroups, every point in one bucket, points outside the plane and
    non-finite ones.  Quarter-cell positions and whole gradients make every
    product and sum exact in float32, so the results are the oracle's."""
    rng = np.random.default_rng(H + W + P)
    B, C = 3, 8
    size = np.array([W, H])
    pos = rng.integers(-8, 4 * size + 8, size=(B, P, 2))
    if one_cell:
        pos = 4 * (size // 2) + rng.integers(0, 4, size=(B, P, 2)) - 4
    c = ((pos / 4 + 0.5) / size).astype(np.float32)
    g = rng.integers(-3, 4, size=(B, C, P)).astype(np.float64)
    ref = PO.point_sample_backward(g[..., : P - 7], c[:, : P - 7], H, W, False)
    c[:, P - 7:] = np.array([np.nan, np.inf, -np.inf, 1e30, -1e30, np.nan, 7.0])[:, None]
    got = ml.point_sample_backward(torch.from_numpy(g).float().cuda(), torch.from_numpy(c).cuda(), H, W, False)
    np.testing.assert_array_equal(got.cpu().numpy(), ref)
