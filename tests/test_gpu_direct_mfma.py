"""The direct potential's matrix-core kernels against float64 sums, at the edges of their tiles and
with states that are not finite."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')

SHAPES = [(1, 1, 1, 16, 64, 4, 4), (2, 1, 1, 17, 65, 5, 7), (1, 1, 1, 8, 8, 13, 13), (3, 2, 2, 33, 17, 26, 9),
          (1, 1, 1, 70, 130, 64, 64), (2, 2, 1, 64, 64, 25, 25), (1, 1, 1, 40, 96, 1, 1), (40, 1, 1, 128, 128, 8, 8)]


def _padding(kh, kw):
    return tuple([(0, 0), (0, 0)] + [(d // 2, d // 2 - 1) if d % 2 == 0 else (d // 2, d // 2) for d in (kh, kw)])


def _kernel_gradient(A, dU, kh, kw, maxk):
    """dK [C * maxk, kh, kw] in float64: every tap's product summed over worlds and cells."""
    A, dU = A.astype(np.float64), dU.astype(np.float64)
    out = np.zeros((dU.shape[1], kh, kw))
    with np.errstate(invalid='ignore'):
        for i in range(kh):
            for j in range(kw):
                moved = np.roll(A, (kh // 2 - i, kw // 2 - j), axis=(2, 3))
                for k in range(dU.shape[1]):
                    out[k, i, j] = (dU[:, k] * moved[:, k // maxk]).sum()
    return out


@pytest.mark.parametrize('N,C,maxk,H,W,kh,kw', SHAPES)
def test_kernel_gradient_matches_float64(N, C, maxk, H, W, kh, kw):
    from leniax_amd import core
    print('kernel gradient', (N, C, maxk, H, W, kh, kw), flush=True)
    rng = np.random.default_rng(kh * 100 + H)
    A = rng.uniform(size=(N, C, H, W)).astype(np.float32)
    K = rng.uniform(size=(C * maxk, 1, kh, kw)).astype(np.float32)
    dU = rng.uniform(size=(N, C * maxk, H, W)).astype(np.float32)
    tK = torch.as_tensor(K).cuda().requires_grad_()
    pot = core.get_potential(torch.as_tensor(A).cuda(), tK, _padding(kh, kw))
    got = torch.autograd.grad(pot, tK, torch.as_tensor(dU).cuda())[0][:, 0].cpu().numpy()
    ref = _kernel_gradient(A, dU, kh, kw, maxk)
    # positive terms: a sum's relative error is at most (additions in a row) x 2^-24; a lane adds at most
    # 4 rows of 64 cells per tile, a block at most the tiles beyond 1024 / K rows of partial sums, then
    # 4 waves, 32 rows and 32 slices
    tiles = -(-N * -(-H // 16) * -(-W // 64) * C * maxk * 4 // 1024)
    bound = (256 * max(tiles, 1) + 84) * 2.0 ** -24
    err = float(np.max(np.abs(got - ref) / ref))
    print('  rel err', err, 'bound', bound)
    assert err <= bound


def test_kernel_gradient_of_a_state_that_is_not_finite():
    """inf x 0 is met nowhere that the sum itself does not meet it: W = 72 leaves a ragged last tile."""
    from leniax_amd import core
    rng = np.random.default_rng(2)
    A = rng.uniform(size=(1, 1, 24, 72)).astype(np.float32)
    A[0, 0, 3, 70] = np.inf
    K = rng.uniform(size=(1, 1, 5, 5)).astype(np.float32)
    dU = rng.uniform(0.5, 1, size=(1, 1, 24, 72)).astype(np.float32)
    tK = torch.as_tensor(K).cuda().requires_grad_()
    pot = core.get_potential(torch.as_tensor(A).cuda(), tK, _padding(5, 5))
    got = torch.autograd.grad(pot, tK, torch.as_tensor(dU).cuda())[0].cpu().numpy()
    assert np.all(np.isposinf(got)), got


@pytest.mark.parametrize('N,C,maxk,H,W,kh,kw', SHAPES + [(70, 2, 1, 64, 128, 6, 11), (600, 1, 1, 20, 36, 7, 3)])
def test_potential_and_state_gradient_match_float64(N, C, maxk, H, W, kh, kw):
    """Every output is kh kw (times the kernels of a channel) multiply-adds of positive terms in a row:
    a relative error of at most that many times 2^-24.  The last two shapes fill the chip (R = 2)."""
    from leniax_amd import core
    print('direct', (N, C, maxk, H, W, kh, kw), flush=True)
    rng = np.random.default_rng(kh * 100 + H)
    A = rng.uniform(size=(N, C, H, W)).astype(np.float32)
    K = rng.uniform(size=(C * maxk, 1, kh, kw)).astype(np.float32)
    dU = rng.uniform(size=(N, C * maxk, H, W)).astype(np.float32)
    tA = torch.as_tensor(A).cuda().requires_grad_()
    pot = core.get_potential(tA, torch.as_tensor(K).cuda(), _padding(kh, kw))
    dA = torch.autograd.grad(pot, tA, torch.as_tensor(dU).cuda())[0].cpu().numpy()
    refU, refA = np.zeros(dU.shape), np.zeros(A.shape)
    for i in range(kh):
        for j in range(kw):
            move = (kh // 2 - i, kw // 2 - j)
            for k in range(C * maxk):
                refU[:, k] += float(K[k, 0, i, j]) * np.roll(A[:, k // maxk].astype(np.float64), move, axis=(1, 2))
                refA[:, k // maxk] += float(K[k, 0, i, j]) * np.roll(dU[:, k].astype(np.float64),
                                                                     (-move[0], -move[1]), axis=(1, 2))
    errs = [float(np.max(np.abs(x - r) / r)) for x, r in ((pot.detach().cpu().numpy(), refU), (dA, refA))]
    print('  rel err', errs)
    assert errs[0] <= kh * kw * 2.0 ** -24 and errs[1] <= kh * kw * maxk * 2.0 ** -24


def test_potential_of_a_state_that_is_not_finite():
    """Exactly the cells whose window holds the infinite cell are infinite."""
    from leniax_amd import core
    A = np.full((1, 1, 40, 80), 0.5, np.float32)
    A[0, 0, 7, 60] = np.inf
    K = np.full((1, 1, 5, 6), 0.25, np.float32)
    pot = core.get_potential(torch.as_tensor(A).cuda(), torch.as_tensor(K).cuda(), _padding(5, 6))[0, 0].cpu().numpy()
    rows, cols = np.nonzero(np.isinf(pot))
    assert not np.isnan(pot).any()
    assert sorted(set(rows)) == list(range(5, 10)) and sorted(set(cols)) == list(range(58, 64)) and len(rows) == 30
    np.testing.assert_allclose(pot[~np.isinf(pot)], 30 * 0.125, rtol=30 * 2.0 ** -24)
