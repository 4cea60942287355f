"""The variants of the inverse row pass by grid size (lx_fft.hip: rows loaded ahead or not) against the pass of
few worlds (lx_small.hip): the same arithmetic in the same order, so a world inside a batch equals the world
alone bit for bit: state, field, potentials, statistics."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')


# dims, worlds: 24 and 32 points a lane with up to and past 256 workgroups; 16 points with fewer than 768, with 769
# to 1024 and with more
@pytest.mark.parametrize('dims,B', [((32, 192), 450), ((32, 192), 700), ((32, 384), 200), ((32, 512), 250), ((32, 512), 270),
                                    ((32, 256), 700), ((32, 256), 900), ((32, 256), 1030), ((32, 128), 1800)])
def test_a_world_in_a_batch_equals_the_world_alone(dims, B):
    from leniax_amd import _lib, engine, runner
    print('inverse rows', dims, B, flush=True)
    C, K = 1, 2
    rng = np.random.default_rng(B)
    rule = engine.make_rule(list(dims), C, [0] * K, [_lib.GROWTH_IDS['gaussian']] * K, 0, False)
    kern = rng.random((K,) + dims)
    half = np.fft.rfftn(kern / kern.sum(axis=(1, 2), keepdims=True), axes=(1, 2)).astype(np.complex64)
    Kh = torch.as_tensor(half)[None].cuda().contiguous()
    gf = torch.as_tensor(rng.uniform(0.3, 0.6, (K, 2)).astype(np.float32)).cuda()
    w = torch.tensor([[0.4, 0.7]]).cuda()
    dt = torch.tensor([0.1]).cuda()
    cells = torch.as_tensor(rng.random((B, C) + dims, dtype=np.float32)).cuda()

    def run(x, keep):
        return runner._scan_plain(rule, None, x, Kh, 0, gf, w, dt, 2, 9., 10., keep)

    for keep in (True, False):  # with fields and potentials as outputs, and statistics alone
        many = run(cells, keep)
        for b in (0, B // 2, B - 1):
            rows1, n1, fin, hist = run(cells[b:b + 1].contiguous(), keep)
            assert torch.equal(fin[0], many[2][b])
            assert torch.equal(rows1[:, 0].nan_to_num(nan=-7.), many[0][:, b].nan_to_num(nan=-7.))
            if keep:
                assert all(torch.equal(one[:, 0], all_[:, b]) for one, all_ in zip(hist, many[3]))
