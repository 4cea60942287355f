"""The passes of a few worlds (lx_small.hip) against the passes of many (lx_fft.hip): the same arithmetic in
the same order, so a world stepped alone equals the same world inside a batch past the rule's 2048 waves,
bit for bit: states, fields, potentials, statistics."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')

# dims, channels, kernels, state function, average, quadrant spectra
SHAPES = [((16, 16), 1, 1, 'v1', True, False), ((48, 96), 2, 3, 'v2', False, False),
          ((64, 512), 4, 16, 'simple', True, False), ((512, 32), 3, 2, 'v1', True, False),
          ((128, 128), 3, 15, 'v1', False, True), ((384, 192), 1, 5, 'v1', True, False),
          ((16, 32, 48), 2, 2, 'v1', False, False)]


def _tpr(n):
    return 4 if n <= 64 else 8 if n <= 192 else 16


@pytest.mark.parametrize('dims,C,K,state_fn,average,quad', SHAPES)
def test_a_world_alone_equals_the_world_in_a_batch(dims, C, K, state_fn, average, quad):
    from leniax_amd import _lib, engine, runner
    n, nd = int(np.prod(dims)), len(dims)
    rows = n // dims[-1]
    # past 2048 waves in the row pass and in the convolution pass, with channels for kernels
    per_rows = rows // 2 * min(C, K) * _tpr(dims[-1]) / 64
    per_lines = min(C, K) * (n // dims[0] // dims[-1]) * (dims[-1] // 2 + 1) * _tpr(dims[0]) / 64
    B = int(2048 / min(per_rows, per_lines)) + 2
    print('few against many', dims, C, K, 'batch', B, flush=True)
    rng = np.random.default_rng(K)
    kinds = [(k % 7) for k in range(K)]
    rule = engine.make_rule(list(dims), C, [k % C for k in range(K)], kinds, _lib.STATE_FN[state_fn], average)
    kern = rng.random((K,) + dims)
    if quad:  # even kernels: their spectra are real and even
        for ax in (1, 2):
            kern = kern + np.roll(np.flip(kern, ax), 1, ax)
    kern /= kern.sum(axis=tuple(range(1, nd + 1)), keepdims=True)
    half = np.fft.rfftn(kern, axes=tuple(range(1, nd + 1))).astype(np.complex64)
    Kh = torch.as_tensor(half)[None].cuda().contiguous()
    if quad:
        Kh, rule = engine.quadrant_spectra(rule, Kh)
    gf = torch.as_tensor(rng.uniform(0.3, 0.6, (K, 2)).astype(np.float32)).cuda()
    w = torch.as_tensor(rng.uniform(0.1, 1, (C, K)).astype(np.float32)).cuda()
    if K > 2:
        w[:, 1] = 0  # a kernel that feeds no channel
    dt = torch.tensor([0.1]).cuda()
    cells = torch.zeros((B, C) + dims)
    cells[:3] = torch.as_tensor(rng.random((min(3, B), C) + dims, dtype=np.float32))
    cells = cells.cuda()

    def run(x):
        return runner._scan_plain(rule, None, x, Kh, 0, gf, w, dt, 2, 9., 10., True)

    many = run(cells)
    for b in range(min(2, B)):
        rows1, n1, fin, hist = run(cells[b:b + 1].contiguous())
        assert torch.equal(fin[0], many[2][b])
        for one, all_ in zip(hist, many[3]):
            assert torch.equal(one[:, 0], all_[:, b])
        assert torch.equal(rows1[:, 0].nan_to_num(nan=-7.), many[0][:, b].nan_to_num(nan=-7.)), (rows1, many[0][:, b])
