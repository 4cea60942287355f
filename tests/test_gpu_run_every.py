"""lx_run without a stop policy and with every world in flight (steps enqueued one by one) against the
per-step entry point, bit for bit: odd and even step counts, states in place, histories."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')


@pytest.mark.parametrize('dims,C,K,B,steps', [((48, 96), 2, 3, 3, 1), ((48, 96), 2, 3, 3, 4), ((256, 16), 1, 2, 1, 3),
                                              ((32, 16, 48), 2, 2, 2, 3), ((256, 256), 3, 6, 40, 2)])
def test_run_without_stop_equals_the_steps(dims, C, K, B, steps):
    from leniax_amd import _lib, engine, runner
    print('run without stop', dims, C, K, B, steps, flush=True)
    rng = np.random.default_rng(steps)
    rule = engine.make_rule(list(dims), C, [k % C for k in range(K)], [_lib.GROWTH_IDS['gaussian']] * K, 0, False)
    kern = rng.random((B, K) + dims)
    axes = tuple(range(2, 2 + len(dims)))
    Kh = torch.as_tensor(np.fft.rfftn(kern / kern.sum(axis=axes, keepdims=True), axes=axes).astype(np.complex64)).cuda()
    gf = torch.as_tensor(rng.uniform(0.3, 0.6, (B, K, 2)).astype(np.float32)).cuda()
    w = torch.as_tensor(rng.uniform(0.1, 1, (B, C, K)).astype(np.float32)).cuda()
    dt = torch.as_tensor(rng.uniform(0.05, 0.2, B).astype(np.float32)).cuda()
    cells = torch.as_tensor(rng.random((B, C) + dims, dtype=np.float32)).cuda()
    assert engine.run_path(rule) == 'passes'
    rows, n, fin, hist = runner._scan_plain(rule, None, cells, Kh, int(Kh[0].numel()), gf, w, dt, steps, 9., 10., True)
    for in_place in (False, True):
        for want_hist in (False, True):
            x = cells.clone()
            r = engine.run_batched(rule, x, Kh, True, gf, w, dt, steps, 'none', 0, 9., 10., want_hist=want_hist,
                                   out=x if in_place else None)
            assert torch.equal(r['cells'], fin)
            assert torch.equal(r['stats'].transpose(0, 1).nan_to_num(nan=-7.), rows.nan_to_num(nan=-7.))
            assert r['steps'].tolist() == [steps] * B and r['n'].float().tolist() == n.tolist()
            if want_hist:
                assert all(torch.equal(a, b) for a, b in zip(r['hist'], hist))
            if not in_place:
                assert torch.equal(x, cells)
