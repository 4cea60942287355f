"""lx_run's live list on grids past the passes of a few worlds (lx_fft.hip's LIST kernels: rows loaded ahead or
not by the grid's size, waves that lie in several worlds) against the same steps taken one lx_step_stats call at a
time, bit for bit, with spectra and parameters per world; worlds that retire after the first step leave
slots to the queue."""
import numpy as np
import pytest

from test_gpu_run import _expected_stop
from test_gpu_tune import _kernels

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')


# dims, slots, the inverse rows' kernel: 24 and 32 points a lane with up to and past 256 workgroups; 16 points with
# up to 768, with 769 to 1024 and with more; waves that straddle worlds
@pytest.mark.parametrize('dims,slots,kernel', [
    ((32, 192), 450, '192, true, true, true, true'), ((32, 192), 700, '192, true, true, true, false'),
    ((32, 384), 200, '384, true, true, true, true'), ((32, 384), 300, '384, true, true, true, false'),
    ((32, 512), 250, '512, true, true, true, true'), ((32, 512), 270, '512, true, true, true, false'),
    ((32, 256), 700, '256, true, true, true, true'), ((32, 256), 900, '256, true, true, true, false'),
    ((32, 256), 1030, '256, true, true, true, true'), ((32, 128), 1000, '128, true, true, true, true'),
    ((32, 128), 1800, '128, true, true, true, false'), ((32, 96), 1300, '96, true, true, true, true'),
    ((48, 64), 700, '64, true, false, true, true')])
def test_live_list_equals_the_step_loop(dims, slots, kernel):
    from leniax_amd import _lib, engine, runner
    print('live list', dims, slots, flush=True)
    C, K, B, steps = 1, 2, slots + 5, 3
    rng = np.random.default_rng(slots)
    rule = engine.make_rule(list(dims), C, [0] * K, [_lib.GROWTH_IDS['gaussian']] * K, 0, False)
    kern = rng.random((7, K) + dims)
    half = np.fft.rfftn(kern / kern.sum(axis=(2, 3), keepdims=True), axes=(2, 3)).astype(np.complex64)
    Kh = torch.as_tensor(half).cuda()[torch.arange(B, device='cuda') % 7].contiguous()
    gf = torch.as_tensor(rng.uniform(0.3, 0.6, (B, K, 2)).astype(np.float32)).cuda()
    w = torch.as_tensor(rng.uniform(0.2, 0.9, (B, C, K)).astype(np.float32)).cuda()
    dt = torch.as_tensor(rng.uniform(0.05, 0.2, B).astype(np.float32)).cuda()
    cells = torch.as_tensor(rng.random((B, C) + dims, dtype=np.float32)).cuda()
    cells[:, :, :12] = 0
    cells[1::3] = 0  # these retire at their first step under the mass policy
    rows, n, fin, hist = runner._scan_plain(rule, None, cells, Kh, int(Kh[0].numel()), gf, w, dt, steps, 9., 10., True)
    res = {}

    def run(stop):
        res.update(engine.run_batched(rule, cells, Kh, True, gf, w, dt, steps, stop, 0, 9., 10., slots=slots))
        torch.cuda.synchronize()

    names = _kernels(lambda: run('none'))
    assert any(f'rows_inv_kernel<{kernel}>' in x for x in names), names
    assert torch.equal(res['cells'], fin)
    assert torch.equal(res['stats'].transpose(0, 1).nan_to_num(nan=-7.), rows.nan_to_num(nan=-7.))
    assert res['n'].float().tolist() == n.tolist() and res['steps'].tolist() == [steps] * B
    run('mass')
    cells_h = hist[0]
    want = _expected_stop(rule, 'mass', 0, steps, rows, n, cells_h.cpu().numpy())
    assert res['steps'].tolist() == want and len(set(want)) > 1
    at = torch.as_tensor(want).cuda()
    states = torch.cat([cells_h, fin[None]])  # after 0 .. steps steps
    assert torch.equal(res['cells'], states[at, torch.arange(B, device='cuda')])
    for t in range(steps):
        ran = at > t
        assert torch.equal(res['stats'][ran, t].nan_to_num(nan=-7.), rows[t][ran].nan_to_num(nan=-7.))
