"""Histories of the fused run: any of the three may be left out, and what is kept does not depend on which."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')


@pytest.mark.parametrize('n', [32, 64, 128])
@pytest.mark.parametrize('kept', [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1)])
def test_a_history_left_out_changes_nothing_else(monkeypatch, n, kept):
    from leniax_amd import _lib, engine
    B, steps, R, T = 3, 5, 9., 10.
    print('fused histories', n, kept, flush=True)
    rng = np.random.default_rng(n)
    cells0 = torch.as_tensor(rng.random((B, 1, n, n), dtype=np.float32)).to(engine.device())
    yy, xx = np.mgrid[:n, :n] - n // 2
    K = np.exp(-(yy * yy + xx * xx) / 18.)[None].astype(np.float32)
    K = np.fft.fftn(np.fft.fftshift(K / K.sum(), axes=(1, 2)), axes=(1, 2))[None, None].astype(np.complex64)
    rule = engine.make_rule([n, n], 1, [0], [_lib.GROWTH_IDS['gaussian']], _lib.STATE_FN['v1'], 1)
    Kh = engine.prepare_spectra(rule, K, [0])
    dev = cells0.device
    gf = torch.tensor([[[0.4, 0.1]]], device=dev)
    w = torch.ones(1, 1, 1, device=dev)
    dt = torch.tensor([0.1], device=dev)
    fields = ('cells_hist_d', 'field_hist_d', 'potential_hist_d')
    call = _lib.call

    def drop(name, *args):
        if name == 'lx_run':
            for field, keep in zip(fields, kept):
                if not keep:
                    setattr(args[1]._obj, field, None)
        return call(name, *args)

    full = engine.run_batched(rule, cells0, Kh, False, gf, w, dt, steps, 'leniax', steps, R, T, want_hist=True)
    with monkeypatch.context() as m:
        m.setattr(_lib, 'call', drop)
        part = engine.run_batched(rule, cells0, Kh, False, gf, w, dt, steps, 'leniax', steps, R, T, want_hist=True)
    torch.cuda.synchronize()
    assert torch.equal(full['hist'][0][0], cells0)
    assert all(bool(h.ne(0).any()) for h in full['hist'])
    for f, p, keep in zip(full['hist'], part['hist'], kept):
        assert torch.equal(p, f) if keep else not bool(p.ne(0).any())
    assert torch.equal(full['cells'], part['cells'])
    assert torch.equal(full['stats'], part['stats'])
