"""One 3-D step gives the same bits whichever entry point takes it: whole planes (lx_plane.hip: lx_update on
arrays that start on 16 bytes), the passes for rows and lines (arrays that do not; steps with statistics),
and the live list of lx_run.  Every side that the plane kernels take, with one channel and kernel (the update
inside the plane kernel) and with several (the update from the potentials)."""
import ctypes

import numpy as np
import pytest

from test_gpu_plane import _shifted
from test_gpu_tune import _kernels, knobs  # noqa: F401

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')

SIDES = (32, 48, 64, 96, 128)


def _case(dims, B, C, K, gf='gaussian', average=False, seed=0):
    from leniax_amd import _lib, engine
    rng = np.random.default_rng(seed + dims[1] + 1000 * dims[2])
    rule = engine.make_rule(list(dims), C, [k % C for k in range(K)], [_lib.GROWTH_IDS[gf]] * K, 0, average)
    kern = rng.random((K,) + dims)
    half = np.fft.rfftn(kern / kern.sum(axis=(1, 2, 3), keepdims=True), axes=(1, 2, 3))
    Kh = torch.as_tensor(half.astype(np.complex64)).cuda()[None].contiguous()
    gfd = torch.as_tensor(rng.uniform(0.3, 0.6, (K, 2)).astype(np.float32)).cuda()
    w = torch.as_tensor(rng.uniform(0.2, 1, (C, K)).astype(np.float32)).cuda()
    A = torch.as_tensor(rng.random((B, C) + dims, dtype=np.float32)).cuda()
    return rule, Kh, gfd, w, A


def _update(rule, Kh, gf, w, A, dt=0.1, pot=True, move=lambda t: t):
    """lx_update_dt's state, field and (pot) potentials."""
    from leniax_amd import _lib, core, engine
    B, dims = A.shape[0], tuple(A.shape[2:])
    A = move(A)
    new, field = move(torch.empty_like(A)), move(torch.empty_like(A))
    u = move(torch.empty((B, rule.K) + dims, device='cuda')) if pot else None
    _lib.call('lx_update_dt', ctypes.byref(rule), engine.ptr(A), B, engine.ptr(Kh), 0, engine.ptr(gf), 0,
              engine.ptr(w), 0, dt, engine.ptr(new), engine.ptr(field), engine.ptr(u),
              engine.ptr(core._workspace(rule, B)), engine.stream_ptr())
    return (new, field, u) if pot else (new, field)


@pytest.mark.parametrize('C,K', [(1, 1), (2, 2)])
@pytest.mark.parametrize('H', SIDES)
def test_entry_points_agree_bit_for_bit(H, C, K):
    from leniax_amd import engine, runner
    for W in SIDES:
        print('same bits', (16, H, W), C, K, flush=True)
        rule, Kh, gf, w, A = _case((16, H, W), 3 if H * W <= 6144 else 33, C, K)  # planes enough to be taken
        names = _kernels(lambda: _update(rule, Kh, gf, w, A))
        assert any(f'plane_inv_kernel<{H}, {W}>' in n for n in names), names
        planes = _update(rule, Kh, gf, w, A)
        general = _update(rule, Kh, gf, w, A, move=_shifted)
        bad = [n for n, a, b in zip(('state', 'field', 'potential'), planes, general) if not torch.equal(a, b)]
        assert not bad, ('planes against rows and lines', H, W, bad)
        dt = torch.tensor([0.1]).cuda()
        rows, n, fin, hist = runner._scan_plain(rule, None, A, Kh, 0, gf, w, dt, 1, 9., 10., True)
        assert torch.equal(fin, planes[0]) and torch.equal(hist[1][0], planes[1]) and torch.equal(hist[2][0], planes[2])
        second = _update(rule, Kh, gf, w, planes[0])[0]
        # fewer slots than worlds: the live list
        r = engine.run_batched(rule, A, Kh, False, gf[None], w[None], dt, 2, 'none', 0, 9., 10., slots=2)
        assert torch.equal(r['cells'], second), ('live list', H, W)


@pytest.mark.parametrize('dims,n', [((16, 32, 128), 2), ((32, 128, 96), 16), ((96, 96, 96), 2), ((48, 64, 64), 2),
                                    ((128, 48, 128), 2)])
def test_transforms_agree_bit_for_bit(dims, n):
    """rfftn and irfftn of arrays that start on 16 bytes (planes) and of arrays that do not."""
    from leniax_amd import _lib, engine
    print('same bits, transforms', dims, flush=True)
    rng = np.random.default_rng(1)
    x = torch.as_tensor(rng.random((n,) + dims, dtype=np.float32)).cuda()
    cd = (ctypes.c_int32 * 3)(*dims)
    spectra, backs = [], []
    for move in (lambda t: t, _shifted):
        a = move(x)
        X = torch.empty((n,) + dims[:2] + (dims[2] // 2 + 1,), dtype=torch.complex64, device='cuda')
        _lib.call('lx_rfft2', 3, cd, n, engine.ptr(a), engine.ptr(X), engine.stream_ptr())
        back, work = move(torch.empty_like(x)), torch.empty_like(X)
        _lib.call('lx_irfft2', 3, cd, n, engine.ptr(X), engine.ptr(back), engine.ptr(work), engine.stream_ptr())
        spectra.append(X)
        backs.append(back)
    assert torch.equal(torch.view_as_real(spectra[0]), torch.view_as_real(spectra[1]))
    assert torch.equal(backs[0], backs[1])


@pytest.mark.parametrize('average', [False, True])
def test_a_kernel_without_weight_adds_nothing(average):
    """One channel, one kernel of weight 0, a state with a NaN: where no potential is asked for, the kernel is
    left out (0 times its growth would be NaN in every cell), by planes as by the row pass; where one is, it
    counts as 0 times the growth in both."""
    print('weight 0', average, flush=True)
    rule, Kh, gf, w, A = _case((16, 32, 48), 2, 1, 1, average=average)
    w.zero_()
    A[0, 0, 3, 5, 7] = float('nan')
    for pot in (False, True):
        outs = [_update(rule, Kh, gf, w, A, pot=pot, move=move) for move in (lambda t: t, _shifted)]
        for a, b in zip(*outs):
            assert torch.equal(a.isnan(), b.isnan())
            assert torch.equal(a.nan_to_num(nan=-7.), b.nan_to_num(nan=-7.))
        if not pot and not average:
            assert int(outs[0][0].isnan().sum()) == 1


def test_a_workspace_that_starts_on_8_bytes():
    """Several kernels without the caller's potentials: they are kept in the workspace, with 16-byte accesses only
    where it starts on 16 bytes."""
    from leniax_amd import _lib, core, engine
    rule, Kh, gf, w, A = _case((16, 32, 48), 2, 2, 2)
    ref = _update(rule, Kh, gf, w, A, pot=False)[0]
    nb = ctypes.c_size_t(0)
    _lib.call('lx_workspace_size', ctypes.byref(rule), 2, ctypes.byref(nb))
    buf = torch.empty(nb.value + 16, dtype=torch.uint8, device='cuda')
    work = buf[(8 - buf.data_ptr()) % 16:]
    assert work.data_ptr() % 16 == 8
    new = torch.empty_like(A)
    _lib.call('lx_update_dt', ctypes.byref(rule), engine.ptr(A), 2, engine.ptr(Kh), 0, engine.ptr(gf), 0,
              engine.ptr(w), 0, 0.1, engine.ptr(new), None, None, engine.ptr(work), engine.stream_ptr())
    assert torch.equal(new, ref)


@pytest.mark.parametrize('dims,few,many', [((16, 128, 128), 1, 17), ((16, 96, 96), 9, 10), ((32, 64, 128), 4, 5),
                                           ((16, 128, 96), 5, 10)])
def test_few_large_planes_take_rows_and_lines(dims, few, many):
    """A large plane is one workgroup's long chain: below a count the passes spread over the chip instead, with the
    same bits."""
    print('few planes', dims, few, many, flush=True)
    rule, Kh, gf, w, A = _case(dims, many, 1, 1)
    names = _kernels(lambda: _update(rule, Kh, gf, w, A))
    assert any('plane_fwd' in n for n in names) and any('plane_inv' in n for n in names), names
    ref = _update(rule, Kh, gf, w, A)
    B = A[:few].contiguous()
    names = _kernels(lambda: _update(rule, Kh, gf, w, B))
    assert not any('plane_inv' in n or dims[1] * dims[2] > 9216 and 'plane' in n for n in names), names
    for a, b in zip(ref, _update(rule, Kh, gf, w, B)):
        assert torch.equal(a[:few], b)


@pytest.mark.parametrize('dims,B', [((64, 96, 96), 3), ((96, 128, 96), 3), ((64, 64, 128), 3)])
def test_reverse_through_large_planes_gives_the_same_bits(knobs, dims, B):  # noqa: F811
    """dL/dA0 of a run of whole planes against rows and lines (a pinned knob of the lines turns the planes off)."""
    from leniax_amd import autograd as AG
    print('reverse', dims, B, flush=True)
    rng = np.random.default_rng(3)
    kern = rng.random(dims)
    K = torch.as_tensor(np.fft.fftn(kern / kern.sum()).astype(np.complex64)).cuda()[None, None, None]
    A0 = torch.as_tensor(rng.random((B, 1) + dims, dtype=np.float32)).cuda().requires_grad_()
    cot = torch.as_tensor(rng.normal(size=(B, 1) + dims).astype(np.float32)).cuda()
    gf, w = torch.tensor([[0.5, 0.1]], device='cuda'), torch.ones((1, 1), device='cuda')

    def gradient():
        out = AG.run(A0, K, gf, w, torch.tensor(0.1, device='cuda'), 3, state_slug='v2', ckpt_every=2)
        return torch.autograd.grad((out * cot).sum(), A0)[0]
    assert any('plane_adj_kernel' in n for n in _kernels(gradient))
    planes = gradient()
    knobs.tune_force('line_xcd', 1)
    assert not any('plane' in n for n in _kernels(gradient))
    assert torch.equal(planes, gradient())
