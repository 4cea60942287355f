"""3-D passes over whole planes (lx_plane.hip) against float64 transforms: planes of every kind of side
(powers of two and three times one, one and several rounds of rows), odd numbers of worlds, and the
accesses that the kernels leave to the general passes (arrays that do not start on 16 bytes)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')

SHAPES = [((16, 32, 32), 1, 1, 1), ((32, 48, 64), 3, 2, 3), ((48, 96, 96), 2, 1, 1), ((16, 128, 128), 1, 1, 2),
          ((32, 64, 48), 5, 1, 1), ((64, 128, 32), 1, 2, 2), ((16, 16, 96), 2, 1, 1)]


def _shifted(x):
    """The same values in a tensor that starts 4 bytes past a 16-byte boundary."""
    buf = torch.empty(x.numel() + 4, dtype=x.dtype, device=x.device)
    at = (4 - buf.data_ptr() // 4 % 4) % 4 + 1
    y = buf[at:at + x.numel()].view(x.shape)
    y.copy_(x)
    return y


@pytest.mark.parametrize('dims,B,C,K', SHAPES)
def test_transforms_and_step_match_float64(dims, B, C, K):
    """FFT round trips within 6 log2(n) roundings of the largest value; the step's potential likewise, its
    field and state within the growth's slope times that; the general passes agree with the planes."""
    from leniax_amd import autograd as AG
    from leniax_amd import core, engine, _lib
    print('planes', dims, B, C, K, flush=True)
    rng = np.random.default_rng(B)
    n = int(np.prod(dims))
    tol = 6 * np.log2(n) * 2.0 ** -24
    x = rng.random((B * C,) + dims, dtype=np.float32)
    ref = np.fft.rfftn(x.astype(np.float64), axes=(1, 2, 3))
    X = AG.rfftn(torch.as_tensor(x).cuda(), 3)
    assert np.abs(X.cpu().numpy() - ref).max() <= tol * np.abs(ref).max()
    back = AG.irfftn(X, dims).cpu().numpy()
    assert np.abs(back - x).max() <= 2 * tol
    rule = engine.make_rule(list(dims), C, [k % C for k in range(K)], [_lib.GROWTH_IDS['gaussian']] * K, 0, True)
    kern = rng.random((K,) + dims)
    kern /= kern.sum(axis=(1, 2, 3), keepdims=True)
    half = np.fft.rfftn(kern, axes=(1, 2, 3))
    Kh = torch.as_tensor(half.astype(np.complex64)).cuda()[None].contiguous()
    gf = np.stack([np.full(K, 0.5), np.full(K, 0.2)], 1).astype(np.float32)
    w = rng.uniform(0.2, 1, (C, K)).astype(np.float32)
    cells = x.reshape((B, C) + dims)
    spec = ref.reshape((B, C) + ref.shape[1:])
    pot64 = np.stack([np.fft.irfftn(spec[:, k % C] * half[k], s=dims, axes=(1, 2, 3)) for k in range(K)], 1)
    g64 = 2 * np.exp(-((pot64 - 0.5) / 0.2) ** 2 / 2) - 1
    field64 = np.einsum('ck,bk...->bc...', w.astype(np.float64), g64) / w.sum(1).reshape((1, C, 1, 1, 1))
    state64 = np.clip(cells + np.float32(0.1) * field64, 0, 1)
    import ctypes
    outs = []
    for move in (lambda t: t, _shifted):
        A = move(torch.as_tensor(cells).cuda())
        new, field = move(torch.empty_like(A)), move(torch.empty_like(A))
        pot = move(torch.empty((B, K) + dims, device='cuda'))
        gfd, wd = torch.as_tensor(gf).cuda(), torch.as_tensor(w).cuda()
        work = core._workspace(rule, B)
        _lib.call('lx_update_dt', ctypes.byref(rule), engine.ptr(A), B, engine.ptr(Kh), 0, engine.ptr(gfd), 0,
                  engine.ptr(wd), 0, 0.1, engine.ptr(new), engine.ptr(field), engine.ptr(pot), engine.ptr(work),
                  engine.stream_ptr())
        outs.append([t.cpu().numpy() for t in (pot, field, new)])
        if K > 1:  # without the caller's potentials
            new2 = move(torch.empty_like(A))
            _lib.call('lx_update_dt', ctypes.byref(rule), engine.ptr(A), B, engine.ptr(Kh), 0, engine.ptr(gfd), 0,
                      engine.ptr(wd), 0, 0.1, engine.ptr(new2), None, None, engine.ptr(work), engine.stream_ptr())
            assert torch.equal(new2, new)
    for pot, field, new in outs:
        assert np.abs(pot - pot64).max() <= 2 * tol
        # |g'| <= 2 exp(-1/2) / 0.2 < 6.1; a few roundings of the growth and the mean besides
        assert np.abs(field - field64).max() <= 6.1 * 2 * tol + 8 * 2.0 ** -23
        assert np.abs(new - state64).max() <= 0.1 * (6.1 * 2 * tol + 8 * 2.0 ** -23) + 2 * 2.0 ** -24


@pytest.mark.parametrize('ste', [True, False])
@pytest.mark.parametrize('slug', ['v1', 'v2'])
def test_reverse_steps_agree_with_the_general_passes(slug, ste):
    """Gradients of a 3-D run through the plane kernels against the same run's single steps composed by
    autograd (pointwise reverse and adjoint potential as separate entry points)."""
    from leniax_amd import autograd as AG
    dims, B = (32, 48, 64), 2
    rng = np.random.default_rng(5)
    kern = rng.random(dims)
    K = torch.as_tensor(np.fft.fftn(kern / kern.sum()).astype(np.complex64)).cuda()[None, None, None]
    A0 = torch.as_tensor(rng.random((B, 1) + dims, dtype=np.float32)).cuda()
    cot = torch.as_tensor(rng.normal(size=(B, 1) + dims).astype(np.float32)).cuda()
    grads = []
    for whole in (True, False):
        A, k = A0.clone().requires_grad_(), K.clone().requires_grad_()
        gf = torch.tensor([[0.5, 0.1]], device='cuda', requires_grad=True)
        w = torch.tensor([[0.7]], device='cuda', requires_grad=True)
        dt = torch.tensor(0.1, device='cuda', requires_grad=True)
        if whole:
            out = AG.run(A, k, gf, w, dt, 5, state_slug=slug, ste=ste, ckpt_every=2)
        else:
            out = A
            for _ in range(5):
                # a cotangent of the field as well: the step's reverse then goes through its two halves
                out, field, _ = AG.update(out, k, gf, w, dt, state_slug=slug, ste=ste)
                out = out + 0 * field
        grads.append(torch.autograd.grad((out * cot).sum(), (A, k, gf, w, dt)))
    for name, a, b in zip(('state', 'K', 'gf', 'w', 'dt'), *grads):
        err = float((a - b).abs().max() / b.abs().max().clamp_min(1e-30))
        print(slug, ste, name, err, flush=True)
        # five steps of float32 transforms either way: 1e-4 is the single steps' own bound against float64
        assert err <= 1e-4 or name == 'w', (name, err)


def test_more_images_than_a_grid_dimension_holds():
    """32770 worlds of two channels (65540 images, past the 65535 of a grid's y dimension): five different worlds
    over and over, each copy equal to the world stepped in a batch of five."""
    from test_gpu_3d_same_bits import _case, _update
    rule, Kh, gf, w, A = _case((16, 32, 32), 5, 2, 1)
    few = _update(rule, Kh, gf, w, A, pot=False)
    copies = 6554
    many = _update(rule, Kh, gf, w, A.repeat(copies, 1, 1, 1, 1), pot=False)
    for a, b in zip(few, many):
        b = b.view((copies,) + tuple(a.shape))
        assert bool((b == a).all())
