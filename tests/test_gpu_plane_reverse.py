"""The reverse of 3-D runs through whole planes (lx_plane.hip: plane_adj_kernel, first step and chained) against the
passes for rows and lines (a pinned knob of the lines turns the planes off) and the float64 oracle: every update
rule, the weighted mean and the weighted sum, two growth functions."""
import numpy as np
import pytest

from oracle import adjoint as ADJ
from oracle import lenia as L
from test_gpu_tune import _kernels, knobs  # noqa: F401

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')

B, STEPS, CKPT, M, S, W, DT = 2, 5, 2, 0.5, 0.1, 0.7, 0.1


def _inputs(dims):
    rng = np.random.default_rng(dims[1])
    kern = rng.random(dims)
    K = np.fft.fftn(kern / kern.sum()).astype(np.complex64)[None, None, None]
    A0 = rng.random((B, 1) + dims, dtype=np.float32)
    cot = rng.normal(size=(B, 1) + dims).astype(np.float32)
    return K, A0, cot


def _gradients(dims, growth, average, slug, ste):
    from leniax_amd import autograd as AG
    from leniax_amd import core
    K, A0, cot = _inputs(dims)
    leaves = [torch.as_tensor(x).cuda().requires_grad_()
              for x in (A0, K, np.array([[M, S]], np.float32), np.array([[W]], np.float32), np.float32(DT))]
    weighted = core.weighted_mean if average else core.weighted_sum
    out = AG.run(*leaves, STEPS, growth_fn_t=(growth,), weighted_fn=weighted, state_slug=slug, ste=ste, ckpt_every=CKPT)
    return [g.cpu().numpy() for g in torch.autograd.grad((out * torch.as_tensor(cot).cuda()).sum(), leaves)]


@pytest.mark.parametrize('dims', [(16, 32, 48), (16, 96, 32), (16, 32, 128)])
@pytest.mark.parametrize('slug,ste', [('v1', True), ('v1', False), ('v2', True), ('simple', True)])
@pytest.mark.parametrize('average', [True, False])
@pytest.mark.parametrize('growth', ['gaussian', 'poly_quad4'])
def test_planes_against_rows_and_lines_and_float64(knobs, growth, average, slug, ste, dims):  # noqa: F811
    """The same per-cell arithmetic and transforms: dL/dA0 and dL/dK bit for bit.  The scalars are float32 sums in
    two orders: of terms that are at most c |dL/dz|, c = 1.7 dt / s (growth's derivatives: at most 1.27 and 1.69
    over s), dt or 2, where sum |dL/dz| grows by 1 + 1.27 dt / s a step; a chain of at most 128 additions (36 points
    of a lane, 6 + 4 in a workgroup, 16 planes, the steps) either way.  The oracle's bound is that of the other
    gradient tests: four times float32's own distance from float64 and 1e-4 of the value."""
    print('plane reverse', dims, growth, average, slug, ste, flush=True)
    names = _kernels(lambda: _gradients(dims, growth, average, slug, ste))
    for bridge in ('true', 'false'):
        assert any(f'plane_adj_kernel<{dims[1]}, {dims[2]}, {bridge}>' in n for n in names), names
    planes = _gradients(dims, growth, average, slug, ste)
    knobs.tune_force('line_xcd', 1)
    assert not any('plane' in n for n in _kernels(lambda: _gradients(dims, growth, average, slug, ste)))
    general = _gradients(dims, growth, average, slug, ste)
    K, A0, cot = _inputs(dims)
    assert np.array_equal(planes[0], general[0])
    assert np.array_equal(planes[1], general[1])
    total = STEPS * float(np.abs(cot).sum()) * (1 + 1.27 * DT / S) ** STEPS
    for name, a, b, c in zip(('gf', 'w', 'dt'), planes[2:], general[2:], (1.7 * DT / S, DT, 2.)):
        assert np.abs(a - b).max() <= 2 * 128 * 2.0 ** -24 * c * total, (name, a, b)
    rule = L.Rule([growth], average=average, state_fn=slug)
    args = (rule, A0, K, np.array([[M, S]], np.float32), np.array([[W]], np.float32), DT, STEPS, cot, ste)
    o64, o32 = ADJ.run_vjp(*args), ADJ.run_vjp(*args, f=np.float32)
    for name, got in (('gf_params', planes[2]), ('weights', planes[3]), ('dt', planes[4])):
        r64, r32 = np.asarray(o64[name]), np.asarray(o32[name])
        err, env = np.abs(got - r64).max(), np.abs(r32 - r64).max()
        print(f'  {name}: |gpu-o64| {err:.3e} |o32-o64| {env:.3e} max|o64| {np.abs(r64).max():.3e}')
        if average and name == 'weights':  # the mean of one kernel does not depend on its weight: rounding of terms
            assert err <= 2 * 128 * 2.0 ** -24 * DT * total  # of both signs, each at most dt |dL/dz|
        else:
            assert err <= 4 * env + 1e-4 * np.abs(r64).max(), name


@pytest.mark.parametrize('dims,many', [((16, 128, 128), 33), ((16, 96, 96), 13), ((64, 96, 96), 9), ((32, 64, 128), 9),
                                       ((16, 32, 48), 5)])
def test_a_worlds_gradients_do_not_depend_on_its_batch(dims, many):
    """lx_adjoint_step of 3-D worlds with parameters of their own, in a batch and alone: dL/d(state in), the
    kernel-spectrum gradient and the gradient scalars of the first worlds bit for bit."""
    import ctypes
    from leniax_amd import _lib, autograd as AG, engine
    print('gradients alone and in a batch', dims, many, flush=True)
    rng = np.random.default_rng(dims[1])
    rule = engine.make_rule(list(dims), 1, [0], [_lib.GROWTH_IDS['gaussian']], _lib.STATE_FN['v2'], 0)
    Kh = torch.as_tensor(np.fft.rfftn(rng.random(dims) / np.prod(dims)).astype(np.complex64)).cuda()[None, None]
    A = torch.rand((many, 1) + dims, device='cuda')
    U, lam0 = 0.4 * torch.rand((many, 1) + dims, device='cuda'), torch.randn((many, 1) + dims, device='cuda')
    gf = torch.tensor([[0.2, 0.05]], device='cuda').repeat(many, 1)
    w, dt = torch.full((many,), 0.7, device='cuda'), torch.full((many,), 0.1, device='cuda')
    FA = AG.rfftn(A, 3)
    outs = []
    for B in (many, 1):
        nb = ctypes.c_size_t(0)
        _lib.call('lx_workspace_size', ctypes.byref(rule), B, ctypes.byref(nb))
        work = torch.empty(nb.value, dtype=torch.uint8, device='cuda')
        _lib.call('lx_adjoint_workspace_size', ctypes.byref(rule), B, ctypes.byref(nb))
        aw = torch.empty(nb.value, dtype=torch.uint8, device='cuda')
        lam = lam0[:B].clone()
        ggf, gw, gdt = torch.zeros_like(gf[:B]), torch.zeros_like(w[:B]), torch.zeros_like(dt[:B])
        dspec = torch.zeros((B, 1) + tuple(FA.shape[2:]), dtype=torch.complex64, device='cuda')
        _lib.call('lx_adjoint_step', ctypes.byref(rule), B, engine.ptr(A), None, engine.ptr(U), engine.ptr(gf), 2,
                  engine.ptr(w), 1, engine.ptr(dt), 1, engine.ptr(Kh), 0, 1, engine.ptr(FA), engine.ptr(dspec),
                  engine.ptr(lam), None, engine.ptr(ggf), engine.ptr(gw), engine.ptr(gdt), engine.ptr(work),
                  engine.ptr(aw), engine.stream_ptr())
        outs.append([x[:1].cpu().numpy() for x in (lam, dspec, ggf, gw, gdt)])
    for x, y in zip(*outs):
        assert np.array_equal(x, y)
    assert all(np.abs(x).max() > 0 for x in outs[1])
