"""Kernels that a shape chooses by itself, each against the kernel it stands in for."""
import ctypes

import numpy as np
import pytest

from test_gpu_direct_mfma import _kernel_gradient
from test_gpu_tune import _kernels, knobs  # noqa: F401

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')


def _case(dims, B, C, K, seed=0, average=True):
    from leniax_amd import _lib, engine
    rng = np.random.default_rng(seed)
    axes = tuple(range(1, len(dims) + 1))
    rule = engine.make_rule(list(dims), C, [k % C for k in range(K)], [k % 7 for k in range(K)], 0, average)
    kern = rng.random((K,) + dims)
    half = np.fft.rfftn(kern / kern.sum(axis=axes, keepdims=True), axes=axes).astype(np.complex64)
    gf = torch.as_tensor(rng.uniform(0.3, 0.6, (K, 2)).astype(np.float32)).cuda()
    w = torch.as_tensor(rng.uniform(0.1, 1, (C, K)).astype(np.float32)).cuda()
    A = torch.as_tensor(rng.random((B, C) + dims, dtype=np.float32)).cuda()
    return rule, torch.as_tensor(half).cuda()[None].contiguous(), gf, w, A


def _calls(rule, Kh, gf, w, A):
    """Name -> a call and its outputs: the step with spectra kept (FA), the step with and without its optional
    outputs, the potential alone, its adjoint (conjugate spectra; the state is added to in place)."""
    from leniax_amd import core, engine, _lib
    B, C, dims, K = A.shape[0], rule.C, tuple(A.shape[2:]), rule.K
    p, st = engine.ptr, engine.stream_ptr()
    work = core._workspace(rule, B)
    dt = torch.tensor([0.1], device='cuda')
    new, field = torch.empty_like(A), torch.empty_like(A)
    new2, lam = torch.empty_like(A), torch.empty_like(A)
    pot, pot2 = torch.empty((B, K) + dims, device='cuda'), torch.empty((B, K) + dims, device='cuda')
    spec = torch.empty((B, C) + dims[:-1] + (dims[-1] // 2 + 1,), dtype=torch.complex64, device='cuda')
    dpot = torch.sin(torch.arange(B * K * int(np.prod(dims)), device='cuda', dtype=torch.float32)).view(pot.shape)
    r = ctypes.byref(rule)

    def adjoint():
        lam.copy_(A)
        _lib.call('lx_adjoint_potential', r, B, p(Kh), 0, p(dpot), None, None, p(lam), p(work), st)
    return {
        'update': (lambda: _lib.call('lx_update', r, p(A), B, p(Kh), 0, p(gf), 0, p(w), 0, p(dt), 0, p(new), p(field),
                                     p(pot), p(work), st), (new, field, pot)),
        'update, state alone': (lambda: _lib.call('lx_update', r, p(A), B, p(Kh), 0, p(gf), 0, p(w), 0, p(dt), 0,
                                                  p(new2), None, None, p(work), st), (new2,)),
        'spectra': (lambda: _lib.call('lx_update_with_spectra', r, p(A), B, p(Kh), 0, p(gf), 0, p(w), 0, p(dt), 0,
                                      p(new2), None, None, p(spec), p(work), st), (new2, spec)),
        'potential': (lambda: _lib.call('lx_potential', r, p(A), B, p(Kh), 0, p(pot2), p(work), st), (pot2,)),
        'adjoint': (adjoint, (lam,)),
    }


def _bits(outs, n=None):
    return [torch.view_as_real(o[:n]).clone() if o.is_complex() else o[:n].clone() for o in outs]


# worlds a lane group: 2, 2, 2, 8 with two left over, 2, 2
@pytest.mark.parametrize('dims,B', [((96, 96, 96), 11), ((32, 96, 96), 21), ((48, 64, 128), 25), ((32, 128, 128), 50),
                                    ((64, 96, 96), 23), ((128, 96, 64), 17)])
def test_shared_spectrum_convolution(knobs, dims, B):  # noqa: F811
    """3-D worlds that share one kernel's spectrum, several worlds a lane group (shared_conv_kernel), against
    lines_kernel bit for bit: with the spectra kept, with the conjugate spectrum."""
    print('shared spectrum', dims, B, flush=True)
    calls = _calls(*_case(dims, B, 1, 1))
    for name in ('update', 'spectra', 'potential', 'adjoint'):
        call, outs = calls[name]
        for unpin in (True, False):
            knobs.tune_force('line_xcd', None if unpin else 1)
            names = _kernels(call)
            assert any('shared_conv_kernel' in x for x in names) == unpin, (name, names)
            if unpin:
                ref = _bits(outs)
        # the planes round as the rows and lines that the pinned knob takes instead
        assert all(torch.equal(a, b) for a, b in zip(ref, _bits(outs))), name


def _tpr(n):
    return 4 if n <= 64 else 8 if n <= 192 else 16


@pytest.mark.parametrize('dims,C,K', [((16, 16), 1, 1), ((48, 96), 2, 3), ((64, 512), 4, 6), ((512, 32), 3, 2),
                                      ((128, 128), 3, 15), ((384, 192), 1, 5), ((32, 384), 1, 2), ((32, 256), 1, 2),
                                      ((16, 32, 16), 2, 2)])
def test_few_worlds_without_statistics(dims, C, K):
    """Entry points without statistics: a world alone (lx_small.hip) equals the world in a batch past the few
    worlds' limits (lx_fft.hip), bit for bit."""
    n, rows = int(np.prod(dims)), int(np.prod(dims[:-1]))
    per_rows = rows // 2 * min(C, K) * _tpr(dims[-1]) / 64
    per_lines = min(C, K) * (n // dims[0] // dims[-1]) * (dims[-1] // 2 + 1) * _tpr(dims[0]) / 64
    B = int(2048 / min(per_rows, per_lines)) + 2
    print('few against many', dims, C, K, 'batch', B, flush=True)
    rule, Kh, gf, w, A = _case(dims, B, C, K, seed=K)
    if K > 2:
        w[:, 1] = 0  # a kernel that feeds no channel
    many, one = _calls(rule, Kh, gf, w, A), _calls(rule, Kh, gf, w, A[:1].contiguous())
    for name, (call, outs) in many.items():
        few, few_outs = one[name]
        names = _kernels(call)
        assert not any('small_' in x for x in names), (name, names)
        names = _kernels(few)
        assert any('small_rows_kernel' in x for x in names), (name, names)
        if name == 'adjoint':  # its inputs follow the flat index: the first world's are the same
            assert any('small_conv_kernel' in x for x in names), names
        assert all(torch.equal(a, b) for a, b in zip(_bits(few_outs), _bits(outs, 1))), name


def test_few_worlds_at_the_most_items_a_thread_takes():
    """4 channels of 512 points: 1024 four-point items for 256 threads, with statistics."""
    from test_gpu_small import test_a_world_alone_equals_the_world_in_a_batch as check
    from leniax_amd import runner
    rule, Kh, gf, w, A = _case((64, 512), 1, 4, 6)
    dt = torch.tensor([0.1], device='cuda')
    names = _kernels(lambda: runner._scan_plain(rule, None, A, Kh, 0, gf, w, dt, 1, 9., 10., True))
    assert any('small_rows_kernel<512, true, false>' in x for x in names), names
    check((64, 512), 4, 6, 'v1', True, False)


@pytest.mark.parametrize('B,C,maxk,H,W,kh,kw', [(2, 2, 1, 17, 65, 5, 7), (1, 1, 2, 40, 24, 1, 8),
                                                (3, 1, 1, 8, 8, 13, 13)])
def test_direct_adjoint_without_a_workspace(B, C, maxk, H, W, kh, kw):
    """lx_potential_direct_adjoint (one workgroup per tap) against float64 sums and the entry with a workspace:
    positive terms, a thread adds B ceil(H W / 256) of them in a row, then six rounds of lanes and four waves."""
    from leniax_amd import core, engine, _lib
    print('direct adjoint without workspace', (B, C, maxk, H, W, kh, kw), flush=True)
    rng = np.random.default_rng(kh)
    K = C * maxk
    A = rng.uniform(size=(B, C, H, W)).astype(np.float32)
    kern = rng.uniform(size=(K, kh, kw)).astype(np.float32)
    dU = rng.uniform(size=(B, K, H, W)).astype(np.float32)
    rule = core._rule((H, W), C, K, [k // maxk for k in range(K)])
    tA, tk, tU = (torch.as_tensor(x).cuda() for x in (A, kern, dU))
    outs = []
    nb = ctypes.c_size_t(0)
    _lib.call('lx_potential_direct_adjoint_size', ctypes.byref(rule), B, kh, kw, ctypes.byref(nb))
    for work in (None, torch.empty(nb.value, dtype=torch.uint8, device='cuda')):
        dA, dk = torch.empty_like(tA), torch.empty_like(tk)
        args = [ctypes.byref(rule), engine.ptr(tA), B, engine.ptr(tk), kh, kw, engine.ptr(tU), engine.ptr(dA),
                engine.ptr(dk)]
        if work is None:
            _lib.call('lx_potential_direct_adjoint', *args, engine.stream_ptr())
        else:
            _lib.call('lx_potential_direct_adjoint_work', *args, engine.ptr(work), engine.stream_ptr())
        outs.append((dA.cpu().numpy(), dk.cpu().numpy()))
    assert np.array_equal(outs[0][0], outs[1][0])
    ref = _kernel_gradient(A, dU, kh, kw, maxk)
    bound = (B * -(-H * W // 256) + 10) * 2.0 ** -24
    assert float(np.max(np.abs(outs[0][1] - ref) / ref)) <= bound


DIRECT = ([(2, 1, 1, 17, 65, 7, 1), (1, 2, 2, 33, 70, 1, 2), (3, 1, 1, 40, 63, 64, 3), (1, 1, 1, 8, 8, 5, 4),
           (2, 1, 1, 64, 64, 5, 5)] +
          [(2, 1, 1, 50, 130, 3, kw) for kw in (6, 9, 12, 16, 17, 21, 25, 33, 37, 41, 48, 49, 64)] +
          [(64, 1, 1, 128, 128, 64, 64), (65, 1, 1, 100, 128, 53, 57)])


@pytest.mark.parametrize('B,C,maxk,H,W,kh,kw', DIRECT)
def test_direct_potential_by_width(B, C, maxk, H, W, kh, kw):
    """Kernels of 1 to 5 columns (direct_narrow_kernel), every split of the tap quads into groups, tiles beyond 64 KB of
    LDS: the potential and its state gradient against float64 correlations.  Every output is kh kw (times the
    kernels of a channel) multiply-adds of positive terms in a row."""
    from leniax_amd import core
    print('direct by width', (B, C, maxk, H, W, kh, kw), flush=True)
    rng = np.random.default_rng(kh * 100 + kw)
    A = rng.uniform(0.5, 1, size=(B, C, H, W)).astype(np.float32)
    K = rng.uniform(0.5, 1, size=(C * maxk, 1, kh, kw)).astype(np.float32)
    dU = rng.uniform(0.5, 1, size=(B, C * maxk, H, W)).astype(np.float32)
    pad = tuple([(0, 0), (0, 0)] + [(d // 2, d // 2 - 1) if d % 2 == 0 else (d // 2, d // 2) for d in (kh, kw)])
    tA = torch.as_tensor(A).cuda().requires_grad_()
    pot = core.get_potential(tA, torch.as_tensor(K).cuda(), pad)
    dA = torch.autograd.grad(pot, tA, torch.as_tensor(dU).cuda())[0].cpu().numpy()
    # U[y][x] = sum k[i][j] A[y + i - kh // 2][x + j - kw // 2], the kernel's taps past the world wrapped onto it
    taps = np.zeros((C * maxk, H, W))
    for i in range(kh):
        for j in range(kw):
            taps[:, (i - kh // 2) % H, (j - kw // 2) % W] += K[:, 0, i, j]
    spec = np.fft.rfft2(taps)
    U64 = np.fft.irfft2(np.fft.rfft2(np.repeat(A.astype(np.float64), maxk, 1)) * np.conj(spec), s=(H, W))
    A64 = np.fft.irfft2(np.fft.rfft2(dU.astype(np.float64)) * spec, s=(H, W)).reshape(B, C, maxk, H, W).sum(2)
    assert float(np.max(np.abs(pot.detach().cpu().numpy() - U64) / U64)) <= kh * kw * 2.0 ** -24
    assert float(np.max(np.abs(dA - A64) / A64)) <= kh * kw * maxk * 2.0 ** -24


def test_narrow_potential_of_a_state_that_is_not_finite():
    """Exactly the cells whose window holds the infinite cell are infinite."""
    from leniax_amd import core
    A = np.full((1, 1, 40, 80), 0.5, np.float32)
    A[0, 0, 7, 60] = np.inf
    pot = core.get_potential(torch.as_tensor(A).cuda(), torch.full((1, 1, 5, 4), 0.25).cuda(),
                             ((0, 0), (0, 0), (2, 2), (2, 1)))[0, 0].cpu().numpy()
    rows, cols = np.nonzero(~np.isfinite(pot))
    assert not np.isnan(pot).any()
    assert sorted(set(rows)) == list(range(5, 10)) and sorted(set(cols)) == list(range(59, 63)) and len(rows) == 20
    assert np.array_equal(pot[np.isfinite(pot)], np.full(3180, 20 * 0.125, np.float32))


@pytest.mark.parametrize('B,H,W,k', [(1, 40, 40, 5), (1, 52, 96, 32), (1, 64, 100, 9), (2, 167, 82, 25),
                                     (2, 195, 58, 18), (4, 42, 177, 19), (3, 159, 154, 8), (1, 128, 128, 40),
                                     (2, 256, 256, 13), (20, 86, 218, 7)])
def test_kernel_gradient_is_as_accurate_as_tap_by_tap(B, H, W, k):
    """The kernel gradient with a workspace is no further from float64 than one block per tap (the entry without one),
    whatever the number of cells: terms of both signs, so a sum's error goes with its longest chains of additions;
    a quarter of room for the sample of k^2 taps."""
    from leniax_amd import core, engine, _lib
    print('kernel gradient accuracy', (B, H, W, k), flush=True)
    rng = np.random.default_rng(k)
    A = rng.uniform(size=(B, 1, H, W)).astype(np.float32)
    dU = rng.normal(size=(B, 1, H, W)).astype(np.float32)
    rule = core._rule((H, W), 1, 1, [0])
    tA, tU, tk = torch.as_tensor(A).cuda(), torch.as_tensor(dU).cuda(), torch.zeros((1, k, k), device='cuda')
    nb = ctypes.c_size_t(0)
    _lib.call('lx_potential_direct_adjoint_size', ctypes.byref(rule), B, k, k, ctypes.byref(nb))
    work = torch.empty(nb.value, dtype=torch.uint8, device='cuda')
    ref = _kernel_gradient(A, dU, k, k, 1)
    errs = []
    for entry, tail in (('lx_potential_direct_adjoint', ()), ('lx_potential_direct_adjoint_work', (engine.ptr(work),))):
        dk = torch.empty_like(tk)
        _lib.call(entry, ctypes.byref(rule), engine.ptr(tA), B, engine.ptr(tk), k, k, engine.ptr(tU), None,
                  engine.ptr(dk), *tail, engine.stream_ptr())
        errs.append(float(np.linalg.norm(dk.cpu().numpy() - ref) / np.linalg.norm(ref)))
    print('  by tap, with a workspace', errs)
    assert errs[1] <= 1.25 * errs[0]
