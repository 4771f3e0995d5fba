"""potential_energy in stream order (nax_potential_grad_on): the same bits as
the synchronous entry point on whatever stream, thread, layout or type z comes,
calls of several streams and threads behind one another, the sampler's own calls
behind them, and refused under graph capture as before."""
import threading

import numpy as np
import pytest
import torch

from numpyro_amd import _lib
from numpyro_amd.models import LogisticRegression, StochasticVolatility, potential_energy

pytestmark = pytest.mark.gpu


def _model(N=20000, D=24, seed=0):
    rng = np.random.default_rng(seed)
    X = rng.normal(size=(N, D)).astype(np.float32)
    y = (rng.uniform(size=N) < 0.4).astype(np.float32)
    return LogisticRegression(X, y, kernel="tile")


def _z(C, D, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return 0.1 * torch.randn((C, D), generator=g, device="cuda")


def _sync_eval(model, z):
    from numpyro_amd.infer.hmc import Engine
    C, D = z.shape
    eng = Engine(model, C, "NUTS", 0)
    pe = torch.empty(C, dtype=torch.float64, device="cuda")
    g = torch.empty((C, D), device="cuda")
    torch.cuda.synchronize()
    _lib.check(_lib.load().nax_potential_grad(eng.h, _lib.ptr(z), D, C, _lib.ptr(pe),
                                              _lib.ptr(g)), "potential_grad")
    return pe, g


def _grad(model, z):
    z = z.clone().requires_grad_(True)
    u = potential_energy(model, z)
    (g,) = torch.autograd.grad(u.sum(), z)
    return u.detach(), g


@pytest.mark.parametrize("C", [1, 5, 64])
def test_same_bits_for_any_layout_type_and_stream(C):
    model = _model()
    z = _z(C, 24, C)
    want_u, want_g = _sync_eval(model, z)
    wide = torch.zeros((C, 40), device="cuda")
    wide[:, 3:27] = z
    side = torch.cuda.Stream()
    for form in (z, wide[:, 3:27], z.T.contiguous().T, z.double()):
        u, g = _grad(model, form)
        assert torch.equal(u, want_u) and torch.equal(g.cuda().float(), want_g)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            u, g = _grad(model, form)
        torch.cuda.current_stream().wait_stream(side)
        assert torch.equal(u, want_u) and torch.equal(g.cuda().float(), want_g)
    assert torch.equal(potential_energy(model, z.cpu()), want_u)


def test_calls_of_two_streams_do_not_share_a_workspace_at_once():
    model = _model(N=300000)
    zs = [_z(40, 24, s) for s in range(8)]
    want = [_sync_eval(model, z) for z in zs]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    got = []
    for i, z in enumerate(zs):
        with torch.cuda.stream(streams[i % 2]):
            got.append(_grad(model, z))
    torch.cuda.synchronize()
    for (u, g), (wu, wg) in zip(got, want):
        assert torch.equal(u, wu) and torch.equal(g, wg)


def test_threads_and_the_samplers_own_calls():
    model = _model(N=300000)
    zs = [_z(40, 24, 10 + s) for s in range(4)]
    want = [_sync_eval(model, z) for z in zs]
    potential_energy(model, zs[0])  # the engine exists before the threads start
    torch.cuda.synchronize()
    got = [None] * 4

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            got[i] = _grad(model, zs[i])
        s.synchronize()

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for (u, g), (wu, wg) in zip(got, want):
        assert torch.equal(u, wu) and torch.equal(g, wg)
    # a call on the sampler's own stream right behind one on the caller's
    eng = model._vg_engines[40]
    pe = torch.empty(40, dtype=torch.float64, device="cuda")
    g = torch.empty((40, 24), device="cuda")
    torch.cuda.synchronize()
    u, _ = _grad(model, zs[0])
    _lib.check(_lib.load().nax_potential_grad(eng.h, _lib.ptr(zs[1]), 24, 40, _lib.ptr(pe),
                                              _lib.ptr(g)), "potential_grad")
    assert torch.equal(u, want[0][0]) and torch.equal(pe, want[1][0]) and torch.equal(g, want[1][1])


def test_refused_under_capture():
    model = StochasticVolatility(np.random.default_rng(0).normal(size=50).astype(np.float32))
    z = _z(4, 52, 1)
    potential_energy(model, z)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with pytest.raises(RuntimeError):
        with torch.cuda.graph(graph):
            potential_energy(model, z)
    torch.cuda.synchronize()
    u = potential_energy(model, z)  # and fine again afterwards
    assert torch.isfinite(u).all()
