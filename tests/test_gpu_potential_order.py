"""Calls that share a model's workspaces, enqueued where a stream's handle does not
tell the streams apart or where the last user is the sampler itself: each gives
the bits that it gives alone.  And the chains that such a call may ask for."""
import threading

import numpy as np
import pytest
import torch

from numpyro_amd import _lib

pytestmark = pytest.mark.gpu

PER_THREAD = 2  # hipStreamPerThread: one handle, a stream of its own in every thread


def _engine(C=40, N=300000, D=24):
    from numpyro_amd.infer.hmc import Engine
    from numpyro_amd.models import LogisticRegression
    rng = np.random.default_rng(0)
    X = rng.normal(size=(N, D)).astype(np.float32)
    y = (rng.uniform(size=N) < 0.4).astype(np.float32)
    return Engine(LogisticRegression(X, y, kernel="tile"), C, "NUTS", 0)


def _positions(eng, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return 0.1 * torch.randn((n, eng.C, eng.D), generator=g, device="cuda")


def _out(eng):
    return (torch.empty(eng.C, dtype=torch.float64, device="cuda"),
            torch.empty((eng.C, eng.D), device="cuda"))


def _alone(eng, z):
    pe, g = _out(eng)
    torch.cuda.synchronize()
    _lib.check(eng.lib.nax_potential_grad(eng.h, _lib.ptr(z), eng.D, eng.C, _lib.ptr(pe),
                                          _lib.ptr(g)), "potential_grad")
    return pe, g


def _on(eng, z, out, stream):
    _lib.check(eng.lib.nax_potential_grad_on(eng.h, _lib.ptr(z), eng.D, eng.C, _lib.ptr(out[0]),
                                             _lib.ptr(out[1]), stream), "potential_grad_on")


def _in_threads(*work):
    failed = []

    def guarded(f):
        try:
            f()
        except BaseException as e:  # noqa: BLE001 - reported by the test
            failed.append(e)

    ts = [threading.Thread(target=guarded, args=(f,)) for f in work]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    assert not failed, failed


def test_threads_on_their_per_thread_streams():
    eng = _engine()
    zs = _positions(eng, 16, 1)
    want = [_alone(eng, z) for z in zs]
    got = [_out(eng) for _ in zs]
    torch.cuda.synchronize()

    def work(first):
        def f():
            for i in range(first, 16, 2):
                _on(eng, zs[i], got[i], PER_THREAD)
            # the device's synchronisation leaves out streams of threads that have ended
            torch.cuda.ExternalStream(PER_THREAD).synchronize()
        return f

    _in_threads(work(0), work(1))
    for (u, g), (wu, wg) in zip(got, want):
        assert torch.equal(u, wu) and torch.equal(g, wg)


def test_waiting_calls_beside_calls_on_a_stream():
    eng = _engine()
    zs = _positions(eng, 16, 2)
    want = [_alone(eng, z) for z in zs]
    got = [_out(eng) for _ in zs]
    side = torch.cuda.Stream()
    torch.cuda.synchronize()

    def on_stream():
        for i in range(0, 16, 2):
            _on(eng, zs[i], got[i], side.cuda_stream)

    def waiting():
        for i in range(1, 16, 2):
            _lib.check(eng.lib.nax_potential_grad(eng.h, _lib.ptr(zs[i]), eng.D, eng.C,
                                                  _lib.ptr(got[i][0]), _lib.ptr(got[i][1])),
                       "potential_grad")

    _in_threads(on_stream, waiting)
    for (u, g), (wu, wg) in zip(got, want):
        assert torch.equal(u, wu) and torch.equal(g, wg)


@pytest.mark.parametrize("degree", [0, 2])
def test_evaluations_around_a_gibbs_update(degree):
    """One stream's evaluation, the update of the subsamples, another stream's
    evaluation, with no wait between them: the first has the old subsamples, the
    second those that the update left."""
    from numpyro_amd.infer.hmc import Engine
    from numpyro_amd.models import SubsampledLogisticRegression
    rng = np.random.default_rng(3)
    N, D, m, C = 100000, 128, 2000, 512
    X = rng.normal(size=(N, D)).astype(np.float32)
    beta = 0.1 * rng.normal(size=D)
    y = (rng.uniform(size=N) < 1 / (1 + np.exp(-X @ beta))).astype(np.float32)
    model = SubsampledLogisticRegression(X, y, m, num_blocks=4, proxy_degree=degree,
                                         reference=beta if degree else None)
    model.idx = torch.as_tensor(rng.integers(0, N, (C, m)).astype(np.int32)).cuda()
    model.keys = torch.as_tensor(rng.integers(0, 2 ** 31, (C, 2)).astype(np.int32)).cuda()
    eng = Engine(model, C, "NUTS", 0)
    eng.init(torch.tensor(beta, dtype=torch.float32).expand(C, D).contiguous(),
             np.arange(2 * C, dtype=np.uint32).reshape(C, 2))
    zs = torch.tensor(beta, dtype=torch.float32, device="cuda") + 0.1 * _positions(eng, 2, 4)
    before = _alone(eng, zs[0])
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = [_out(eng) for _ in range(2)]
    idx = model.idx.clone()
    torch.cuda.synchronize()
    _on(eng, zs[0], got[0], streams[0].cuda_stream)
    _lib.check(eng.lib.nax_ecs_gibbs(eng.h, None), "gibbs")
    _on(eng, zs[1], got[1], streams[1].cuda_stream)
    torch.cuda.synchronize()
    after = _alone(eng, zs[1])
    assert not torch.equal(idx, model.idx)
    for (u, g), (wu, wg) in zip(got, (before, after)):
        assert torch.equal(u, wu) and torch.equal(g, wg)


@pytest.mark.parametrize("degree", [0, 2])
def test_more_chains_than_subsamples_are_refused(degree):
    from numpyro_amd.infer.hmc import Engine
    from numpyro_amd.models import SubsampledLogisticRegression, potential_energy
    X = np.random.default_rng(0).normal(size=(200, 3)).astype(np.float32)
    model = SubsampledLogisticRegression(X, np.zeros(200, np.float32), 10, proxy_degree=degree,
                                         reference=np.zeros(3) if degree else None)
    model.idx = torch.zeros((4, 10), dtype=torch.int32, device="cuda")
    model.keys = torch.zeros((4, 2), dtype=torch.int32, device="cuda")
    eng = Engine(model, 4, "NUTS", 0)
    z = torch.zeros((5, 3), device="cuda")
    pe, g = torch.zeros(5, dtype=torch.float64, device="cuda"), torch.zeros((5, 3), device="cuda")
    torch.cuda.synchronize()
    for call, tail in ((eng.lib.nax_potential_grad, ()), (eng.lib.nax_potential_grad_on, (None,))):
        args = (_lib.ptr(z), 3, 5, _lib.ptr(pe), _lib.ptr(g)) + tail
        assert call(eng.h, *args) != 0
    with pytest.raises(ValueError, match="subsamples of 4"):
        potential_energy(model, z)
    assert torch.isfinite(potential_energy(model, z[:4])).all()


def test_model_data_still_on_its_way_on_another_stream():
    from numpyro_amd.models import StochasticVolatility, potential_energy
    r = torch.randn(500, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda")
    z = 0.1 * torch.ones((3, 502), device="cuda")
    want = potential_energy(StochasticVolatility(r, noncentred=True), z)
    data, work = torch.cuda.Stream(), torch.cuda.Stream()
    late = torch.zeros_like(r)
    torch.cuda.synchronize()
    with torch.cuda.stream(data):
        torch.cuda._sleep(100_000_000)  # some tens of milliseconds
        late.copy_(r)
        model = StochasticVolatility(late, noncentred=True)
    with torch.cuda.stream(work):
        got = potential_energy(model, z)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
