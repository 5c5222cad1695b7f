"""A persistent slice loop whose barrier gives up: the call runs again by the
sweeps from its incident waves, with the bits of the sweeps, and the context's
later calls take the sweeps.  The limit of polls is set to one, so that a
barrier gives up unless every work-group has arrived at its first look; each
kernel still ends."""
import ctypes as C

import numpy as np
import pytest

import multislice_amd as msx

pytestmark = pytest.mark.gpu

N, NS, A, KEV = 256, 24, 25.6, 200.0


@pytest.fixture
def short():
    """A context whose loops give up."""
    c = msx.Context(0)
    fn = msx.load().msx_test_loop_polls
    fn.argtypes = [C.c_void_p, C.c_uint]
    assert fn(c.h, 1) == 0
    yield c
    c.close()


def gave_up_once(c):
    return c.loop_stats() == (c.loop_stats()[0], 1) and c.loop_stats()[0] >= 1


def trans(f64=False):
    import torch
    g = torch.Generator(device="cuda").manual_seed(5)
    ph = torch.rand((NS, N, N), generator=g, device="cuda", dtype=torch.float64 if f64 else torch.float32)
    return torch.polar(torch.ones_like(ph), ph)


CZ, LAYER = np.full(NS, 2.0), np.arange(NS)


@pytest.mark.parametrize("form", ["in place", "psi0 apart", "psi0 in psi", "host", "host psi0"])
@pytest.mark.parametrize("f64", [False, True])
def test_exit_waves(ctx, short, form, f64):
    import torch
    t = trans(f64)
    g = torch.Generator(device="cuda").manual_seed(7)
    first = torch.randn((2, N, N), dtype=t.dtype, device="cuda", generator=g)
    if form == "psi0 in psi":
        first = first[:1].clone()  # the only wave is its own incident wave

    def run(c):
        w = first.clone()
        if form == "in place":
            c.multislice(t, CZ, LAYER, w, A, A, KEV)
        elif form == "psi0 apart":
            c.multislice(t, CZ, LAYER, w, A, A, KEV, psi0=first[1].clone())
        elif form == "psi0 in psi":
            c.multislice(t, CZ, LAYER, w, A, A, KEV, psi0=w[0])
        else:
            w = w.cpu().numpy()
            c.multislice(t.cpu().numpy(), CZ, LAYER, w, A, A, KEV,
                         psi0=first[1].cpu().numpy() if form == "host psi0" else None)
            return w
        return w.cpu().numpy()
    ctx.set_graphs(True)  # the sweeps
    want = run(ctx)
    ctx.set_graphs(False)
    np.testing.assert_array_equal(run(short), want)
    assert gave_up_once(short)
    n = short.loop_stats()
    np.testing.assert_array_equal(run(short), want)
    assert short.loop_stats() == n


def test_stem(ctx, short):
    t = trans()
    pos = np.random.default_rng(0).uniform(0, A, (9, 2))
    args = (t, CZ, LAYER, A, A, KEV, dict(alpha_max=0.02), pos, [(0, 0.4), (1.0, 3.0)], [18, NS])
    ctx.set_graphs(True)
    want = ctx.stem(*args, batch=4)
    ctx.set_graphs(False)
    got = short.stem(*args, batch=4, weight=0.5, out=np.ones_like(want))
    np.testing.assert_array_equal(got, 1.0 + 0.5 * want)
    assert gave_up_once(short)


def test_partial_coherence(ctx, short):
    t = trans()
    args = (t, CZ, LAYER, A, A, KEV, dict(cs=1e7, df=500.0, aobj=0.02), 0.0, 3e-3, 30.0, 15.0)
    ctx.set_graphs(True)
    want = ctx.partial_coherence(*args, batch=8)[0]
    ctx.set_graphs(False)
    got = short.partial_coherence(*args, batch=8)[0]
    assert bool((got == want).all())
    assert gave_up_once(short)


@pytest.mark.parametrize("own", [False, True])
def test_job_set(ctx, short, own):
    import torch
    t = trans()
    g = torch.Generator(device="cuda").manual_seed(9)
    first = [torch.randn((N, N), dtype=t.dtype, device="cuda", generator=g) for _ in range(4)]

    def run(c):
        jobs = []
        for k, w in enumerate(first):
            j = dict(trans=t, psi=w.clone(), ax=A, by=A, kev=KEV, cz=CZ, layer=LAYER[:NS - 3 * k])
            if not own and k % 2:
                j["psi0"] = w
            jobs.append(j)
        c.multislice_batch(jobs)
        return [j["psi"].cpu().numpy() for j in jobs]
    ctx.profile(True)  # the sweeps
    want = run(ctx)
    ctx.profile(False)
    for a, b in zip(run(short), want):
        np.testing.assert_array_equal(a, b)
    assert gave_up_once(short)
