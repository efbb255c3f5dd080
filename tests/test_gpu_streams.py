"""Calls without a stream run on their engine's own stream: the memory of a dropped output goes
back to that stream, never to another engine's call while the first still writes it."""
import numpy as np
import pytest

from tests.synth import flat_weights, spectrum

pytestmark = pytest.mark.gpu


def test_outputs_belong_to_the_engines_stream():
    import torch
    from coffe_amd.engine import Batch, Engine
    k, p = spectrum(1024)
    sep = np.linspace(20.0, 200.0, 40)
    kt, pt = torch.tensor(k, device="cuda"), torch.tensor(p, device="cuda")
    A = torch.tensor(flat_weights([0, 2, 4], 1.5, 0.87, 0.6, 40), device="cuda")
    gout = torch.ones((1, 1, 3, 40), dtype=torch.float64, device="cuda")
    batches = [Batch(Engine(0), [1024], [1024], [k[0]], [k[-1]], [(0, 0), (0, 2), (0, 4)], sep, 1, 3) for _ in range(2)]
    want = [t.clone() for t in batches[0].vjp(kt, pt, A, gout)]
    for call in (lambda b: b.forward(kt, pt, A), lambda b: b.vjp(kt, pt, A, gout), lambda b: (b.tables_full(kt, pt),)):
        first = {t.data_ptr() for t in call(batches[0])}      # dropped at once, maybe still written
        assert not first & {t.data_ptr() for t in call(batches[1])}
    # results read on torch's default stream, between calls of the two engines
    for _ in range(20):
        got = batches[0].vjp(kt, pt, A, gout)
        batches[1].vjp(kt, 2.0 * pt, A, gout)
        again = batches[0].vjp(kt, pt, A, gout)
        for g, h, w in zip(got, again, want):
            assert torch.allclose(g, w, rtol=1e-12, atol=0) and torch.allclose(h, w, rtol=1e-12, atol=0)
    # on a stream of the caller's the outputs are that stream's
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = batches[0].vjp(kt, pt, A, gout)
    side.synchronize()
    for g, w in zip(got, want):
        assert torch.allclose(g, w, rtol=1e-12, atol=0)
    for b in batches:
        b.close()


def test_overlapping_passes_of_two_engines():
    """three forward + adjoint passes with nothing between them, the second on another engine's batch
    of other spectra and dropped at once, at the benchmark's size (256 ragged spectra, 512
    separations, 130 us a pass): the third pass' outputs are what a pass alone gives.  Its
    memory must not be that of the second pass, which may still be written: every element was at
    risk when both came from the default stream's pool (1e-12: the sums' order is the same)."""
    import torch
    from coffe_amd.engine import Batch, Engine
    from tests.synth import batch_spectra
    sep = np.linspace(5.0, 300.0, 512) / 0.67
    A = torch.tensor(flat_weights([0, 2, 4], 1.5, 0.87, 0.6, 512), device="cuda")
    sets = []
    for seed in (0, 1):
        specs = batch_spectra(256, seed=seed)
        n = [len(s[0]) for s in specs]
        b = Batch(Engine(0), n, n, [s[0][0] for s in specs], [s[0][-1] for s in specs], [(0, 0), (0, 2), (0, 4)], sep, 1, 3)
        rng = np.random.default_rng(seed)
        sets.append((b, torch.tensor(np.concatenate([s[0] for s in specs]), device="cuda"),
                     torch.tensor(np.concatenate([s[1] for s in specs]), device="cuda"), A,
                     torch.tensor(rng.standard_normal((256, 1, 3, 512)), device="cuda")))
    run = lambda s: s[0].vjp(*s[1:])  # noqa: E731
    want = [t.clone() for t in run(sets[0])]
    for _ in range(10):
        torch.cuda.synchronize()
        got = run(sets[0])
        run(sets[1])
        got = run(sets[0])
        torch.cuda.synchronize()
        for g, w in zip(got, want):
            assert float((g - w).norm()) <= 1e-12 * float(w.norm())
    for s in sets:
        s[0].close()


def test_outputs_by_the_context_manager():
    """the same outputs where the stream is switched by torch's context manager: allocated as the engine's, and
    the caller's stream and device stay current"""
    import torch
    from coffe_amd.engine import Batch, Engine
    k, p = spectrum(512)
    kt, pt = torch.tensor(k, device="cuda"), torch.tensor(p, device="cuda")
    eng = Engine(0)
    b = Batch(eng, [512], [512], [k[0]], [k[-1]], [(0, 0)], np.array([30.0, 60.0]), 1, 1)
    want = b.forward(kt, pt)[0].clone()
    by_ids, eng._switch = eng._switch, ()
    first = b.forward(kt, pt)[0]
    ptr = first.data_ptr()
    assert torch.equal(first, want)
    del first
    eng._switch = by_ids
    again = b.forward(kt, pt)[0]   # the block of the engine's pool that the other way gave back
    assert again.data_ptr() == ptr and torch.equal(again, want)
    assert torch.cuda.current_device() == 0 and torch.cuda.current_stream() == torch.cuda.default_stream()
    b.close()
    eng.close()
