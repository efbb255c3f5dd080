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
