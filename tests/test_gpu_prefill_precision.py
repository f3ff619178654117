"""Prefill attention's rounding on an MI355X: a query's output does not depend on the queries of the other 16-query half of
its workgroup, and where a workgroup sees few key tiles (windows, key splits) its largest probability is exact."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
CASES = [(0, 0, 1), (0, 0, 8), (256, 4, 1), (256, 0, 1)]   # window, sinks, key splits


def draw(n, heads, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(n, heads, 128, generator=g, device=DEV).to(torch.bfloat16)


def positions(S, T, window, nsink):
    """Key positions of T queries that end a row of S positions, as its layer keeps them."""
    lo = max(0, S - T - window + 1) if window else 0
    return np.concatenate([np.arange(min(nsink, lo)), np.arange(lo, S)]).astype(np.int32)


@pytest.mark.parametrize("window,nsink,splits", CASES)
@pytest.mark.parametrize("half", [0, 1])
def test_halves_apart(hip, window, nsink, splits, half):
    """Queries of 16 times the size outgrow their running maxima, which the other half's probabilities must not feel."""
    S, T = 2048, 64
    kp = positions(S, T, window, nsink)
    K, V, q = draw(len(kp), 4, 1), draw(len(kp), 4, 2), draw(T, 16, 3)
    own = torch.arange(T, device=DEV) // 16 % 2 == half
    big = torch.where(own[:, None, None], q, q * 16)
    print("[gpu-prefill-precision] halves", window, nsink, splits, half, flush=True)
    a, b = (hip.prefill(x, [0, T], [S - T], K, V, torch.from_numpy(kp).to(DEV), [0, len(kp)], window, nsink, splits)
            for x in (q, big))
    assert torch.equal(a[own].view(torch.int16), b[own].view(torch.int16))
    assert not torch.equal(a[~own], b[~own])


@pytest.mark.parametrize("window,nsink,splits", CASES[1:])
def test_largest_probability_exact(hip, window, nsink, splits):
    """Output errors beyond the output's own rounding, with values of one size. If every probability is rounded to bf16
    (8 bits: relative rms 2^-8 / sqrt(3) / 1.39 = 1.6e-3 over a binade) they come to about 1.45e-3 of the result; with the
    largest of each query exact, its share of the squares, here more than a third, is gone: below 1.2e-3."""
    S, T = 4096, 512 if window else 64
    kp = positions(S, T, window, nsink)
    K, V, q = draw(len(kp), 4, 4), draw(len(kp), 4, 5), 2 * draw(T, 16, 6)
    print("[gpu-prefill-precision] largest", window, nsink, splits, flush=True)
    out = hip.prefill(q, [0, T], [S - T], K, V, torch.from_numpy(kp).to(DEV), [0, len(kp)], window, nsink, splits).double()
    p, at = torch.from_numpy(kp).to(DEV)[None], torch.arange(S - T, S, device=DEV)[:, None]
    keep = p <= at
    if window:
        keep &= (p > at - window) | (p < nsink)
    want = torch.empty_like(out)
    for h in range(16):
        x = q[:, h].double() @ K[:, h // 4].double().T.contiguous() * 128 ** -0.5
        want[:, h] = torch.softmax(x.masked_fill(~keep, -torch.inf), -1) @ V[:, h // 4].double()
    square = lambda e: (e.norm() / want.norm()).item() ** 2
    beyond = square(out - want) - square(want.to(torch.bfloat16).double() - want)
    print("[gpu-prefill-precision] beyond the output's rounding: %.3e" % max(beyond, 0.0) ** 0.5, flush=True)
    assert beyond <= 1.2e-3 ** 2
