"""Prefill attention over window + sink keys on an MI355X: the key tiles that hold sinks and window keys together, the
sink tile of its own behind 2^20 keys, and tiles that need no mask, against float64."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
# Per output with A = sum w |v|: the probabilities and the output are rounded to bf16, 2^-8 A and 2^-8 |want| (8 significant bits; the weights'
# sum is of unrounded ones); fp32 scores (products of up to 60, 128 of them: below 2^-24 x 128 x 60 / 11 = 4e-5 absolute),
# exponentials and sums stay below 1e-3 A together.
BF16, REST = 2.0 ** -8, 1e-3


def check(hip, q, K, V, kp, qsl, ksl, pos0, window, nsink, splits=None):
    given = None if kp is None else torch.from_numpy(kp).to(DEV)
    print("[gpu-prefill-window]", qsl, ksl, pos0, window, nsink, splits, flush=True)
    out = hip.prefill(q, qsl, pos0, K, V, given, ksl, window, nsink, splits)
    o = out.float().cpu().numpy().astype(np.float64)
    for r in range(len(pos0)):
        n = ksl[r + 1] - ksl[r]
        p = np.arange(n) if kp is None else kp[ksl[r]:ksl[r + 1]].astype(np.int64)
        qp = pos0[r] + np.arange(qsl[r + 1] - qsl[r])
        see = np.flatnonzero((p <= qp[-1]) & ((p > qp[0] - window) | (p < nsink)))
        at = torch.from_numpy(see + ksl[r]).to(DEV)
        k, v = (x[at].float().cpu().numpy().astype(np.float64).repeat(4, axis=1) for x in (K, V))
        qf = q[qsl[r]:qsl[r + 1]].float().cpu().numpy().astype(np.float64)
        sc = np.einsum("thd,shd->hts", qf, k) * 128 ** -0.5
        keep = (p[see] <= qp[:, None]) & ((p[see] > qp[:, None] - window) | (p[see] < nsink))
        sc = np.where(keep[None], sc, -np.inf)
        w = np.exp(sc - sc.max(-1, keepdims=True))
        w /= w.sum(-1, keepdims=True)
        want, size = np.einsum("hts,shd->thd", w, v), np.einsum("hts,shd->thd", w, np.abs(v))
        d = np.abs(o[qsl[r]:qsl[r + 1]] - want)
        assert (d <= BF16 * (size + np.abs(want)) + REST * size).all(), (r, d.max())


def draw(n, heads, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(n, heads, 128, generator=g, device=DEV).to(torch.bfloat16)


@pytest.mark.parametrize("nsink", [0, 1, 4, 63, 64, 65, 130])
@pytest.mark.parametrize("window", [1, 63, 256])
def test_window_tiles(hip, window, nsink):
    prev, new = [0, 3, 190, 700, 5000], [33, 70, 1, 64, 31]
    kps = []
    for p, t in zip(prev, new):   # the rows' keys as window layers keep them: sinks, then the window's positions
        lo = max(0, p - window + 1)
        kps.append(np.concatenate([np.arange(min(nsink, lo)), np.arange(lo, p + t)]))
    kp = np.concatenate(kps).astype(np.int32)
    ksl = [0, *np.cumsum([len(x) for x in kps]).tolist()]
    qsl = [0, *np.cumsum(new).tolist()]
    q, K, V = draw(qsl[-1], 16, 1), draw(ksl[-1], 4, 2), draw(ksl[-1], 4, 3)
    for splits in (1, 3):
        check(hip, q, K, V, kp, qsl, ksl, prev, window, nsink, splits)


@pytest.mark.parametrize("end", [1000, (1 << 20) + 250, (1 << 20) + 700])   # the window starts below / behind 2^20
def test_window_within_all_keys(hip, end):
    new, window, nsink = 40, 256, 70
    K, V = (torch.zeros(end, 4, 128, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    for x, s in ((K, 4), (V, 5)):
        x[:200], x[-600:] = draw(200, 4, s), draw(600, 4, s + 2)
    check(hip, draw(new, 16, 6), K, V, None, [0, new], [0, end], [end - new], window, nsink)
