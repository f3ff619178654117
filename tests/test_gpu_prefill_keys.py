"""The one-launch key assembly of prefill rows on an MI355X (kv800_hip.window_keys, kv800_hip.prefill_keys), bit for bit
against plain torch gathers and the fp32 rotation rounded to bf16: rows around the window's and the copy tile's edges,
page sizes from one token up, sources that are not 16-byte aligned, rows without history or without new rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rotate(k, pos, cos, sin):
    """bf16 keys rotated on the dim pairs (d, d + 64), d < 32; positions past the tables clamped."""
    pos = pos.clamp(max=cos.shape[0] - 1)
    c = torch.cat([cos[pos].float(), torch.ones(len(pos), 32, device=DEV)], 1)[:, None]
    s = torch.cat([sin[pos].float(), torch.zeros(len(pos), 32, device=DEV)], 1)[:, None]
    lo, hi = k[..., :64].float(), k[..., 64:].float()
    return torch.cat([lo * c + (-hi) * s, hi * c + lo * s], -1).to(torch.bfloat16)


def same(a, b):
    return torch.equal(a.contiguous().view(torch.int16), b.contiguous().view(torch.int16))


def rows_of(prev, new, counts):
    from lfm3_kv800_amd import kv800_hip
    qsl = [sum(new[:i]) for i in range(len(new) + 1)]
    ksl = [sum(counts[:i]) + qsl[i] for i in range(len(new) + 1)]
    return kv800_hip.PrefillRows(qsl, ksl, prev, torch.device(DEV, 0))


@pytest.mark.parametrize("ebs,shift,sinks,rot", [(1, 0, True, True), (64, 0, False, False), (96, 4, True, True),
                                                 (128, 1, True, False)])
def test_window_keys(hip, ebs, shift, sinks, rot):
    import lfm3_kv800_amd.kv800 as kv
    g = torch.Generator(device=DEV).manual_seed(ebs)
    bf = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)
    prev, new = [0, 1, 255, 256, 257, 259, 700, 300], [5, 32, 0, 33, 1, 31, 64, 7]
    R, pages = len(prev), 700 // ebs + 2
    raw = bf(R * pages * 4 * ebs * 256 + 8)
    ev = raw[shift:shift + R * pages * 4 * ebs * 256].view(R * pages, 4, ebs, 256)
    eoff = torch.randperm(R * pages, generator=g, device=DEV).view(R, pages) * ev.stride(0)
    sk, sv, so = bf(R, 4, 4, 128), bf(R, 4, 4, 128), torch.randperm(R, generator=g, device=DEV) * 2048
    k, v = bf(sum(new), 4, 128), bf(sum(new), 4, 128)
    cos, sin = bf(720, 32), bf(720, 32)               # the longest rows run past the tables
    P = kv.Paged(epool=ev, eoff=eoff, ebs=ebs, e_hs=ev.stride(1), e_ts=ev.stride(2), e_v=128, sk=sk, sv=sv, skoff=so,
                 svoff=so)
    n = 4 if sinks else 0
    lo = [max(0, p - 255) for p in prev]
    rows = rows_of(prev, new, [p - a + min(n, a) for p, a in zip(prev, lo)])
    print("window_keys", ebs, shift, sinks, rot, flush=True)
    K, V, kp = hip.window_keys(P, rows, k, v, cos if rot else None, sin if rot else None, 256, n)
    for r in range(R):
        a, b = rows.qsl[r], rows.qsl[r + 1]
        pos = torch.arange(lo[r], prev[r], device=DEV)
        pg, sl = eoff[r, pos // ebs] // ev.stride(0), pos % ebs
        m, blk = min(n, lo[r]), so[r] // 2048
        want_k = torch.cat([sk[blk, :m], ev[pg, :, sl, :128], k[a:b]])
        want_v = torch.cat([sv[blk, :m], ev[pg, :, sl, 128:], v[a:b]])
        at = torch.cat([torch.arange(m, device=DEV), torch.arange(lo[r], prev[r] + new[r], device=DEV)])
        s = slice(rows.ksl[r], rows.ksl[r + 1])
        assert torch.equal(kp[s].long(), at), r
        assert same(V[s], want_v) and same(K[s], rotate(want_k, at, cos, sin) if rot else want_k), r


def test_prefill_keys_new_rows(hip):
    """History rows as kv800_hip.history writes them, then the new rows, rotated."""
    import lfm3_kv800_amd.kv800 as kv
    g = torch.Generator(device=DEV).manual_seed(5)
    bf = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)
    prev, new = [0, 700, 384, 31, 1000], [33, 1, 32, 0, 65]
    R, ebs, pages, nq = len(prev), 64, 17, [max(p - 128, 0) // 256 for p in prev]
    ev = bf(R * pages, 4, ebs, 256)
    eoff = torch.randperm(R * pages, generator=g, device=DEV).view(R, pages) * ev.stride(0)
    pool = hip.quantize_blocks(bf(8, 256, 4, 128), bf(8, 256, 4, 128))
    boff = torch.randint(0, 8, (R, 3), generator=g, device=DEV) * 51200
    P = kv.Paged(qpool=pool, boff=boff, epool=ev, eoff=eoff, ebs=ebs, e_hs=ev.stride(1), e_ts=ev.stride(2), e_v=128,
                 NQ=torch.tensor(nq, dtype=torch.int32, device=DEV))
    cos, sin = bf(1100, 32), bf(1100, 32)
    k, v = bf(sum(new), 4, 128), bf(sum(new), 4, 128)
    rows = rows_of(prev, new, prev)
    print("prefill_keys", flush=True)
    K, V = hip.prefill_keys(P, rows, k, v, cos, sin)
    hk, hv, offs = hip.history(P, prev, cos, sin)
    for r in range(R):
        a, b, o, s = rows.qsl[r], rows.qsl[r + 1], offs[r], rows.ksl[r]
        at = torch.arange(prev[r], prev[r] + new[r], device=DEV)
        assert same(K[s:s + prev[r]], hk[o:o + prev[r]]) and same(V[s:s + prev[r]], hv[o:o + prev[r]]), r
        assert same(K[s + prev[r]:rows.ksl[r + 1]], rotate(k[a:b], at, cos, sin)), r
        assert same(V[s + prev[r]:rows.ksl[r + 1]], v[a:b]), r


def test_window_keys_many_rows(hip):
    """More rows than the y extent of one grid."""
    import lfm3_kv800_amd.kv800 as kv
    R, ebs = 65535 + 5, 4
    g = torch.Generator(device=DEV).manual_seed(9)
    bf = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)
    prev = [r % 3 for r in range(R)]
    ev, page = bf(7, 4, ebs, 256), torch.randint(0, 7, (R, 1), generator=g, device=DEV)
    sk, sv, so = bf(3, 4, 4, 128), bf(3, 4, 4, 128), torch.randint(0, 3, (R,), generator=g, device=DEV)
    k, v, cos, sin = bf(R, 4, 128), bf(R, 4, 128), bf(8, 32), bf(8, 32)
    P = kv.Paged(epool=ev, eoff=page * ev.stride(0), ebs=ebs, e_hs=ev.stride(1), e_ts=ev.stride(2), e_v=128, sk=sk, sv=sv,
                 skoff=so * 2048, svoff=so * 2048)
    rows = rows_of(prev, [1] * R, hip.window_counts(prev, 2, 4))   # the last position, and position 0 as a sink before it
    print("window_keys", R, flush=True)
    K, V, kp = hip.window_keys(P, rows, k, v, cos, sin, 2, 4)
    p = torch.tensor(prev, device=DEV)
    at = torch.tensor(rows.ksl, device=DEV)
    new, old, sink = at[1:] - 1, at[1:][p > 0] - 2, at[:-1][p > 1]
    want_k, want_v = torch.empty_like(K), torch.empty_like(V)
    pos = torch.zeros(len(K), dtype=torch.int64, device=DEV)
    want_k[new], want_v[new], pos[new] = k, v, p
    last = ev[page[p > 0, 0], :, p[p > 0] - 1]
    want_k[old], want_v[old], pos[old] = last[..., :128], last[..., 128:], p[p > 0] - 1
    want_k[sink], want_v[sink] = sk[so[p > 1], 0], sv[so[p > 1], 0]
    assert torch.equal(kp.long(), pos) and same(V, want_v) and same(K, rotate(want_k, pos, cos, sin))


@pytest.mark.parametrize("rot", [True, False])
def test_history_negative_key_scales(hip, oracle, rot):
    """Sub-blocks written by hand with negative K scales and a lo of -0, which the quantizer never writes: a zero code times
    such a scale is -0, whose sign the rotation of the dims without a frequency (cos 1, sin 0) can change."""
    import numpy as np
    import lfm3_kv800_amd.kv800 as kv
    rng = np.random.default_rng(8)
    sb = rng.integers(0, 256, (2, 51200), dtype=np.uint8)
    scale = rng.choice(np.arange(0x20, 0x50, dtype=np.uint8), (2, 2048)).reshape(2, -1)
    scale[:, 512:1024] &= 0x7F                       # V scales
    scale[:, 1024:1536] = np.where(rng.random((2, 512)) < 0.5, 0x80, scale[:, 1024:1536])        # lo -0
    scale[:, 1536:] |= np.where(rng.random((2, 512)) < 0.5, np.uint8(0x80), np.uint8(0))
    sb[:, 49152:] = scale
    kb, vf = oracle.dequantize_blocks(sb)
    k = torch.from_numpy(kb.reshape(-1, 4, 128).view(np.int16)).view(torch.bfloat16).to(DEV)
    assert ((k == 0) & torch.signbit(k)).any()
    want_v = torch.from_numpy(vf.reshape(-1, 4, 128)).to(DEV).to(torch.bfloat16)
    g = torch.Generator(device=DEV).manual_seed(8)
    cos, sin = (torch.randn(512, 32, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    at = torch.arange(512, device=DEV)
    ev = torch.zeros(1, 4, 64, 256, dtype=torch.bfloat16, device=DEV)
    P = kv.Paged(qpool=torch.from_numpy(sb).to(DEV), boff=torch.tensor([[0, 51200]], device=DEV), epool=ev,
                 eoff=torch.zeros(1, 8, dtype=torch.int64, device=DEV), ebs=64, e_hs=ev.stride(1), e_ts=ev.stride(2), e_v=128,
                 NQ=torch.tensor([2], dtype=torch.int32, device=DEV))
    print("history negative scales", rot, flush=True)
    K, V, _ = hip.history(P, [512], *((cos, sin) if rot else ()))
    assert same(V, want_v) and same(K, rotate(k, at, cos, sin) if rot else k)
