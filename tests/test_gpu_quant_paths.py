"""The quantizer's branches on an MI355X, byte for byte against the oracle: K codes by per-channel thresholds (rounding
near zero, constant channels, infinities, NaN channels by the arithmetic per element), V by the bounded bf16 products and
by the exact chain (lattice values put outputs on the bit thresholds, tuned rows a few roundings beside them; wide ranges,
infinities and NaN leave no bound to settle by), dense and paged, in the throughput and the latency flush."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def dev(bits):
    return torch.from_numpy(np.ascontiguousarray(bits).view(np.int16)).view(torch.bfloat16).to(DEV)


def draw(kind, rng, shape):
    x = rng.standard_normal(shape)   # scales stay below fp8's largest value, 448
    if kind == "wide":
        x = x * np.exp2(rng.integers(-40, 4, shape))
    elif kind == "channels":
        x = x * np.exp2(rng.integers(-20, 5, (shape[0], 1, *shape[2:])))
    elif kind == "lattice":
        x = rng.integers(-6, 7, shape) * 0.25
    elif kind == "constant":
        x = np.broadcast_to(x[:, :1], shape) * 1.0
    elif kind == "positive":
        x = np.abs(x) + 0.25
    elif kind == "cancel":
        x[..., 64:] = -x[..., :64] * (1 + 2.0 ** -7)
    elif kind == "near_zero":
        x = np.where(rng.random(shape) < 0.5, x, x * np.exp(-40 * rng.random(shape)))
    elif kind == "tiny":
        x = x * 1e-39
    return x.astype(np.float32)


@pytest.mark.parametrize("kind", ["normal", "wide", "channels", "lattice", "constant", "positive", "cancel", "near_zero",
                                  "tiny"])
def test_quantize_kinds(hip, oracle, kind):
    rng = np.random.default_rng(len(kind))
    kb, vb = (oracle.f32_to_bf16(draw(kind, rng, (5, 256, 4, 128))) for _ in range(2))
    print("quantize", kind, flush=True)
    got = hip.quantize_blocks(dev(kb), dev(vb)).cpu().numpy()
    assert np.array_equal(got, oracle.quantize_blocks(kb, vb))


def test_quantize_nan_keys(hip, oracle):
    """A NaN key is no minimum or maximum and has code 0: the bytes of the same data with the channel's minimum there."""
    rng = np.random.default_rng(3)
    k = draw("normal", rng, (4, 256, 4, 128))
    holes = rng.random(k.shape) < 0.01
    holes[0] = False                                  # a sub-block without any
    kb, vb = oracle.f32_to_bf16(np.where(holes, np.inf, k)), oracle.f32_to_bf16(draw("normal", rng, k.shape))
    fill = oracle.f32_to_bf16(np.where(holes, np.inf, k).min(1, keepdims=True) + np.zeros_like(k))
    want = oracle.quantize_blocks(np.where(holes, fill, kb), vb)
    print("quantize NaN keys", flush=True)
    got = hip.quantize_blocks(dev(np.where(holes, np.uint16(0x7FC1), kb)), dev(vb)).cpu().numpy()
    assert np.array_equal(got, want)


@pytest.mark.parametrize("latency", [False, True])
@pytest.mark.parametrize("ebs", [64, 96, 640])
def test_flush_kinds(hip, oracle, ebs, latency):
    """Paged rows of every kind, one sub-block each, through both flushes."""
    kinds = ["normal", "lattice", "wide", "near_zero", "constant"]
    rng = np.random.default_rng(ebs)
    R, pages = len(kinds), -(-640 // ebs)
    kb, vb = (np.stack([oracle.f32_to_bf16(draw(k, rng, (1, 640, 4, 128)))[0] for k in kinds]) for _ in range(2))
    perm = rng.permutation(R * pages).reshape(R, pages)
    ev = np.zeros((R * pages, 4, ebs, 256), np.uint16)
    for r in range(R):
        for p in range(640):
            ev[perm[r, p // ebs], :, p % ebs, :128] = kb[r, p]
            ev[perm[r, p // ebs], :, p % ebs, 128:] = vb[r, p]
    e = dev(ev)
    eoff = torch.from_numpy(perm.astype(np.int64)).to(DEV) * e.stride(0)
    qbt = torch.arange(R, device=DEV).view(R, 1)
    j = torch.tensor([0, 1, 1, 0, 1], dtype=torch.int32, device=DEV)
    qv = torch.zeros(R, 262144, dtype=torch.uint8, device=DEV)
    print("flush", ebs, latency, flush=True)
    hip.flush(e, eoff, ebs, e.stride(1), e.stride(2), 128, qv, qbt, 1280, 262144, j, j + 1, 1, latency=latency)
    got, j = qv.cpu().numpy(), j.tolist()
    for r in range(R):
        s = slice(256 * j[r], 256 * j[r] + 256)
        want = oracle.quantize_blocks(kb[r, s][None], vb[r, s][None])[0]
        assert np.array_equal(got[r, j[r] * 51200:(j[r] + 1) * 51200], want), kinds[r]


@pytest.mark.parametrize("blocks,shift", [(1, 0), (3, 1), (2, 12)])
def test_dequantize_anywhere(hip, oracle, blocks, shift):
    """Sub-blocks at any byte of their storage."""
    rng = np.random.default_rng(shift)
    sb = oracle.quantize_blocks(*(oracle.f32_to_bf16(draw("normal", rng, (blocks, 256, 4, 128))) for _ in range(2)))
    raw = torch.zeros(blocks * 51200 + 16, dtype=torch.uint8, device=DEV)
    at = raw[shift:shift + blocks * 51200].view(blocks, 51200)
    at.copy_(torch.from_numpy(sb))
    print("dequantize", blocks, shift, flush=True)
    k, v = hip.dequantize_blocks(at)
    kw, vw = oracle.dequantize_blocks(sb)
    assert np.array_equal(k.cpu().view(torch.int16).numpy().view(np.uint16), kw)
    assert np.array_equal(v.cpu().numpy(), vw)


@pytest.mark.parametrize("tokens", [1, 3, 5, 33, 64])
def test_fake_quant_v_counts(hip, oracle, tokens):
    """Token counts around the groups of four and the waves' two groups."""
    v = draw("normal", np.random.default_rng(tokens), (tokens, 4, 128)) * np.float32(1.7)
    print("fake_quant_v", tokens, flush=True)
    assert np.array_equal(hip.fake_quant_v(torch.from_numpy(v).to(DEV)).cpu().numpy(), oracle.fake_quant_v(v))


@pytest.mark.parametrize("channels,shift", [(4, 0), (60, 0), (64, 0), (68, 0), (64, 1), (63, 0)])
def test_fake_quant_k_channels(hip, oracle, channels, shift):
    """Channel counts around the 64 of a workgroup, and tensors that are not 16-byte aligned (the per-channel kernel)."""
    x = draw("channels", np.random.default_rng(channels), (3, 256, 1, channels))[:, :, 0] * np.float32(1.3)
    raw = torch.zeros(x.size + 4, device=DEV)
    at = raw[shift:shift + x.size].view(x.shape)
    at.copy_(torch.from_numpy(x))
    print("fake_quant_k", channels, shift, flush=True)
    assert np.array_equal(hip.fake_quant_k(at).cpu().numpy(), oracle.fake_quant_k(x))


def by_every_kernel(hip, kb, vb):
    """The sub-blocks of (M, 256, 4, 128) bf16 bits by the dense kernel, the flush and the latency flush."""
    M, ebs = kb.shape[0], 64
    rows = dev(np.concatenate([kb, vb], -1)).view(M * 4, ebs, 4, 256).transpose(1, 2).contiguous()
    eoff = torch.arange(M * 4, device=DEV).view(M, 4) * rows.stride(0)
    yield "dense", hip.quantize_blocks(dev(kb), dev(vb)).cpu().numpy()
    for latency in (False, True):
        qv = torch.zeros(M, 262144, dtype=torch.uint8, device=DEV)
        j = torch.zeros(M, dtype=torch.int32, device=DEV)
        hip.flush(rows, eoff, ebs, rows.stride(1), rows.stride(2), 128, qv, torch.arange(M, device=DEV).view(M, 1), 1280,
                  262144, j, j + 1, 1, latency=latency)
        yield "latency" if latency else "flush", qv[:, :51200].cpu().numpy()


def fp8(x):
    """fp8 byte of a float32 array (past 448: 0x7F with the sign), and its value with the NaN bytes read as +-480."""
    with np.errstate(over="ignore"):
        b = torch.from_numpy(np.ascontiguousarray(x, np.float32)).to(torch.float8_e4m3fn)
    v = b.float().numpy()
    return b.view(torch.uint8).numpy(), np.where(np.isnan(v), np.copysign(np.float32(480), x), v).astype(np.float32)


@pytest.mark.parametrize("kind", ["+inf", "-inf", "inf", "inf and nan", "nan channels", "all nan", "large"])
def test_quantize_special_keys(hip, oracle, kind):
    """K's bytes for infinities, NaN and values past fp8's range, from the definition in float32: a NaN is no minimum or
    maximum and has code 0, a channel of NaN alone the range (inf, -inf), hence the scale of 1e-8."""
    rng = np.random.default_rng(11)
    k = draw("normal", rng, (3, 256, 4, 128))
    some = {"+inf": [np.inf], "-inf": [-np.inf], "inf": [np.inf, -np.inf], "inf and nan": [np.inf, -np.inf, np.nan]}
    if kind in some:
        k[rng.random(k.shape) < 0.003] = some[kind][0]
        for x in some[kind][1:]:
            k[rng.random(k.shape) < 0.003] = x
    elif kind == "nan channels":
        k[:, :, 1, 5] = k[:, :, 3, 100:] = np.nan
    elif kind == "all nan":
        k[:2] = np.nan
    else:
        k = k * np.float32(300)
    kb = np.where(np.isnan(k), np.uint16(0x7FC1), oracle.f32_to_bf16(np.where(np.isnan(k), 0, k)))
    k = np.where(np.isnan(k), np.nan, oracle.bf16_to_f32(np.where(np.isnan(k), 0, kb).astype(np.uint16)))
    vb = oracle.f32_to_bf16(draw("normal", rng, k.shape))
    with np.errstate(all="ignore"):
        lo, hi = np.fmin.reduce(k, 1), np.fmax.reduce(k, 1)
        lo, hi = np.where(np.isnan(lo), np.float32(np.inf), lo), np.where(np.isnan(hi), np.float32(-np.inf), hi)
        lo8, lof = fp8(lo)
        sc8, scf = fp8(np.maximum((hi - lo) / np.float32(3), np.float32(1e-8)))
        code = np.rint((k - lof[:, None]) / np.maximum(scf, np.float32(1e-8))[:, None])
    c = np.where(np.isnan(code), 0, np.clip(code, 0, 3)).astype(np.uint8)
    kc = c[..., :32] | c[..., 32:64] << 2 | c[..., 64:96] << 4 | c[..., 96:] << 6
    want = oracle.quantize_blocks(np.zeros_like(kb), vb)
    want[:, :32768], want[:, 50176:50688], want[:, 50688:] = (x.reshape(3, -1) for x in (kc, lo8, sc8))
    print("quantize special keys", kind, flush=True)
    for name, got in by_every_kernel(hip, kb, vb):
        assert np.array_equal(got, want), name


@pytest.mark.parametrize("kind", ["nan", "+inf", "-inf", "inf", "large"])
def test_quantize_special_values(hip, oracle, kind):
    """V rows with infinities, NaN or values whose transform leaves fp8's range, in one head of a pair: NaN outputs have bit
    0 and are no minimum or maximum, infinite or huge outputs of both signs give the scale bytes 0xFF and 0x7F, read as
    -480 and 480, so that every output above -240 has bit 1. All other bytes are the oracle's."""
    rng = np.random.default_rng(12)
    v = draw("normal", rng, (3, 256, 4, 128))
    for head in (0, 3):   # one special element in a row, past k = 0 (whose column of H has one sign)
        rows = np.argwhere(rng.random((3, 256)) < 0.2)
        for n, (m, t) in enumerate(rows):
            x = {"nan": np.nan, "+inf": np.inf, "-inf": -np.inf, "inf": np.inf, "large": 3.3e38}[kind]
            v[m, t, head, rng.integers(1, 128)] = x if n % 2 or kind != "large" else -x
            if kind == "inf":   # the other sign too: outputs inf, -inf and NaN
                v[m, t, head, rng.integers(1, 128)] = -np.inf
    vb = np.where(np.isnan(v), np.uint16(0x7FC1), oracle.f32_to_bf16(np.where(np.isnan(v), 0, v)))
    kb = oracle.f32_to_bf16(draw("normal", rng, v.shape))
    want = oracle.quantize_blocks(kb, vb)
    if kind != "nan":
        x = np.where(np.isnan(v), np.nan, oracle.bf16_to_f32(vb)).astype(np.float64)
        with np.errstate(all="ignore"):
            y = (x.reshape(-1, 128)[:, :, None] * oracle.hadamard().astype(np.float64)).sum(1).reshape(3, 256, 2, 256)
        special = ~(np.abs(y) < 480).all(-1)                       # (3, 256, 2): the pairs that hold such a row
        assert special.any() and (y[special].min(-1, where=~np.isnan(y[special]), initial=0) < -480).all()
        assert (y[special].max(-1, where=~np.isnan(y[special]), initial=0) > 480).all()
        bits = (y > -240).reshape(3, 256, 4, 8, 16)
        vbits = sum((bits[..., i, :].astype(np.uint8) << i) for i in range(8)).astype(np.uint8)   # (3, 256, 4, 16)
        heads = special.repeat(2, -1)
        body = want[:, 32768:49152].reshape(3, 256, 4, 16)
        body[heads] = vbits[heads]
        for at, byte in ((49152, 0xFF), (49664, 0x7F)):
            part = want[:, at:at + 512].reshape(3, 256, 2)
            part[special] = byte
    print("quantize special values", kind, flush=True)
    for name, got in by_every_kernel(hip, kb, vb):
        assert np.array_equal(got, want), name


@pytest.mark.parametrize("kind", ["one large", "two cancel", "wide", "denormal"])
def test_quantize_values_beside_thresholds(hip, oracle, kind):
    """Token pairs whose head 0 has an output within 60 x 2^-24 of its row's l1 of the pair's bit threshold, where the chain's
    128 roundings decide the bit: one large value among 127 of 2^-20 to 2^-28 of it, all of one sign at that output (the
    chain's and the matrix core's largest errors), two large values that cancel there, a wide range, denormals. Three
    elements place the output, the other head sets the pair's scales."""
    rng = np.random.default_rng(13)
    M, n = 8, 8 * 512
    r = np.arange(n)
    h = oracle.hadamard().astype(np.float64)
    bf = lambda x: oracle.bf16_to_f32(oracle.f32_to_bf16(np.asarray(x, np.float32))).astype(np.float64)
    sign = np.sign(h[:, rng.integers(0, 128, n)].T)                  # of each element at the row's output
    at = np.argsort(rng.random((n, 128)), 1)[:, :5]                  # the placing elements, and two more
    v = np.zeros((n, 2, 128))
    if kind == "wide":
        v[:, 0] = bf(rng.uniform(-1, 1, (n, 128)) * np.exp2(-rng.integers(2, 30, (n, 128))))
    elif kind == "denormal":
        v[:, 0] = bf(rng.uniform(-1, 1, (n, 128)) * 1e-39)
    else:
        v[:, 0] = sign * (rng.choice([-1, 1], n) * rng.choice([1.0078125, 1.5, 1.9921875], n) *
                          np.exp2(-rng.integers(20, 29, n)))[:, None]
    if kind == "two cancel":
        v[r, 0, at[:, 3]], v[r, 0, at[:, 4]] = sign[r, at[:, 3]], -sign[r, at[:, 4]]
    v[r, 1, 0] = bf(rng.uniform(2.5, 4, n))
    v[r, 0, at[:, 0]] = sign[r, at[:, 0]]
    kb = np.zeros((M, 256, 4, 128), np.uint16)
    quantize = lambda: oracle.quantize_blocks(kb, oracle.f32_to_bf16(v.astype(np.float32)).reshape(kb.shape))
    pair = lambda sb, a: oracle.f8_decode(sb[:, a:a + 512].reshape(-1)).astype(np.float64)
    threshold = lambda sb: (pair(sb, 49152) + pair(sb, 49664) / 2) / h[0, 0]
    for _ in range(4):   # the threshold may move with the placing elements
        goal = threshold(quantize()) + rng.integers(-60, 61, n) * 2.0 ** -24 * np.abs(v[:, 0]).sum(1)
        v[r[:, None], 0, at[:, :3]] = 0
        rest = goal - (v[:, 0] * sign).sum(1)
        for i in range(3):
            x = bf(rest)
            v[r, 0, at[:, i]], rest = x * sign[r, at[:, i]], rest - x
    want = quantize()
    d = ((v[:, 0] * sign).sum(1) - threshold(want)) / np.abs(v[:, 0]).sum(1) * 2.0 ** 24
    assert (np.abs(d) < 100).sum() > n // 8, "too few rows beside their threshold"
    if kind == "one large":   # the exact sum lies on the other side than the chain's: only the margin keeps these right
        chain = np.zeros(n)
        for k in range(128):
            chain = (chain + v[:, 0, k] * sign[:, k] * h[0, 0]).astype(np.float32).astype(np.float64)
        assert (((chain / h[0, 0] > threshold(want)) != (d > 0)) & (np.abs(d) < 100)).sum() > 50
    print("quantize values beside thresholds", kind, flush=True)
    for name, got in by_every_kernel(hip, kb, oracle.f32_to_bf16(v.astype(np.float32)).reshape(kb.shape)):
        assert np.array_equal(got, want), name
