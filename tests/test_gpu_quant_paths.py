"""The quantizer's branches on an MI355X, byte for byte against the oracle: K codes by per-channel thresholds (rounding
near zero, constant channels, NaN channels by the arithmetic per element), V by the bounded bf16 products and by the
exact chain (lattice values put outputs on the bit thresholds, wide ranges and infinities leave no bound to settle by),
dense and paged, in the throughput and the latency flush."""
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
