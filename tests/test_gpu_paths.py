"""GPU tests of kernel variants and dispatch rules at the sizes where they
change: key-mask bits of the attention tiles and its split of the query heads."""
import struct

import numpy as np
import pytest

import oracle
from parity_util import rel_err_norm
from textsift_amd import _native, synth

pytestmark = pytest.mark.gpu


def u32s(*vals):
    return np.array(vals, np.uint32).tobytes()


def f16(bits):
    return np.asarray(bits, np.uint16).view(np.float16).astype(np.float32)


@pytest.fixture(scope="module")
def be():
    b = _native.Backend(0)
    yield b
    b.close()


def run(be, name, inputs, out_bytes, pushb):
    """Dispatches with the inputs and one output binding at the end; returns the output's bytes."""
    bufs = [be.buffer(np.ascontiguousarray(a)) for a in inputs]
    out = be.buffer(nbytes=out_bytes)
    be.dispatch(name, bufs + [out], pushb)
    data = out.read(np.uint8)
    for b in bufs + [out]:
        b.release()
    return data


# ---------------------------------------------------------------- attention

@pytest.mark.parametrize("hw_exp", [0, 1], ids=["wasm-exp", "hw-exp"])
@pytest.mark.parametrize("T,W", [(1, 128), (45, 128), (161, 128), (1000, 128), (130, 8), (12900, 128)])
def test_attention_key_mask(be, T, W, hw_exp):
    """Masked runs that empty whole 32-key chunks, scattered masked keys and
    mask bytes other than 0 and 1, against the oracle with the tolerances of
    the unmasked test: fp16 outputs (2^-11) of the same arithmetic, and in the
    hardware-exp form one more fp16 rounding of the weights. 12900 tokens make
    more workgroups than CUs (one workgroup per KV head), the others split the heads."""
    Hq, Hkv, hd = 14, 2, 64
    q = synth.to_fp16_bits(synth.normal(900 + T, T * Hq * hd, 0, 0.35))
    k = synth.to_fp16_bits(synth.normal(901 + T, T * Hkv * hd, 0, 0.35))
    v = synth.to_fp16_bits(synth.normal(902 + T, T * Hkv * hd))
    snk = synth.normal(903, Hq).astype(np.float32)
    mask = (synth.uniform(904 + T, T) > 0.2).astype(np.uint8) * np.array([1, 2, 128, 255], np.uint8)[np.arange(T) % 4]
    mask[T // 3:T // 3 + 300] = 0   # whole chunks, and (W = 8) whole windows
    mask[2 * T // 3 + 10:] = 0      # padding at the end
    attn = oracle.banded_attention_wgsl if hw_exp else oracle.banded_attention
    ref = attn(q, k, v, snk, (mask != 0).astype(np.uint8), T, Hq, Hkv, hd, W)
    out = run(be, "banded_attention", [q, k, v, snk, mask], T * Hq * hd * 2,
              u32s(T, Hq, Hkv, hd, W, 1) + struct.pack("<f", 1.0) + u32s(hw_exp)).view(np.uint16).reshape(T, Hq * hd)
    zero = ~np.any(f16(ref), axis=1)  # rows whose every key is masked
    assert not np.any(f16(out)[zero])
    err, same = rel_err_norm(f16(out), f16(ref)), np.mean(out == ref)
    print(f"attention mask T={T} W={W} hw_exp={hw_exp}: rel-err {err:.3e}, identical {same:.4f}, {zero.sum()} empty rows")
    assert err < (5e-4 if hw_exp else 2e-3) and same > (0.5 if hw_exp else 0.97)


# ---------------------------------------------------------------- conversions

@pytest.mark.parametrize("scale", [1.0, 2.0 ** -14, 2.0 ** -24])
def test_fp16_narrowing_below_normal(be, scale):
    """fp16 narrowing with round-half-up below 2^-14: values around every
    subnormal's halfway points, signed zeros, the normal boundary, infinities and NaN, bit for bit."""
    n = np.arange(0, 1026, dtype=np.float64)
    v = np.concatenate([(n + d) * 2.0 ** -24 for d in (-0.5, -0.4999999, 0.0, 0.4999999, 0.5, 0.5000001)])
    v = np.concatenate([v, -v, [0.0, -0.0, 2.0 ** -26, 65504.0, 65519.0, 65520.0, np.inf, -np.inf, np.nan, 1e-40]])
    s = np.resize((v.astype(np.float32) / np.float32(scale)).astype(np.float32), 12800)
    got = run(be, "cast_f32_to_fp16_scaled", [s], s.size * 2,
              u32s(s.size, 0, 0, 0) + struct.pack("<f", scale) + u32s(0, 0, 0)).view(np.uint16)
    ref = oracle.f32_to_fp16(s * np.float32(scale))
    assert np.array_equal(got, np.asarray(ref, np.uint16))
