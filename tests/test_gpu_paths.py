"""GPU tests of kernel variants and dispatch rules at the sizes where they
change: key-mask bits of the attention tiles and its split of the query heads."""
import struct
import subprocess
import sys

import numpy as np
import pytest

import oracle
from conftest import ROOT
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
@pytest.mark.parametrize("T,W", [(1, 128), (45, 128), (161, 128), (1000, 128), (130, 8), (12900, 128), (16500, 128),
                                 (9600, 16), (32000, 16), (24000, 32), (8320, 64)])
def test_attention_key_mask(be, T, W, hw_exp):
    """Masked runs that empty whole 32-key chunks, scattered masked keys and
    mask bytes other than 0 and 1, against the oracle with the tolerances of
    the unmasked test: fp16 outputs (2^-11) of the same arithmetic, and in the
    hardware-exp form one more fp16 rounding of the weights. Every tile (windows 8,
    16, 32, 64 and 128) and splits of the 7 heads into 1, 2 and more, with
    fewer workgroups than CUs (up to 12900 tokens at window 128) and more (16500)."""
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


# ---------------------------------------------------------------- int4 GEMM, split numerics

@pytest.mark.parametrize("x_f32", [True, False], ids=["f32", "fp16"])
@pytest.mark.parametrize("T,N,K,zp", [(1, 33, 128, 8), (31, 64, 640, None), (33, 96, 896, None), (70, 130, 384, 8),
                                      (65, 640, 1024, None), (4111, 72, 640, 8)])
def test_matmul_int4_chunked(be, T, N, K, zp, x_f32):
    """The K % 128 == 0 kernel: partial token and column tiles, odd, even and
    compile-time chunk counts, zero-points of every block and both activation
    forms. The f32 output against the oracle: both sum the
    same per-block products in f32, so the difference is a few f32 ulps of the
    largest partial sum (K / 32 blocks: 2^-23 sqrt(K / 32) relative, times 4), plus 2^-22 for the hi/lo split."""
    w = synth.qweight(1300 + K, N, K, zp=zp)
    x = synth.normal(1301 + T, T * K).astype(np.float32).reshape(T, K)
    xin = x if x_f32 else synth.to_fp16_bits(x).reshape(T, K)
    name = "matmul_int4_f32_f32" if x_f32 else "matmul_int4_fp16_f32"
    got = run(be, name, [xin, w["int4"], w["scales"], w["zp"], w["bias"]], T * N * 4, u32s(T, N, K, 0))
    ref = oracle.matmul(xin, w["int4"], w["scales"], w["zp"], w["bias"], N, K, x_f32=x_f32, out_f32=True)
    err = rel_err_norm(got.view(np.float32), ref.ravel())
    print(f"matmul T={T} N={N} K={K} zp={zp} x_f32={x_f32}: rel-err {err:.2e}")
    assert err < 4 * 2.0 ** -23 * np.sqrt(K / 32) + 2.0 ** -22


@pytest.mark.parametrize("x_f32", [True, False], ids=["f32", "fp16"])
@pytest.mark.parametrize("T,N,K", [(2432, 640, 896), (2433, 640, 896), (4544, 1152, 640), (4545, 1150, 640),
                                   (4545, 1152, 384), (40897, 97, 128), (40897, 160, 128)])
def test_matmul_int4_tile_rule(be, T, N, K, x_f32):
    """Each side of the lines of the dense tile rule on 256 CUs (64 x 64 for fp16 input
    from 2433 x 640, 64 x 128 for f32 from 4545 x 1152 and 40897 x 97, not where 160
    columns would be padded to 256), with partial tiles, even and odd chunk counts: the bits of
    the small tiles, which calls of at most 700 rows take."""
    w = synth.qweight(1320 + K, N, K)
    wb = [be.buffer(w[k]) for k in ("int4", "scales", "zp", "bias")]
    x = synth.normal(1321, T * K).astype(np.float32).reshape(T, K)
    x = x if x_f32 else synth.to_fp16_bits(x).reshape(T, K)
    for o, dt in (("f16", np.uint16), ("f32", np.uint32)):
        name = ("matmul_int4_f32_" if x_f32 else "matmul_int4_fp16_") + o
        got = []
        for rows in (T, 700):
            for i in range(0, T, rows):
                xb = be.buffer(np.ascontiguousarray(x[i:i + rows]))
                n = min(rows, T - i)
                out = be.buffer(nbytes=n * N * dt().nbytes)
                be.dispatch(name, [xb] + wb + [out], u32s(n, N, K, 0))
                got.append(out.read(dt).reshape(n, N))
                xb.release()
                out.release()
        assert np.array_equal(got[0], np.concatenate(got[1:])), name
    for b in wb:
        b.release()


@pytest.mark.parametrize("x_f32,N", [(True, 2052), (False, 4100)], ids=["f32", "fp16"])
def test_matmul_int4_grid_limit(x_f32, N):
    """Products whose small tiles (32 x 64 for 2052 columns, 64 x 64 for 4100) would be 2^24
    workgroups of 256 threads or more (a launch holds fewer than 2^32 threads) run on
    larger ones: 64 and 128 GiB of output, checked at the first, middle and last rows
    against a small call."""
    T, K, n = (1 << 24) - 1, 128, 40
    w = synth.qweight(1350, N, K)
    x = synth.normal(1351, 3 * n * K).astype(np.float32).reshape(3, n, K)
    x, name = (x, "matmul_int4_f32_f16") if x_f32 else (synth.to_fp16_bits(x).reshape(3, n, K), "matmul_int4_fp16_f16")
    row = x[0, 0].nbytes
    be = _native.Backend(0)  # its own: the scratch planes (8 GiB) go with it
    try:
        wb = [be.buffer(w[k]) for k in ("int4", "scales", "zp", "bias")]
        xb, out = be.buffer(nbytes=T * row), be.buffer(nbytes=T * N * 2)
        be.dispatch("zero_f32", [xb], u32s(T * row // 4, 0, 0, 0))
        at = [0, T // 2, T - n]
        for r, v in zip(at, x):
            xb.write(v, r * row)
        be.dispatch(name, [xb] + wb + [out], u32s(T, N, K, 0))
        for r, v in zip(at, x):
            ref = run(be, name, [v] + [w[k] for k in ("int4", "scales", "zp", "bias")], n * N * 2,
                      u32s(n, N, K, 0)).view(np.uint16)
            assert np.array_equal(out.read(np.uint16, n * N, r * N * 2), ref), r
        for b in wb + [xb, out]:
            b.release()
    finally:
        be.close()


@pytest.mark.parametrize("T", [100, 1025, 2049])
def test_moe_layer_split_expert_tiles(be, T):
    """The split MoE layer on the 16-, 32- and 64-row expert tiles (3, 32 and
    64 rows per expert on average) with partial tiles, against the oracle fed the
    GPU's routing: 32-bit sums rounded once to fp16 (2^-11)."""
    from textsift_amd.config import PF_CONFIG as cfg
    D, E, K, F = cfg.hidden_size, 128, 4, cfg.intermediate_size
    x = synth.normal(1400 + T, T * D).astype(np.float32)
    r = synth.qweight(1401, E, D)
    gu, dn = synth.qweight(1402, 2 * F, D, lead=(E,)), synth.qweight(1403, D, F, lead=(E,))
    bufs = [be.buffer(np.ascontiguousarray(a)) for a in
            [x] + [r[k] for k in ("int4", "scales", "zp", "bias")] +
            [q[k] for q in (gu, dn) for k in ("int4", "scales", "zp", "bias")]]
    outs = [be.buffer(nbytes=n) for n in (T * D * 2, T * K * 4, T * K * 4)]
    be.dispatch("moe_ffn", bufs + outs, u32s(T, D, E, K, F, 1, 1, 0))
    y = outs[0].read(np.uint16).reshape(T, D)
    ridx, rwt = outs[1].read(np.int32).reshape(T, K), outs[2].read(np.float32).reshape(T, K)
    for b in bufs + outs:
        b.release()
    w = {f"layers.0.experts.{n}.{k}": v for n, q in (("gate_up", gu), ("down", dn)) for k, v in q.items()}
    for nm in ("attn.q_proj", "attn.k_proj", "attn.v_proj", "attn.o_proj", "router"):
        w.update({f"layers.0.{nm}.{k}": v for k, v in synth.qweight(9, 64, 64).items()})
    w["layers.0.input_layernorm"] = w["layers.0.post_attention_layernorm"] = np.zeros(D, np.uint16)
    w["layers.0.attn.sinks"] = np.zeros(cfg.num_heads, np.float32)
    ref = oracle.expert_dispatch(cfg, w, 0, x.reshape(T, D), ridx, rwt * np.float32(0.25), n_slices=8)
    err = rel_err_norm(f16(y), f16(ref))
    print(f"split MoE T={T}: rel-err {err:.2e}")
    assert err < 2.0 ** -11


def test_moe_layer_split_matrix_of_2_gib(be):
    """An expert weight of 2^31 bytes is beyond the K % 128 == 0 kernel's
    buffer descriptor: the other kernel runs the 16- and 32-row plans too. A
    token's output depends on its row alone, so every plan tile gives the bits of the 64-row one."""
    D, E, K, F = 1024, 1, 1, 1 << 21
    rng = np.random.default_rng(1450)

    def weight(rows, cols, scale):
        return [np.frombuffer(rng.bytes(rows * cols // 2), np.uint8),
                synth.to_fp16_bits(np.full(rows * cols // 32, scale)),
                np.full(rows * cols // 64, 0x88, np.uint8), np.zeros(rows, np.uint16)]

    T = 80
    x = synth.to_fp16_bits(synth.normal(1451, T * D)).reshape(T, D)
    none = np.zeros(16, np.uint8)
    fixed = [be.buffer(a) for a in [synth.to_fp16_bits(synth.normal(1452, D * E)), none, none, np.zeros(8, np.uint16)] +
             weight(2 * F, D, 2.0 ** -7) + weight(D, F, 2.0 ** -10)]
    got = {}
    try:
        for n in (T, 40, 20):
            bufs = [be.buffer(x[:n])] + [be.buffer(nbytes=b) for b in (n * D * 2, n * K * 4, n * K * 4)]
            be.dispatch("moe_ffn", bufs[:1] + fixed + bufs[1:], u32s(n, D, E, K, F, 0, 0, 0))
            got[n] = bufs[1].read(np.uint16).reshape(n, D)
            for b in bufs:
                b.release()
    finally:
        for b in fixed:
            b.release()
    y = f16(got[T])
    assert np.all(np.isfinite(y)) and np.mean(y != 0) > 0.99
    for n in (40, 20):
        assert np.array_equal(got[n], got[T][:n]), n


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


# ---------------------------------------------------------------- fp16 GEMM tiles

def prepared(be, q, rows, K):
    src = [be.buffer(q[k]) for k in ("int4", "scales", "zp")]
    out = [be.buffer(nbytes=rows * K // 2), be.buffer(nbytes=rows * (K // 32) * 4)]
    be.dispatch("w4_prepare", src + out, u32s(rows, K, 1, 0))
    for b in src:
        b.release()
    return out + [be.buffer(q["bias"])]


@pytest.mark.parametrize("T,N,K", [(672, 1152, 640), (673, 1152, 640), (5440, 1152, 640), (5441, 1152, 640),
                                   (6528, 1152, 640), (6529, 1152, 640), (1216, 640, 896), (1217, 640, 896),
                                   (704, 1152, 640), (705, 1152, 640), (1280, 640, 896), (1281, 640, 896),
                                   (10240, 1152, 640), (10241, 1152, 640), (10241, 640, 896), (300, 72, 256)])
def test_matmul_w4_tile_rule(be, T, N, K):
    """The dense tile the library chooses gives the bits of the 64 x 64 tile: on
    each side of the first lines of its rule on 256 CUs (16 x 64, 64 x 128, 128 x 256 and
    back at N = 1152; 16 x 64 to 64 x 128 at K = 896), and at larger and odd sizes."""
    w = prepared(be, synth.qweight(1500 + N, N, K), N, K)
    x, out = be.buffer(synth.to_fp16_bits(synth.normal(1501, T * K))), be.buffer(nbytes=T * N * 2)
    got = []
    for tile, wf in ((0, 0), (64, 1)):
        be.dispatch("matmul_w4", [x] + w + [out], u32s(T, N, K, 0, tile, wf))
        got.append(out.read(np.uint16))
    for b in [x, out] + w:
        b.release()
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("T", [767, 768, 1535, 1536, 10239, 10240])
def test_moe_expert_tile_rule(be, T):
    """The expert tile on each side of every line of its rule (16, 32, 64 and
    128 rows) gives the bits of the 64 x 64 tile."""
    D, E, K, F = 640, 128, 4, 640
    rw, rb = synth.zipf_router(6, D, E)
    fixed = [be.buffer(np.ascontiguousarray(rw.T)), be.buffer(rb)] + \
        prepared(be, synth.qweight(1600, 2 * F, D, lead=(E,)), E * 2 * F, D) + \
        prepared(be, synth.qweight(1601, D, F, lead=(E,)), E * D, F)
    x = be.buffer(synth.to_fp16_bits(synth.normal(1602, T * D)))
    outs = [be.buffer(nbytes=n) for n in (T * D * 2, T * K * 4, T * K * 4)]
    got = []
    for tile, wf in ((0, 0), (64, 1)):
        be.dispatch("moe_ffn_w4", [x] + fixed + outs, u32s(T, D, E, K, F, tile, wf, 1))
        got.append(outs[0].read(np.uint16))
    with pytest.raises(_native.PfhipError):  # the 32-row tile is the library's own choice only
        be.dispatch("moe_ffn_w4", [x] + fixed + outs, u32s(T, D, E, K, F, 32, 2, 1))
    for b in [x] + fixed + outs:
        b.release()
    assert np.array_equal(got[0], got[1])


# ---------------------------------------------------------------- host-in / host-out staging

def test_host_forward_staging(be):
    """pfhip_model_forward through pinned staging (logits written by the
    classifier up to 64 KiB, by a copy kernel above) and through pageable copies
    (above 32 MiB of logits) gives the device-resident forward's bits, call after
    call with other ids, masks and sizes (a smaller call after a larger one
    included, and the captured and replayed forms)."""
    from textsift_amd.config import PF_CONFIG
    V, C = 512, PF_CONFIG.num_classes
    m = _native.Model(be, PF_CONFIG, num_layers=1, num_experts=8, vocab_size=V)
    for k, v in synth.make_model_weights(PF_CONFIG, seed=5, num_layers=1, num_experts=8, vocab_size=V).items():
        m.set_weight(k, v)
    m.finalize()
    edge = (64 << 10) // (4 * C)  # the largest direct call: 496 rows
    try:
        for i, (B, T, masked) in enumerate([(1, 5, True), (1, edge, False), (1, edge + 1, True), (3, 701, True),
                                            (1, 5, False), (1, 5, False), (1, 5, False), (125, 2048, True),
                                            (3, 701, True), (3, 701, True), (1, edge, False)]):
            n = B * T
            ids = synth.token_ids(1700 + i, n, V)
            mask = (synth.uniform(1800 + i, n) > 0.3).astype(np.uint8) if masked else np.ones(n, np.uint8)
            got = m.forward(ids, mask, B, T)
            ib, mb, lb = be.buffer(ids), be.buffer(mask), be.buffer(nbytes=n * C * 4)
            m.forward_device(ib, mb if masked else None, B, T, lb)
            ref = lb.read(np.float32)
            for b in (ib, mb, lb):
                b.release()
            assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (B, T, masked)
        for B, T in ((0, 5), (1, 0), (2049, 2048)):  # refused before any copy
            with pytest.raises(_native.PfhipError):
                m.forward(np.zeros(B * T, np.int32), None, B, T)
    finally:
        m.close()


# hipHostMalloc in front of the runtime's: the first `pass` calls go through, later ones report no memory
# (and record an error, which hipGetDevice(NULL) does here)
NO_PINNED = """
#include <dlfcn.h>
#include <stddef.h>
extern int hipGetDevice(int*);
int pass;
int hipHostMalloc(void** p, size_t n, unsigned flags) {
  static int (*real)(void**, size_t, unsigned);
  if (!real) {
    Dl_info info;
    dladdr((void*)&hipGetDevice, &info);
    real = (int (*)(void**, size_t, unsigned))dlsym(dlopen(info.dli_fname, RTLD_NOW), "hipHostMalloc");
  }
  if (pass-- > 0) return real(p, n, flags);
  hipGetDevice(NULL);
  return 2;
}
"""

NO_PINNED_RUN = """
import ctypes, sys
import numpy as np
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
passes = ctypes.c_int.in_dll(stub, "pass")
from textsift_amd import _native, synth
from textsift_amd.config import PF_CONFIG
V, C = 512, PF_CONFIG.num_classes
w = synth.make_model_weights(PF_CONFIG, seed=5, num_layers=1, num_experts=8, vocab_size=V)
be = _native.Backend(0)
for allowed in (0, 1, 2):  # none, the ids', the ids' and the logits' memory
    m = _native.Model(be, PF_CONFIG, num_layers=1, num_experts=8, vocab_size=V)
    for k, v in w.items():
        m.set_weight(k, v)
    m.finalize()
    passes.value = allowed
    for i, (B, T, masked) in enumerate([(1, 5, True), (1, 5, True), (1, 5, True), (2, 700, True), (1, 600, False)]):
        n = B * T
        ids = synth.token_ids(1900 + i, n, V)
        mask = (synth.uniform(1950 + i, n) > 0.3).astype(np.uint8) if masked else np.ones(n, np.uint8)
        got = m.forward(ids, mask, B, T)
        ib, mb, lb = be.buffer(ids), be.buffer(mask), be.buffer(nbytes=n * C * 4)
        m.forward_device(ib, mb if masked else None, B, T, lb)
        assert np.array_equal(got.view(np.uint32), lb.read(np.uint32)), (allowed, B, T)
        for b in (ib, mb, lb):
            b.release()
    assert passes.value < 0  # pinned memory was refused
    m.close()
be.close()
print("equal without pinned memory")
"""


def test_host_forward_without_pinned_memory(tmp_path):
    """Where pinned memory cannot be had (all of it, or only some of the three
    blocks) pfhip_model_forward copies pageable memory and gives the
    device-resident forward's bits."""
    src, so = tmp_path / "no_pinned.c", tmp_path / "no_pinned.so"
    src.write_text(NO_PINNED)
    subprocess.run(["gcc", "-shared", "-fPIC", "-D_GNU_SOURCE", str(src), "-o", str(so), "-L/opt/rocm/lib",
                    "-lamdhip64", "-ldl", "-Wl,-rpath,/opt/rocm/lib"], check=True)
    r = subprocess.run([sys.executable, "-c", NO_PINNED_RUN, str(so)], cwd=ROOT, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and "equal without pinned memory" in r.stdout, r.stdout + r.stderr


# ---------------------------------------------------------------- routing plan

@pytest.mark.parametrize("T,E,tile_rows", [(255, 128, 0), (256, 200, 0), (257, 128, 0), (1025, 128, 16), (4097, 37, 64),
                                           (16383, 128, 16), (16384, 128, 64), (1300, 128, 512), (1025, 256, 0),
                                           (65535, 64, 0), (65536, 64, 0)])
def test_routing_plan_block_sizes(be, T, E, tile_rows):
    """The plan on each side of its rules (256- and 1024-token blocks; tile_rows
    0: from the picks alone, in one, two or three kernels, else from tile counts):
    expert offsets, slots and tiles equal a stable sort by expert, bit for bit."""
    K, tt = 4, 64
    r = np.random.RandomState(T)
    idx = np.argsort(r.rand(T, E) * np.linspace(1, 3, E), axis=1)[:, :K].astype(np.int32)
    order = np.argsort(idx.ravel(), kind="stable")
    cnt = np.bincount(idx.ravel(), minlength=E)
    off = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32)
    slot_of = np.empty(T * K, np.int32)
    slot_of[order] = np.arange(T * K)
    tiles = [(e, off[e] + i, min(tt, cnt[e] - i), 0) for e in range(E) for i in range(0, cnt[e], tt)]
    ins = [be.buffer(idx)]
    if tile_rows:
        counts = np.stack([np.bincount(idx[i:i + tile_rows].ravel(), minlength=E) for i in range(0, T, tile_rows)])
        ins.append(be.buffer(counts.astype(np.int32)))
    outs = [be.buffer(nbytes=n) for n in ((E + 1) * 4, T * K * 4, T * K * 4, (T * K // tt + 1 + E) * 16, 4)]
    if tile_rows:
        be.dispatch("moe_route_counts", ins + outs, u32s(T, K, E, tt, tile_rows))
    else:
        be.dispatch("moe_route", ins + outs, u32s(T, K, E, tt))
    got = [o.read(np.int32) for o in outs]
    for b in ins + outs:
        b.release()
    assert np.array_equal(got[0], off) and np.array_equal(got[1], order // K) and np.array_equal(got[2], slot_of)
    assert got[4][0] == len(tiles) and np.array_equal(got[3][:4 * len(tiles)], np.array(tiles, np.int32).ravel())
