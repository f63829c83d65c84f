// gemm_int4.hip — MatMulNBits int4 GEMM for gfx950 (fp16 MFMA, f32 accumulate).
//
// Computes out[t][n] = sum_b scale[n][b] * sum_{k in b} x[t][k] * (q[n][k] - zp[n][b]) + bias[n]
// over the ONNX MatMulNBits layout (uint4 packed two per byte along K, low
// nibble first; fp16 scales [N][K/32]; packed uint4 zero-points
// [N][ceil(K/64)], even block in the low nibble) — the semantics of
// matmulInt4BlockImpl, packages/textsift/src/zig/wasm_exports.zig:560-707.
//
// Mapping to CDNA4:
//  * One v_mfma_f32_16x16x32_f16 K-step is exactly one 32-wide quant block.
//    Weights enter the MFMA as the exact small integers (q - zp) in fp16, so
//    every product is exact; the block's f32 partial sum is then scaled with
//    one fmaf per accumulator, as the reference scales per block.
//  * The GEMM is computed transposed (D = W . X^T): the MFMA's M dimension
//    runs over weight rows, so each lane ends up holding 4 consecutive output
//    columns of one token. That makes the epilogues lane-local: RoPE pairs
//    (2p, 2p+1) and SwiGLU's interleaved (gate, up) columns sit in one lane,
//    and stores are 8-16 byte vectors.
//  * f32 activations (the WASM path feeds f32 to Q/K/V, router and experts,
//    browser/inference/block.ts:126-176) enter as an exact fp16 hi + lo pair
//    (two MFMAs into the same block partial), carrying 22 significant bits.
//  * Workgroup tile: 128 weight rows x BT tokens, K staged 64 at a time
//    through LDS (W dequantised once per workgroup, X split once), global
//    loads for the next stage issued before the current stage's MFMAs.
//  * Workgroup ids are remapped so each XCD walks a contiguous range of
//    (token tile, n tile) pairs: the n tiles of one token tile share an L2.
//  * Grouped mode: tiles come from a device list of (expert, row0, rows)
//    built by the MoE routing kernels; weights are offset per expert and
//    activation rows may be gathered through row_map.
#include "common.h"
#include "epilogue.h"
#include "pfhip_internal.h"
#include <type_traits>

namespace pf {

namespace {

constexpr int BN = 128;         // weight rows (output columns) per workgroup
constexpr int BK = 64;          // K per LDS stage = two quant blocks
constexpr int LDW = BK + 8;     // padded LDS row (halves)

// (1024 + a, 1024 + b) - (1024 + zp, 1024 + zp) on packed fp16: exact.
// Scalars only: __builtin_bit_cast applied to an ext-vector element (r.y)
// is lowered by this clang as a cast of the previously assigned element.
__device__ __forceinline__ uint32_t sub_zp(uint32_t v, h2_t off) {
  const h2_t h = __builtin_bit_cast(h2_t, v) - off;
  return __builtin_bit_cast(uint32_t, h);
}

// 8 nibbles of one dword -> 8 exact fp16 values (q - zp), natural k order.
__device__ __forceinline__ u4_t dequant8(uint32_t w, uint32_t zp_pair) {
  const uint32_t lo = w & 0x0F0F0F0Fu;          // k0 k2 k4 k6
  const uint32_t hi = (w >> 4) & 0x0F0F0F0Fu;   // k1 k3 k5 k7
  const h2_t off = __builtin_bit_cast(h2_t, zp_pair);  // (1024+zp, 1024+zp)
  const uint32_t p0 = __builtin_amdgcn_perm(hi, lo, 0x0C040C00u) | 0x64006400u;  // 1024+k0, 1024+k1
  const uint32_t p1 = __builtin_amdgcn_perm(hi, lo, 0x0C050C01u) | 0x64006400u;
  const uint32_t p2 = __builtin_amdgcn_perm(hi, lo, 0x0C060C02u) | 0x64006400u;
  const uint32_t p3 = __builtin_amdgcn_perm(hi, lo, 0x0C070C03u) | 0x64006400u;
  return u4_t{sub_zp(p0, off), sub_zp(p1, off), sub_zp(p2, off), sub_zp(p3, off)};
}

__device__ __forceinline__ int xcd_remap(int bid, int total) {
  const int xcd = bid & 7, idx = bid >> 3;
  const int per = total >> 3, rem = total & 7;
  return xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
}

template <int BT, bool SPLIT, Epi EPI, bool GROUPED>
__global__ __launch_bounds__(256) void k_gemm_int4(GemmArgs p) {
  constexpr int NPL = SPLIT ? 2 : 1;
  constexpr int WT = BT / 2;   // tokens per wave
  constexpr int WN = BN / 2;   // weight rows per wave
  constexpr int TI = WN / 16;  // n sub-tiles per wave
  constexpr int TJ = WT / 16;  // token sub-tiles per wave
  // X loader geometry: 8 x 16-byte chunks per row per plane per stage
  constexpr int XCH = 8;
  constexpr int XRP = 256 / XCH;                 // rows per pass
  constexpr int XPASS = BT / XRP;                // passes

  __shared__ __attribute__((aligned(16))) _Float16 Wl[BN * LDW];
  __shared__ __attribute__((aligned(16))) float Sl[2 * BN];
  __shared__ __attribute__((aligned(16))) _Float16 Xl[NPL * BT * LDW];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wn = (wave & 1) * WN;
  const int wt = (wave >> 1) * WT;
  const int l16 = lane & 15, lg = lane >> 4;

  const int n_tiles = (p.N + BN - 1) / BN;
  // grouped: the XCD remap over the workgroups that have tiles (the grid
  // covers the largest possible tile list)
  int active = (int)gridDim.x;
  if constexpr (GROUPED) {
    active = min(active, *p.num_tiles * n_tiles);
    if ((int)blockIdx.x >= active) return;
  }
  const int bid = xcd_remap(blockIdx.x, active);
  const int nt = bid % n_tiles;
  const int tt = bid / n_tiles;
  int expert = 0, row0, rows;
  if constexpr (GROUPED) {
    if (tt >= *p.num_tiles) return;
    const int4 ti = reinterpret_cast<const int4*>(p.tiles)[tt];
    expert = ti.x;
    row0 = ti.y;
    rows = ti.z;
  } else {
    row0 = tt * BT;
    rows = min(BT, p.M - row0);
    if (rows <= 0) return;
  }
  const int n0 = nt * BN;
  const int K = p.K;
  const int nb = K >> 5;
  const int zstride = (nb + 1) >> 1;
  const uint8_t* __restrict__ W = p.w + (size_t)expert * p.w_gs;
  const uint16_t* __restrict__ WS = p.ws + (size_t)expert * p.ws_gs;
  const uint8_t* __restrict__ WZ = p.wz ? p.wz + (size_t)expert * p.wz_gs : nullptr;

  // ---- loader roles
  const int wr = tid >> 1, wb = tid & 1;       // W: row, block within stage
  const int wrow = n0 + wr;
  const bool w_ok = wrow < p.N;
  const uint8_t* wsrc = W + (size_t)wrow * (K >> 1);

  const int xr = tid / XCH, xc = tid % XCH;
  int xoff[XPASS];                              // element offset of each X row, -1 = zero row
#pragma unroll
  for (int i = 0; i < XPASS; ++i) {
    const int r = xr + i * XRP;
    if (r < rows) {
      const int lr = row0 + r;
      const int g = p.row_map ? p.row_map[lr] : lr;
      xoff[i] = g * p.ldx;
    } else {
      xoff[i] = -1;
    }
  }

  // ---- prefetch registers: raw bytes only. Nothing loaded here is consumed
  // before store_stage, so the next stage's loads stay in flight across the
  // current stage's MFMAs (decoding a scale or zero-point here would make the
  // compiler wait for the load right away).
  u4_t wreg;
  uint32_t sraw;   // fp16 scale bits
  uint32_t zraw;   // zero-point byte (nibble selected in store_stage)
  bool wvalid;
  u4_t xreg[NPL][XPASS];
  const uint16_t* __restrict__ xhi = static_cast<const uint16_t*>(p.x);
  const uint16_t* __restrict__ xlo = p.x_lo;
  int kb_cur = 0;

  auto load_stage = [&](int s) {
    const int kb = s * 2 + wb;
    kb_cur = kb;
    wvalid = w_ok && kb < nb;
    if (wvalid) {
      wreg = *reinterpret_cast<const u4_t*>(wsrc + kb * 16);
      sraw = WS[(size_t)wrow * nb + kb];
      zraw = WZ ? (uint32_t)WZ[(size_t)wrow * zstride + (kb >> 1)] : 0u;
    }
#pragma unroll
    for (int i = 0; i < XPASS; ++i) {
      const int k = s * BK + xc * 8;
      if (xoff[i] >= 0 && k < K) {
        xreg[0][i] = *reinterpret_cast<const u4_t*>(xhi + xoff[i] + k);
        if constexpr (SPLIT) xreg[1][i] = *reinterpret_cast<const u4_t*>(xlo + xoff[i] + k);
      } else {
        xreg[0][i] = u4_t{0u, 0u, 0u, 0u};
        if constexpr (SPLIT) xreg[1][i] = u4_t{0u, 0u, 0u, 0u};
      }
    }
  };

  auto store_stage = [&]() {
    // W: 32 nibbles -> 32 exact fp16 at Wl[wr][wb*32 ...]; invalid rows /
    // blocks store q = 8 with zp = 8 (exact zeros) and scale 0.
    u4_t wq = u4_t{0x88888888u, 0x88888888u, 0x88888888u, 0x88888888u};
    uint32_t zp = 8;
    float sc = 0.0f;
    if (wvalid) {
      wq = wreg;
      sc = wasm_h2f((uint16_t)sraw);
      zp = WZ ? ((kb_cur & 1) ? (zraw >> 4) : (zraw & 0xFu)) : 0u;
    }
    const uint32_t hz = 0x6400u + zp;  // fp16 bits of 1024 + zp
    const uint32_t zreg = hz | (hz << 16);
    u4_t* wdst = reinterpret_cast<u4_t*>(&Wl[wr * LDW + wb * 32]);
    wdst[0] = dequant8(wq.x, zreg);
    wdst[1] = dequant8(wq.y, zreg);
    wdst[2] = dequant8(wq.z, zreg);
    wdst[3] = dequant8(wq.w, zreg);
    Sl[wb * BN + wr] = sc;
#pragma unroll
    for (int i = 0; i < XPASS; ++i) {
      const int r = xr + i * XRP;
#pragma unroll
      for (int pl = 0; pl < NPL; ++pl)
        *reinterpret_cast<u4_t*>(&Xl[pl * BT * LDW + r * LDW + xc * 8]) = xreg[pl][i];
    }
  };

  f4_t acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};

  const int S = (nb + 1) >> 1;
  load_stage(0);
  for (int s = 0; s < S; ++s) {
    if (s > 0) __syncthreads();
    store_stage();
    __syncthreads();
    if (s + 1 < S) load_stage(s + 1);
    const int nblk = min(2, nb - 2 * s);
    for (int b = 0; b < nblk; ++b) {
      h8_t wf[TI], xh[TJ], xl[TJ];
      f4_t sc[TI];
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        wf[i] = *reinterpret_cast<const h8_t*>(&Wl[(wn + 16 * i + l16) * LDW + b * 32 + 8 * lg]);
        sc[i] = *reinterpret_cast<const f4_t*>(&Sl[b * BN + wn + 16 * i + 4 * lg]);
      }
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        xh[j] = *reinterpret_cast<const h8_t*>(&Xl[(wt + 16 * j + l16) * LDW + b * 32 + 8 * lg]);
        if constexpr (SPLIT)
          xl[j] = *reinterpret_cast<const h8_t*>(&Xl[BT * LDW + (wt + 16 * j + l16) * LDW + b * 32 + 8 * lg]);
      }
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
          f4_t t = mfma16x16x32(wf[i], xh[j], f4_t{0.f, 0.f, 0.f, 0.f});
          if constexpr (SPLIT) t = mfma16x16x32(wf[i], xl[j], t);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][j][r] = fmaf(t[r], sc[i][r], acc[i][j][r]);
        }
    }
  }

  // ---- epilogue: lane holds out[token = wt+16j+l16][n = wn+16i+4lg+r]
  const uint16_t* __restrict__ BIAS = p.bias ? p.bias + (size_t)expert * p.bias_gs : nullptr;
#pragma unroll
  for (int i = 0; i < TI; ++i) {
    const int n = n0 + wn + 16 * i + 4 * lg;
    float bv[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) bv[r] = (BIAS && n + r < p.N) ? wasm_h2f(BIAS[n + r]) : 0.0f;
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      const int lt = wt + 16 * j + l16;
      if (lt >= rows) continue;
      const size_t orow = (size_t)(row0 + lt);
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = acc[i][j][r] + bv[r];
      int pos = 0;
      if constexpr (EPI == Epi::ROPE_F16) pos = (int)((uint32_t)orow % (uint32_t)p.seq_len);  // rows < 2^31
      store_out<EPI>(p, orow, n, v, pos);
    }
  }
}

template <int BT, bool SPLIT, Epi EPI, bool GROUPED>
void launch(pfhip_backend* b, const GemmArgs& a, const char* name) {
  const int n_tiles = (a.N + BN - 1) / BN;
  const int t_tiles = GROUPED ? a.max_tiles : (a.M + BT - 1) / BT;
  const long grid = (long)n_tiles * t_tiles;
  if (grid == 0) return;
  PF_CHECK(grid <= MAX_GRID_256, "gemm_int4: grid too large");
  ProfScope ps(b, name);
  hipLaunchKernelGGL((k_gemm_int4<BT, SPLIT, EPI, GROUPED>), dim3((unsigned)grid), dim3(256), 0, b->stream, a);
  PF_HIP(hipGetLastError());
}

// ---------------------------------------------------------------- K a multiple of 128
//
// The same product, scaled per block in the same order (bit-identical results), for K % 128 == 0, with the
// memory side rebuilt: the kernel above stages 64 K values per two barriers
// through registers, dequantises into LDS and has few workgroups.
//  * Weights are not staged: each of the 4 waves owns WF x 16 weight rows.
//    Lane (l16, lg) reads block lg of the chunk of row l16 as 16 bytes; a 4 x 4
//    transpose over the lane groups (two permlane swaps per pair of dwords)
//    leaves it dword lg of each block, its A fragment of that block's MFMA. A
//    wave's weights are dequantised once for all BT tokens.
//  * Activations go HBM -> LDS with global_load_lds (both planes), 128 K
//    values at a time, double buffered, in 256-byte rows whose 16-byte units
//    are XOR-swizzled by (row & 15): conflict-free fragment reads, one
//    barrier per 4 quant blocks.
//  * The lane's accumulator rows are 4 lg .. + 3 of a fragment, so the f32
//    scales of the chunk are kept in LDS as [block][row] and read as one
//    16-byte vector per fragment and block; each thread converts WF of them per chunk.
// 2048 x 1152 x 640 with the RoPE epilogue: 51.2 us in the kernel above, 21.5
// here; the 2048-token layer's gate_up and down 84 / 46 -> 65 / 32 us. Of that
// the 16-byte weight loads and their transpose (instead of four 4-byte loads) are
// a fifth, and the RoPE epilogue's branch-free subnormal path 4 us.
// Bound: per 16 x 16 x 32 block two MFMAs (32 cycles) and 4 fmaf (16), plus
// the dequantisation (17 VALU, 68 cycles) per fragment and BT tokens.
constexpr int KC = 128;  // K per chunk

//  * CT > 0 (K / 128 at compile time): weights are loaded two chunks ahead
//    and the barrier waits only for the activations, which are one ahead
//    (the L2 serves them; the weights come from HBM).
template <int WF, int BT, bool SPLIT, Epi EPI, bool GROUPED, int CT>
__global__ __launch_bounds__(256, 2) void k_gemm_int4_k128(GemmArgs p) {
  constexpr int NPL = SPLIT ? 2 : 1;
  constexpr int NW = 4, BNW = NW * WF * 16;  // weight rows per workgroup
  constexpr int TJ = BT / 16;
  constexpr int PLANE = BT * KC;             // halves per plane per buffer
  constexpr int XI = BT / (4 * NW);          // 4-row copies per wave and plane
  static_assert(BT % (4 * NW) == 0, "whole 4-row copies per wave");
  extern __shared__ __attribute__((aligned(16))) _Float16 xs[];  // [2][NPL][BT][KC], then f32 scales [2][4][BNW]
  float* sl = reinterpret_cast<float*>(xs + 2 * NPL * PLANE);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const int n_tiles = (p.N + BNW - 1) / BNW;
  int active = (int)gridDim.x;
  if constexpr (GROUPED) {
    active = min(active, *p.num_tiles * n_tiles);
    if ((int)blockIdx.x >= active) return;
  }
  const int bid = xcd_remap(blockIdx.x, active);
  const int nt = bid % n_tiles, tt = bid / n_tiles;
  int expert = 0, row0, rows;
  if constexpr (GROUPED) {
    const int4 ti = reinterpret_cast<const int4*>(p.tiles)[tt];
    expert = ti.x;
    row0 = ti.y;
    rows = ti.z;
  } else {
    row0 = tt * BT;
    rows = min(BT, p.M - row0);
  }
  const int n0 = nt * BNW, K = p.K, C = K / KC, nb = K >> 5;

  // Weights, zero-points and scales by buffer loads: one descriptor each in
  // scalar registers, 32-bit byte offsets per lane, the chunk in the scalar
  // offset (64-bit addresses per load spilled). Rows past N read row N - 1
  // (never stored). The host checks that one matrix stays below 2^31 bytes.
  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(p.w + (size_t)expert * p.w_gs), 0, p.N * (K >> 1), 0x00020000);
  const __amdgpu_buffer_rsrc_t srs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(p.ws + (size_t)expert * p.ws_gs), 0, p.N * nb * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t zrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(p.wz + (size_t)expert * p.wz_gs), 0, p.wz ? p.N * (nb >> 1) : 0, 0x00020000);
  uint32_t woff[WF], zoff[WF];  // (a chunk's 4 zero-point nibbles are 2 bytes of a row of nb / 2)
#pragma unroll
  for (int f = 0; f < WF; ++f) {
    const int n = min(n0 + (wave * WF + f) * 16 + l16, p.N - 1);
    woff[f] = (uint32_t)n * (uint32_t)(K >> 1) + lg * 16;
    zoff[f] = (uint32_t)n * (uint32_t)(nb >> 1);
  }
  // scales: thread tid converts WF consecutive blocks of row tid WF / 4
  const int srow = tid * WF / 4, sblk = tid * WF % 4;
  const uint32_t soff = ((uint32_t)min(n0 + srow, p.N - 1) * (uint32_t)nb + sblk) * 2u;
  const uint16_t* __restrict__ xsrc[NPL];
  xsrc[0] = static_cast<const uint16_t*>(p.x);
  if constexpr (SPLIT) xsrc[1] = p.x_lo;
  int xoff[XI];  // rows past the tile read its last row (never stored)
#pragma unroll
  for (int m = 0; m < XI; ++m) {
    const int r = (m * NW + wave) * 4 + lg;
    const int lr = row0 + min(r, rows - 1);
    const int g = p.row_map ? p.row_map[lr] : lr;
    xoff[m] = g * p.ldx + ((l16 ^ (r & 15)) << 3);
  }

  struct Wts {
    u4_t q[WF];
    uint32_t z[WF];
    uint32_t s;  // WF fp16 scales
  };
  // vector memory instructions of one chunk's weights
  constexpr int VM_W = 2 * WF + 1;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)xs;
  auto load_x = [&](int c, int buf) {
#pragma unroll
    for (int pl = 0; pl < NPL; ++pl)
#pragma unroll
      for (int m = 0; m < XI; ++m)
        copy16_to_lds_async(reinterpret_cast<const char*>(xsrc[pl]) + (uint32_t)(xoff[m] + c * KC) * 2u,
                            __builtin_amdgcn_readfirstlane(
                                lds0 + (uint32_t)((buf * NPL + pl) * PLANE + (m * NW + wave) * 512) * 2));
  };
  auto load_w = [&](int c, Wts& w) {
#pragma unroll
    for (int f = 0; f < WF; ++f) {
      w.q[f] = __builtin_amdgcn_raw_buffer_load_b128(wrs, woff[f], c * 64, 0);
      w.z[f] = __builtin_amdgcn_raw_buffer_load_b16(zrs, zoff[f], c * 2, 0);  // (0 without zero-points: out of range)
    }
    if constexpr (WF == 2) w.s = __builtin_amdgcn_raw_buffer_load_b32(srs, soff, c * 8, 0);
    else w.s = __builtin_amdgcn_raw_buffer_load_b16(srs, soff, c * 8, 0);
  };

  // the bias of the lane's 4 columns of each fragment, loaded here so the
  // epilogue does not wait for it (columns past N: unused values)
  const uint16_t* __restrict__ BIAS = p.bias ? p.bias + (size_t)expert * p.bias_gs : nullptr;
  int ncol[WF];
  uint16_t braw[WF][4];
#pragma unroll
  for (int f = 0; f < WF; ++f) {
    ncol[f] = n0 + (wave * WF + f) * 16 + 4 * lg;
#pragma unroll
    for (int r = 0; r < 4; ++r) braw[f][r] = BIAS ? BIAS[min(ncol[f] + r, p.N - 1)] : (uint16_t)0;
  }

  f4_t acc[WF][TJ];
#pragma unroll
  for (int f = 0; f < WF; ++f)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[f][j] = f4_t{0.f, 0.f, 0.f, 0.f};

  // One chunk = 4 blocks, software-pipelined: block j's MFMAs (hi for every
  // fragment pair, then lo onto them: independent chains) are issued with
  // block j + 1's fragment reads in flight, block j + 1's dequantisation and
  // block j - 1's scaling fmaf between them.
  // Chunk c: its weights' scales to LDS, the workgroup barrier (after it every
  // wave is done with the other activation buffer), the next loads, the MFMAs.
  // ahead: vector memory instructions issued after chunk c's activation copies.
  auto step = [&](int c, int buf, Wts& w, auto ahead, auto next) {
    constexpr int A = decltype(ahead)::value;
    static_assert(A < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt((A & 15) | (7 << 4) | (15 << 8) | ((A >> 4) << 14));
#pragma unroll
    for (int f = 0; f < WF; ++f) {
      // (landed: no further wait for them once newer loads are in flight)
      asm volatile("" : "+v"(w.q[f]), "+v"(w.z[f]));
      sl[(buf * 4 + sblk + f) * BNW + srow] = wasm_h2f((uint16_t)(w.s >> (16 * f)));
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    next();
    uint32_t wq[WF][4];  // block j's dword of this lane
#pragma unroll
    for (int f = 0; f < WF; ++f) {
      const uint32_t q0 = w.q[f][0], q1 = w.q[f][1], q2 = w.q[f][2], q3 = w.q[f][3];
      const auto a = __builtin_amdgcn_permlane16_swap(q0, q1, false, false);
      const auto b = __builtin_amdgcn_permlane16_swap(q2, q3, false, false);
      const auto e = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);
      const auto o = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
      wq[f][0] = e[0];
      wq[f][1] = o[0];
      wq[f][2] = e[1];
      wq[f][3] = o[1];
    }
    const _Float16* xb = xs + buf * NPL * PLANE;
    h8_t xf[2][NPL][TJ], wd[2][WF];
    f4_t sc[2][WF], d[2][WF][TJ];
    auto read = [&](int j) {
      const int unit = ((4 * j + lg) ^ l16) << 3;
#pragma unroll
      for (int t = 0; t < TJ; ++t)
#pragma unroll
        for (int pl = 0; pl < NPL; ++pl)
          xf[j & 1][pl][t] = *reinterpret_cast<const h8_t*>(xb + pl * PLANE + (16 * t + l16) * KC + unit);
#pragma unroll
      for (int f = 0; f < WF; ++f)
        sc[j & 1][f] = *reinterpret_cast<const f4_t*>(&sl[(buf * 4 + j) * BNW + (wave * WF + f) * 16 + 4 * lg]);
    };
    auto dequant = [&](int j) {
#pragma unroll
      for (int f = 0; f < WF; ++f) {
        const uint32_t hz = 0x6400u + ((w.z[f] >> (4 * j)) & 0xFu);  // fp16 bits of 1024 + zp
        wd[j & 1][f] = __builtin_bit_cast(h8_t, dequant8(wq[f][j], hz | (hz << 16)));
      }
    };
    auto scale = [&](int j, const f4_t (&s)[WF]) {
#pragma unroll
      for (int f = 0; f < WF; ++f)
#pragma unroll
        for (int t = 0; t < TJ; ++t) {
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[f][t][r] = fmaf(d[j & 1][f][t][r], s[f][r], acc[f][t][r]);
          // final here: the compiler otherwise moves every block's scaling to the chunk's end (spills)
          asm volatile("" : "+v"(acc[f][t]));
        }
    };
    read(0);
    dequant(0);
    f4_t sp[WF];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j > 0) {
#pragma unroll
        for (int f = 0; f < WF; ++f) sp[f] = sc[(j - 1) & 1][f];
      }
      if (j < 3) read(j + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < TJ; ++t)
#pragma unroll
        for (int f = 0; f < WF; ++f) d[j & 1][f][t] = mfma16x16x32(wd[j & 1][f], xf[j & 1][0][t], f4_t{0.f, 0.f, 0.f, 0.f});
      if constexpr (SPLIT) {
#pragma unroll
        for (int t = 0; t < TJ; ++t)
#pragma unroll
          for (int f = 0; f < WF; ++f) d[j & 1][f][t] = mfma16x16x32(wd[j & 1][f], xf[j & 1][NPL - 1][t], d[j & 1][f][t]);
      }
      if (j < 3) dequant(j + 1);
      if (j > 0) scale(j - 1, sp);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int f = 0; f < WF; ++f) sp[f] = sc[1][f];
    scale(3, sp);
  };
  using I0 = std::integral_constant<int, 0>;
  if constexpr (CT > 0) {
    Wts w[CT];  // three sets live at a time
    load_w(0, w[0]);
    load_x(0, 0);
    if constexpr (CT > 1) load_w(1, w[1]);
    auto chunks = [&](auto self, auto ci) {
      constexpr int c = decltype(ci)::value;
      step(c, c & 1, w[c], std::integral_constant<int, c + 1 < CT ? VM_W : 0>{}, [&]() {
        if constexpr (c + 1 < CT) load_x(c + 1, (c + 1) & 1);
        if constexpr (c + 2 < CT) load_w(c + 2, w[c + 2]);
      });
      if constexpr (c + 1 < CT) self(self, std::integral_constant<int, c + 1>{});
    };
    chunks(chunks, I0{});
  } else {
    Wts wa, wb;
    load_x(0, 0);
    load_w(0, wa);
    for (int c = 0; c < C; c += 2) {
      step(c, 0, wa, I0{}, [&]() {
        if (c + 1 < C) {
          load_x(c + 1, 1);
          load_w(c + 1, wb);
        }
      });
      if (c + 1 < C)
        step(c + 1, 1, wb, I0{}, [&]() {
          if (c + 2 < C) {
            load_x(c + 2, 0);
            load_w(c + 2, wa);
          }
        });
    }
  }

  // ---- epilogue: lane holds out[token 16 t + l16][n = n0 + (wave WF + f) 16 + 4 lg + r]
  // RoPE: the lane's (cos, sin) entries, every load issued before the first use
  [[maybe_unused]] f2_t cs[WF][TJ], sn[WF][TJ];
  if constexpr (EPI == Epi::ROPE_F16) {
#pragma unroll
    for (int t = 0; t < TJ; ++t) {
      const uint32_t pos = (uint32_t)(row0 + min(16 * t + l16, rows - 1)) % (uint32_t)p.seq_len;  // rows < 2^31
#pragma unroll
      for (int f = 0; f < WF; ++f) {
        const uint32_t at = pos * 32 + ((ncol[f] & 63) >> 1);
        cs[f][t] = *reinterpret_cast<const f2_t*>(p.rope_cos + at);
        sn[f][t] = *reinterpret_cast<const f2_t*>(p.rope_sin + at);
      }
    }
  }
#pragma unroll
  for (int f = 0; f < WF; ++f) {
    const int n = ncol[f];
    if (n >= p.N) continue;
    float bv[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) bv[r] = n + r < p.N ? wasm_h2f(braw[f][r]) : 0.0f;
#pragma unroll
    for (int t = 0; t < TJ; ++t) {
      const int lt = 16 * t + l16;
      if (lt >= rows) continue;
      const size_t orow = (size_t)(row0 + lt);
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = acc[f][t][r] + bv[r];
      if constexpr (EPI == Epi::ROPE_F16) {
        store_f16x4(p, orow, n, n < p.rope_cols ? rope_f16x4(v, cs[f][t], sn[f][t]) : to_f16x4(v));
      } else {
        store_out<EPI>(p, orow, n, v);
      }
    }
  }
}

// false: more workgroups than a launch holds (the larger tiles of the kernel above may still fit)
template <int WF, int BT, bool SPLIT, Epi EPI, bool GROUPED, int CT>
bool launch_k128_ct(pfhip_backend* b, const GemmArgs& a, const char* name) {
  constexpr int BNW = 64 * WF;
  const int t_tiles = GROUPED ? a.max_tiles : (a.M + BT - 1) / BT;
  const long grid = (long)((a.N + BNW - 1) / BNW) * t_tiles;
  if (grid == 0) return true;
  if (grid > MAX_GRID_256) return false;
  const size_t lds = (size_t)2 * (SPLIT ? 2 : 1) * BT * KC * 2 + (size_t)2 * 4 * BNW * 4;
  const auto kern = &k_gemm_int4_k128<WF, BT, SPLIT, EPI, GROUPED, CT>;
  allow_lds(reinterpret_cast<const void*>(kern), lds);
  ProfScope ps(b, name);
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), lds, b->stream, a);
  PF_HIP(hipGetLastError());
  return true;
}

// K = 640 (the model's width) is built with its chunk count, others loop.
template <int WF, int BT, bool SPLIT, Epi EPI, bool GROUPED>
bool launch_k128(pfhip_backend* b, const GemmArgs& a, const char* name) {
  if (a.K == 5 * KC) return launch_k128_ct<WF, BT, SPLIT, EPI, GROUPED, 5>(b, a, name);
  if constexpr (!GROUPED && !SPLIT && EPI == Epi::F16)
    if (a.K == 7 * KC) return launch_k128_ct<WF, BT, SPLIT, EPI, GROUPED, 7>(b, a, name);
  return launch_k128_ct<WF, BT, SPLIT, EPI, GROUPED, 0>(b, a, name);
}

// The tiles below, for the forms that the split forward and the named
// products use; false: not built, or too many workgroups (the kernel above takes them).
// Dense: 32 tokens x 64 columns while the tiles are few. Above 1.5 64 x 64 tiles per
// CU, 64 x 64 for one fp16 plane; from 2.5 64 x 128 tiles per CU on, 64 x 128 for
// split planes, unless 128 columns pad N by over an eighth more than 64 do. A tile of
// twice the size dequantises (64 tokens) and reads activations (128 columns) half as
// often, which counts once every CU has several to run; the line by rows (4096,
// fp16 only) before this one left 9000 x 8192 x 512 behind the kernel above. Over 938
// products every choice is ahead of the kernel above; the larger tile is up to 3 % behind 32 x 64
// for split planes and 5 % for one (1602 x 1280 x 640, just above two rounds).
// us on the kernel above / 32 x 64 / 64 x 64 / 64 x 128 (events around the call: 15 to 20 us
// more than the kernel; split with the f32 -> hi + lo pass):
//   fp16   1290 x 1152 x 640  52.1 / 30.4 / 30.8 / -        1400 x 1152 x 640  52.4 / 32.9 / 31.2 / 33.4
//          4095 x 4096 x 1024  169.7 / 174.1 / 141.2 / 139.9   20000 x 1152 x 640  168.8 / 153.8 / 126.9 / 134.7
//   split  3622 x 1152 x 640  110.6 / 80.7 / - / 83.1       4908 x 1152 x 640  122.5 / 97.1 / - / 92.6
//          9000 x 8192 x 512  529.8 / 542.6 / 546.0 / 441.2   20000 x 1152 x 640  265.9 / 249.6 / 250.8 / 211.1
// With the RoPE epilogue 32 x 64 at every size (2048 x 1152 x 640: 21.7 us, against 24.4 with
// 64 x 64 and 34.7 with 64 x 128; 32768 rows: 207, 232 and 207).
// Grouped: the expert plan's tile. 16 and 32 rows take 64 columns, 64 rows 128 (gate_up
// over 13.6 rows per expert: 26.6 / 30.0 / 41.0 us on tiles of 16 / 32 / 64
// rows; over 64: 75.7 / 66.3 / 66.3; over 256: 281 / 227 / 197).
bool dispatch_k128(pfhip_backend* b, const GemmArgs& a, bool split, Epi epi, bool grouped, int tile_t,
                   const char* name) {
  if (grouped) {
    auto tile = [&](auto wf, auto bt) {
      constexpr int WF = decltype(wf)::value, BT = decltype(bt)::value;
      if (epi == Epi::SWIGLU_SPLIT) {
        if (split) return launch_k128<WF, BT, true, Epi::SWIGLU_SPLIT, true>(b, a, name);
        return launch_k128<WF, BT, false, Epi::SWIGLU_SPLIT, true>(b, a, name);
      }
      if (epi == Epi::F32 && split) return launch_k128<WF, BT, true, Epi::F32, true>(b, a, name);
      return false;
    };
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    if (tile_t == 16) return tile(I1{}, std::integral_constant<int, 16>{});
    if (tile_t == 32) return tile(I1{}, std::integral_constant<int, 32>{});
    if (tile_t == 64) return tile(I2{}, std::integral_constant<int, 64>{});
    return false;
  }
  const auto up = [](long n, long d) { return (n + d - 1) / d; };
  const long rows64 = up(a.M, 64), cols64 = up(a.N, 64), cols128 = up(a.N, 128);
  const bool large = split ? 2 * rows64 * cols128 >= 5L * b->num_cus && 16 * cols128 <= 9 * cols64
                           : 2 * rows64 * cols64 > 3L * b->num_cus;
  switch (epi) {
    case Epi::F16:
      if (split && large) return launch_k128<2, 64, true, Epi::F16, false>(b, a, name);
      if (split) return launch_k128<1, 32, true, Epi::F16, false>(b, a, name);
      if (large) return launch_k128<1, 64, false, Epi::F16, false>(b, a, name);
      return launch_k128<1, 32, false, Epi::F16, false>(b, a, name);
    case Epi::F32:
      if (split && large) return launch_k128<2, 64, true, Epi::F32, false>(b, a, name);
      if (split) return launch_k128<1, 32, true, Epi::F32, false>(b, a, name);
      if (large) return launch_k128<1, 64, false, Epi::F32, false>(b, a, name);
      return launch_k128<1, 32, false, Epi::F32, false>(b, a, name);
    case Epi::ROPE_F16:
      return split && launch_k128<1, 32, true, Epi::ROPE_F16, false>(b, a, name);
    default: return false;
  }
}

template <int BT, bool SPLIT, bool GROUPED>
void dispatch_epi(pfhip_backend* b, const GemmArgs& a, Epi epi, const char* name) {
  switch (epi) {
    case Epi::F16: return launch<BT, SPLIT, Epi::F16, GROUPED>(b, a, name);
    case Epi::F32: return launch<BT, SPLIT, Epi::F32, GROUPED>(b, a, name);
    case Epi::ROPE_F16: return launch<BT, SPLIT, Epi::ROPE_F16, GROUPED>(b, a, name);
    case Epi::SWIGLU_SPLIT: return launch<BT, SPLIT, Epi::SWIGLU_SPLIT, GROUPED>(b, a, name);
    case Epi::SWIGLU_F16: return launch<BT, SPLIT, Epi::SWIGLU_F16, GROUPED>(b, a, name);
    case Epi::F32_TOPK: break;
  }
  throw Error("gemm_int4: unsupported epilogue");
}

}  // namespace

void gemm_int4(pfhip_backend* b, const GemmArgs& a, XKind xk, Epi epi, bool grouped, int tile_t,
               const char* prof_name) {
  PF_CHECK(a.K > 0 && a.K % 32 == 0, "gemm_int4: K must be a positive multiple of 32");
  PF_CHECK(a.N > 0, "gemm_int4: N must be positive");
  PF_CHECK(a.x && a.w && a.ws && (a.out || a.out_f32w), "gemm_int4: null operand");
  if (a.out_f32w) PF_CHECK(epi == Epi::F16 && !grouped, "gemm_int4: the widened f32 output is for the dense F16 epilogue");
  PF_CHECK(a.ldx % 8 == 0 && a.K % 8 == 0, "gemm_int4: activation row stride must allow 16-byte loads");
  PF_CHECK((reinterpret_cast<uintptr_t>(a.x) & 15) == 0 && (reinterpret_cast<uintptr_t>(a.w) & 15) == 0,
           "gemm_int4: activations and weights must be 16-byte aligned");
  if (xk == XKind::SPLIT)
    PF_CHECK(a.x_lo && (reinterpret_cast<uintptr_t>(a.x_lo) & 15) == 0, "gemm_int4: SPLIT needs an aligned lo plane");
  PF_CHECK(a.K / 2 % 16 == 0, "gemm_int4: packed weight rows must be 16-byte multiples");
  if (epi == Epi::SWIGLU_SPLIT || epi == Epi::SWIGLU_F16) PF_CHECK(a.N % 4 == 0, "gemm_int4: SwiGLU needs N % 4 == 0");
  if (epi == Epi::SWIGLU_SPLIT) PF_CHECK(a.out_lo, "gemm_int4: SWIGLU_SPLIT needs an output lo plane");
  if (epi == Epi::ROPE_F16)
    PF_CHECK(a.rope_cos && a.rope_sin && a.seq_len > 0 && a.rope_cols % 64 == 0,
             "gemm_int4: RoPE epilogue needs tables, seq_len and head-aligned rope_cols");
  if (epi == Epi::ROPE_F16) PF_CHECK(!grouped && (long)a.M < (1L << 31), "RoPE epilogue: dense rows below 2^31");
  if (grouped) PF_CHECK(a.tiles && a.num_tiles && a.max_tiles > 0, "gemm_int4: grouped mode needs a tile list");
  else PF_CHECK(a.M >= 0, "gemm_int4: M must be non-negative");
  // activation rows are addressed with 32-bit element offsets (grouped: a.M
  // slots bound every row the tile list or the row map can name)
  PF_CHECK((long)a.M * a.ldx < (1L << 31), "gemm_int4: activation offsets exceed 32 bits");
  const bool split = xk == XKind::SPLIT;
  if (a.K % KC == 0) {
    const bool k128 = ((reinterpret_cast<uintptr_t>(a.wz) & 1) | (reinterpret_cast<uintptr_t>(a.ws) & 3)) == 0 &&
                      ((a.wz_gs & 1) | (a.ws_gs & 1)) == 0 && (long)a.N * a.K / 2 < (1L << 31);
    if (k128 && dispatch_k128(b, a, split, epi, grouped, tile_t, prof_name)) return;
  }
  // The kernel above takes what that one does not (its descriptors hold one matrix below 2^31 bytes):
  // any plan of up to 64 rows per tile on 64-row tiles, whose rows come from the tile list.
  if (tile_t == 64 || (grouped && (tile_t == 16 || tile_t == 32))) {
    if (split) {
      if (grouped) dispatch_epi<64, true, true>(b, a, epi, prof_name);
      else dispatch_epi<64, true, false>(b, a, epi, prof_name);
    } else {
      if (grouped) dispatch_epi<64, false, true>(b, a, epi, prof_name);
      else dispatch_epi<64, false, false>(b, a, epi, prof_name);
    }
  } else {
    PF_CHECK(tile_t == 128, "gemm_int4: tile_t must be 64 or 128 (grouped: 16, 32, 64 or 128)");
    if (split) {
      if (grouped) dispatch_epi<128, true, true>(b, a, epi, prof_name);
      else dispatch_epi<128, true, false>(b, a, epi, prof_name);
    } else {
      if (grouped) dispatch_epi<128, false, true>(b, a, epi, prof_name);
      else dispatch_epi<128, false, false>(b, a, epi, prof_name);
    }
  }
}

// ---------------------------------------------------------------- layout probe

__global__ void k_probe_mfma(const uint16_t* A, const uint16_t* B, float* D) {
  // A: 16x32 row-major fp16, B: 32x16 row-major fp16, D: 16x16 row-major f32
  const int l = threadIdx.x, l16 = l & 15, lg = l >> 4;
  h8_t a, bb;
  for (int i = 0; i < 8; ++i) {
    a[i] = __builtin_bit_cast(_Float16, A[l16 * 32 + 8 * lg + i]);
    bb[i] = __builtin_bit_cast(_Float16, B[(8 * lg + i) * 16 + l16]);
  }
  f4_t d = mfma16x16x32(a, bb, f4_t{0.f, 0.f, 0.f, 0.f});
  for (int r = 0; r < 4; ++r) D[(4 * lg + r) * 16 + l16] = d[r];
}

void probe_mfma_f16(pfhip_backend* b, const uint16_t* a, const uint16_t* bm, float* d) {
  ProfScope ps(b, "probe_mfma_f16");
  hipLaunchKernelGGL(k_probe_mfma, dim3(1), dim3(64), 0, b->stream, a, bm, d);
  PF_HIP(hipGetLastError());
}

}  // namespace pf
