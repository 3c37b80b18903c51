// Gated DeltaNet chunked prefill on gfx950 (UT form, chunk C = 64).
//
// Reference: Qwen35HybridTextBackend::run_linear_delta_prefill_gpu_batched
// (src/models/Qwen35HybridTextBackend.cpp:1306-1508) applies the decode
// recurrence token by token inside one workgroup per value head. Here the
// same recurrence (host form :1729-1780) is evaluated chunk-wise:
//
// For a chunk with state S0 [dk, dv] (rows = key dims), normalisers
// ik_t = 1/sqrt(|k_t|^2+eps), iq_t likewise, beta_t, cumulative log-decay
// G_t = sum_{s<=t} g_t, and the inputs K, Q, V:
//   A[t,s]  = beta_t e^(G_t-G_s) ik_t ik_s (K K^T)[t,s]          (s < t)
//   T       = (I + A)^-1,  To = T - I                            (fp32)
//   R       = diag(beta) V - diag(sw) (K S0),   sw = beta e^G ik
//   D       = R + To R
//   O       = scale * ( fq (Q S0) + P D ),   fq = e^G iq,
//             P[t,s] = e^(G_t-G_s) iq_t ik_s (Q K^T)[t,s]          (s <= t)
//   S1      = e^(G_last) S0 + K^T (fk D),      fk = e^(G_last-G) ik
// All decays are formed as exp of differences with s <= t (never a ratio),
// so they stay in [0, 1]. T is computed in fp32 (diagonal 16x16 blocks by
// substitution, off-diagonal blocks on the fp32 matrix cores), its unit
// diagonal is applied in fp32, and every product that feeds the state
// carries its inexact operands as a hi + lo pair of bf16 (x = bf16(x) +
// bf16(x - bf16(x)), 2^-16 relative): S (and K, when it is the fp32 conv
// output) in K S0, To and R in To R, fk D (and K) in the state update, each
// as hi*hi + hi*lo + lo*hi. With decays near 1 sw K S0 nearly cancels beta V;
// forming that difference first, in fp32, keeps T's operand small. The
// output-only products (Q S, P D) use single bf16 (S as hi + lo in the layer).
//
// Kernel 1 (deltanet_chunk_prep_kernel): one workgroup per (chunk, key head,
//   sequence), or several that share the key head's value heads where the grid
//   is small, forms what the recurrence needs and S does not enter: K, Q,
//   K K^T and Q K^T once, then To and P for each of its value heads (four waves
//   per value head).
// Kernel 2 (deltanet_chunk_scan_kernel): one workgroup of 8 waves (12 at NT = 1)
//   per (slab of 16 NT columns of dv, value head, sequence) walks the chunks in order with
//   its state slab in registers of four "state" waves, while four "output"
//   waves form the outputs beside them, bring the K tiles of later chunks to
//   LDS by DMA and form the V rows.
// T is applied to R inside the scan: storing W = T diag(sw) K and U = T
// diag(beta) V per value head instead made its chunk record 73 KiB (now 25)
// and both products part of the prep. Layer, T = 4096, 16 key and 32 value
// heads: prep 113 -> 44 us, scan 103 -> 85 us, call 214 -> 152 us; the
// recurrence alone 144 -> 106 us.
//
// Token/key "slot" order: every MFMA that contracts over an index whose
// B operand is published from C-layout registers (the state rows, the
// tokens of R and D) uses, within each 32-wide k-step, the order in which lane
// group g (= lane / 16) supplies k = {4g..4g+3, 16+4g..16+4g+3}. The
// workspace stores To and P (over tokens) and Q (over key dims) in that order.
#include "common.hpp"
#include "deltanet_generic.hpp"

#include <algorithm>
#include <type_traits>

namespace aila {
namespace {

constexpr int kC = 64;          // chunk length
constexpr int kD = 128;         // key and value head dim
constexpr int kRB = kD * 2;     // bytes per K/Q row
constexpr int kTile = kC * kRB; // bytes of a K or Q tile
constexpr int kHeadThreads = 256;   // prep threads per value head
// Scan threads: four state and four output waves, and with one column tile
// (whose registers allow a third wave per SIMD) four helper waves.
constexpr int scan_threads(int NT) { return NT == 1 ? 768 : 512; }
constexpr int kNumXcd = 8;      // MI355X: 8 accelerator complex dies, one L2 each

__device__ __forceinline__ bf16x8_t cat8x2(const u32x2& a, const u32x2& b) {
  const u32x4 r = {a[0], a[1], b[0], b[1]};
  return as_bf16x8(r);
}
// Low 16 bits' / high 16 bits' bf16 of element e of a packed vector, as fp32.
template <class V>
__device__ __forceinline__ float bf_at(const V& w, int e) {
  return __uint_as_float((e & 1) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16));
}
// bf16 hi + lo of eight / four fp32 values.
__device__ __forceinline__ void split8(const float* x, u32x4& hi, u32x4& lo) {
  hi = u32x4{pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]), pack_bf16x2(x[4], x[5]), pack_bf16x2(x[6], x[7])};
  float r[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = x[e] - bf_at(hi, e);
  lo = u32x4{pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3]), pack_bf16x2(r[4], r[5]), pack_bf16x2(r[6], r[7])};
}
__device__ __forceinline__ void split4(const f32x4& x, u32x2& hi, u32x2& lo) {
  hi = u32x2{pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3])};
  lo = u32x2{pack_bf16x2(x[0] - bf_at(hi, 0), x[1] - bf_at(hi, 1)), pack_bf16x2(x[2] - bf_at(hi, 2), x[3] - bf_at(hi, 3))};
}

// K and Q tiles in LDS: rows of 256 bytes, 16-byte chunks swizzled by the row.
// kSlot tiles (formed by the prep from the fused rows) hold each 32-wide k-step
// in slot order, so that a row's MFMA operand is one 16-byte read; tiles DMA'd
// from the input rows keep the key order (two 8-byte reads). Both swizzles give
// 16 rows of one chunk distinct banks; the slot tiles' also the transposing
// reads' four rows of four half chunks.
template <bool kSlot>
__device__ __forceinline__ int swz_rows(int r) {
  return kSlot ? ((r & 3) << 2) | ((r ^ (r >> 2)) & 3) : r & 15;
}
// 16x16 tile (I, J), J <= I, of a packed lower triangle of tiles.
__device__ __forceinline__ constexpr int tri(int I, int J) { return I * (I + 1) / 2 + J; }

// MFMA A/B operand over 32 tokens in slot order from a tile by transposing
// reads: lane (g4, m16) gets M[tokens of g4][16*dt + m16].
template <bool kSlot>
__device__ __forceinline__ bf16x8_t tr_operand(const unsigned char* tile, int ks, int dt, int m16, int g4) {
  const int p = m16 & 3;   // keys 4p .. 4p+3 of tile dt
  const int chunk = kSlot ? 4 * (dt >> 1) + p : 2 * dt + (p >> 1), half = kSlot ? dt & 1 : p & 1;
  const int r0 = ks * 32 + 4 * g4 + (m16 >> 2), r1 = r0 + 16;
  const u32x2 lo = ds_read_tr4(tile + r0 * kRB + ((chunk ^ swz_rows<kSlot>(r0)) << 4) + (half << 3));
  const u32x2 hi = ds_read_tr4(tile + r1 * kRB + ((chunk ^ swz_rows<kSlot>(r1)) << 4) + (half << 3));
  return cat8x2(lo, hi);
}
// MFMA A operand over 32 key dims in slot order: row r of a tile.
template <bool kSlot>
__device__ __forceinline__ bf16x8_t row_operand(const unsigned char* tile, int ks, int r, int g4) {
  if constexpr (kSlot) {
    return as_bf16x8(*reinterpret_cast<const u32x4*>(tile + r * kRB + (((4 * ks + g4) ^ swz_rows<kSlot>(r)) << 4)));
  } else {
    const unsigned char* row = tile + r * kRB + ((g4 & 1) << 3);
    const int c = 4 * ks + (g4 >> 1);
    const u32x2 a = *reinterpret_cast<const u32x2*>(row + ((c ^ swz_rows<kSlot>(r)) << 4));
    const u32x2 b = *reinterpret_cast<const u32x2*>(row + (((c + 2) ^ swz_rows<kSlot>(r)) << 4));
    return cat8x2(a, b);
  }
}

// Workspace records of one chunk. Scan operands that go to registers are
// stored in register order - [tile][k-step][lane][16 bytes] - so that one wave
// load is one contiguous KiB (a 16-row gather would cost the memory pipe 16
// cache lines per instruction). Per (sequence, value head, chunk):
//   F  fq[C], fk[C], beta[C], sw[C], gamma (C copies: a vector load) (f32)
//   T  [4 token tiles][2 token k-steps][64][8 bf16]  To[16w+l%16][32s2 + slots of l/16]
//   TLo  the bf16 residual To - bf16(To), laid out as T
//   P  as T
// and once per (sequence, key head, chunk):
//   K  the K tile as it lies in LDS (row-major, swizzled 16-byte chunks)
//   KLo (split inputs only) its bf16 residual
//   Q  [4 token tiles][4 k-steps][64][8 bf16]        Q[16w+l%16][32ks + slots of l/16]
// (k-step 1 of the first two token tiles of T and P is zero: neither written
// nor read.) The key-head records follow all value-head records.
struct ChunkRec {
  static constexpr size_t kF = 0;
  static constexpr size_t kT = 5 * kC * 4;
  static constexpr size_t kTLo = kT + size_t(kC) * kC * 2;
  static constexpr size_t kP = kTLo + size_t(kC) * kC * 2;
  static constexpr size_t kBytes = kP + size_t(kC) * kC * 2;
};
template <bool kLo>
struct KeyRec {
  static constexpr size_t kK = 0;
  static constexpr size_t kQ = kK + kTile;
  static constexpr size_t kKLo = kQ + kTile;
  static constexpr size_t kBytes = kKLo + (kLo ? kTile : 0);
};
static_assert(ChunkRec::kBytes % 256 == 0 && ChunkRec::kT % 256 == 0, "records keep 256-byte alignment");
// Key-head record (b, hk, c) of a workspace laid out for B, Hv, nch.
template <bool kLo>
__host__ __device__ __forceinline__ size_t key_rec_offset(int b, int hk, int c, int B, int Hk, int Hv, int nch) {
  return static_cast<size_t>(B) * Hv * nch * ChunkRec::kBytes +
         ((static_cast<size_t>(b) * Hk + hk) * nch + c) * KeyRec<kLo>::kBytes;
}

// ---------------------------------------------------------------------------
// kLo: the inputs are fp32 values (conv + SiLU of the fused rows, ConvIn)
// carried as bf16 hi + residual tiles. The residuals enter where the rounding
// of an input would reach the state beyond fp32 accuracy - the key norms,
// K K^T, K S and K^T (fk D) - and where it would reach the outputs of rows
// whose q.k nearly cancels (the gated RMSNorm after the layer then magnifies
// an output far below sqrt(eps)): Q K^T takes Q_hi K_hi + Q_hi K_lo +
// Q_lo K_hi and the scan's Q S takes S as hi + lo.
//
// A workgroup takes `per` of its key head's value heads (see launch_prep), GP at
// a time by 4 waves each; more run in passes. The conv, norms and two products
// are formed once a workgroup, and GP heads' serial inversions are
// in flight side by side: the kernel is bound by those dependent chains (about
// 14 us at one chunk) and, over many chunks, by its ~120 MB of traffic at
// T = 4096, Hk = 16, Hv = 32 (44 us, 2.7 TB/s; two workgroups of 67 KiB a CU).
template <bool kLo, int GP>
__global__ __launch_bounds__(kHeadThreads * GP, GP == 2 ? 4 : GP == 1 ? 2 : GP) void deltanet_chunk_prep_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, ConvIn cv, const bf16* __restrict__ a,
    const bf16* __restrict__ bg, int ab_stride, const bf16* __restrict__ dt_bias, const float* __restrict__ A_log,
    unsigned char* __restrict__ ws, int T, int Hk, int Hv, int per, float eps) {
  using R = ChunkRec;
  using RK = KeyRec<kLo>;
  constexpr int kThr = kHeadThreads * GP, NW = 4 * GP;
  constexpr int kRaw = 20 * 1024;            // raw K K^T and Q K^T tiles
  constexpr int kTri = 10 * 1024;            // ten 16x16 fp32 tiles
  constexpr int kTiles = (kLo ? 4 : 2) * kTile;
  constexpr int kSmem = kTiles > kRaw + GP * 2 * kTri ? kTiles : kRaw + GP * 2 * kTri;
  // first the input tiles, then the raw products and each head's A and To
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kSmem];
  __shared__ __attribute__((aligned(16))) float sG2[GP][kC], sGn[GP][kC], sBeta[GP][kC], sIk[kC], sIq[kC];
  unsigned char* const sK = smem;
  unsigned char* const sQ = smem + kTile;
  unsigned char* const sKl = smem + (kLo ? 2 * kTile : 0);
  unsigned char* const sQl = smem + (kLo ? 3 * kTile : 0);

  const int c = blockIdx.x, hk = static_cast<int>(blockIdx.y) % Hk, b = blockIdx.z;
  const int nch = (T + kC - 1) / kC;
  // value heads of this workgroup: hv0 .. hv0 + nv - 1
  const int share = static_cast<int>(blockIdx.y) / Hk;
  const int hv0 = hk * (Hv / Hk) + share * per, nv = min(per, Hv / Hk - share * per);
  const int t0 = c * kC;
  const int n = min(kC, T - t0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2, w4 = wave & 3;
  const int m16 = lane & 15, g4 = lane >> 4;
  unsigned char* krec = ws + key_rec_offset<kLo>(b, hk, c, static_cast<int>(gridDim.z), Hk, Hv, nch);

  // gates of this chunk and one value head (one wave): beta, g, prefix sum G
  auto gates = [&](int pass) __attribute__((always_inline)) {
    if (w4 != 0) return;
    const int hv = hv0 + min(pass * GP + grp, nv - 1);
    float beta = 0.f, g = 0.f;
    if (lane < n) {
      const size_t gi = (static_cast<size_t>(b) * T + t0 + lane) * ab_stride + hv;
      beta = 1.0f / (1.0f + expf(-bf2f(bg[gi])));
      const float dtb = dt_bias ? bf2f(dt_bias[hv]) : 0.0f;
      const float negA = A_log ? -expf(A_log[hv]) : -1.0f;
      g = softplus_f(bf2f(a[gi]) + dtb) * negA;
    }
    float Gs = g;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float o = __shfl_up(Gs, off);
      if (lane >= off) Gs += o;
    }
    sGn[grp][lane] = Gs;
    sG2[grp][lane] = Gs * kLog2e;
    sBeta[grp][lane] = beta;
  };

  // ---- 1. K and Q tiles (rows past T are zero) ---------------------------------
  if constexpr (kLo) {
    // Item (tensor, cc, r0) forms 16-byte chunk cc of rows r0 .. r0+3 of the K
    // (tensor 0) or Q tile: conv of the 7 raw rows r0-3 .. r0+3 (rows before
    // token 0 from the ring), SiLU, then bf16 hi and residual.
    const int head = ((cv.head % 3) + 3) % 3;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16*>(cv.qkv + static_cast<size_t>(b) * T * cv.stride), 0, T * cv.stride * 2, kBufferRsrcWord3);
    const int cc1 = tid & 15, r01 = ((tid & 255) >> 4) * 4;
    // raw rows r0-3 .. r0+3 of 8 channels from ch0 (token rows by buffer
    // load: rows past T read as zeros; rows before token 0 from the ring)
    struct Raw { u32x4 x[7]; f32x4 rg[3][2]; };
    auto load_rows = [&](int c0, Raw& o) __attribute__((always_inline)) {
      const int ch0 = c0 + cc1 * 8;
#pragma unroll
      for (int j = 0; j < 7; ++j) {
        const int t = t0 + r01 - 3 + j;
        o.x[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (t * cv.stride + ch0) * 2, 0, 0));
      }
      if (t0 + r01 < 3) {   // only the first chunk's first rows reach back before token 0
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const int t = t0 + r01 - 3 + j;
          const float* rr = cv.ring + (static_cast<size_t>(b) * 3 + (head + 3 + (t < 0 ? t : 0)) % 3) * cv.ch + ch0;
          o.rg[j][0] = *reinterpret_cast<const f32x4*>(rr);
          o.rg[j][1] = *reinterpret_cast<const f32x4*>(rr + 4);
        }
      }
    };
    // conv (4 taps) + SiLU of those rows -> bf16 hi and residual tiles
    auto conv_rows = [&](int c0, const Raw& in, unsigned char* th, unsigned char* tl) __attribute__((always_inline)) {
      const int ch0 = c0 + cc1 * 8;
      float w[8][4];
#pragma unroll
      for (int v4i = 0; v4i < 4; ++v4i) {      // 16 bytes = the taps of two channels
        const u32x4 r = *reinterpret_cast<const u32x4*>(cv.w + static_cast<size_t>(ch0) * 4 + v4i * 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) w[2 * v4i + (e >> 2)][e & 3] = bf_at(r, e);
      }
      float x[7][8];
#pragma unroll
      for (int j = 0; j < 7; ++j) {
        unpack8(in.x[j], x[j]);
        if (j < 3 && t0 + r01 - 3 + j < 0) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x[j][e] = in.rg[j][0][e];
            x[j][4 + e] = in.rg[j][1][e];
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float acc = x[i][e] * w[e][0];
          acc += x[i + 1][e] * w[e][1];
          acc += x[i + 2][e] * w[e][2];
          acc += x[i + 3][e] * w[e][3];
          // SiLU from the hardware exp2 and reciprocal (about 1 ulp each,
          // far below the 2^-16 the hi + lo pair carries)
          const float sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-acc * kLog2e));
          y[e] = (r01 + i < n) ? acc * sg : 0.f;
        }
        u32x4 h, l;
        split8(y, h, l);
        // keys 8 cc1 .. + 3 and + 4 .. 7 go to slots of lane groups g and g + 1
        const int r = r01 + i, g = 4 * (cc1 >> 2) + 2 * (cc1 & 1), half = ((cc1 >> 1) & 1) << 3;
        const int a0 = r * kRB + ((g ^ swz_rows<kLo>(r)) << 4) + half, a1 = r * kRB + (((g + 1) ^ swz_rows<kLo>(r)) << 4) + half;
        *reinterpret_cast<u32x2*>(th + a0) = u32x2{h[0], h[1]};
        *reinterpret_cast<u32x2*>(th + a1) = u32x2{h[2], h[3]};
        *reinterpret_cast<u32x2*>(tl + a0) = u32x2{l[0], l[1]};
        *reinterpret_cast<u32x2*>(tl + a1) = u32x2{l[2], l[3]};
      }
    };
    const int qc0 = hk * kD, kc0 = Hk * kD + hk * kD;   // first q / k channel
    if constexpr (GP == 1) {
      Raw ra, rb;
      load_rows(kc0, ra);
      load_rows(qc0, rb);
      gates(0);
      conv_rows(kc0, ra, sK, sKl);
      conv_rows(qc0, rb, sQ, sQl);
    } else {
      Raw ra;
      if (wave < 8) load_rows(wave < 4 ? kc0 : qc0, ra);
      gates(0);
      if (wave < 4) conv_rows(kc0, ra, sK, sKl);
      else if (wave < 8) conv_rows(qc0, ra, sQ, sQl);
    }
  } else {
    const int row = Hk * kRB;   // source row stride (bytes)
    const size_t off = (static_cast<size_t>(b) * T + t0) * Hk * kD + hk * kD;
    const u32x4 rk = buffer_rsrc(k + off, (n - 1) * row + kRB);
    const u32x4 rq = buffer_rsrc(q + off, (n - 1) * row + kRB);
    for (int slot = wave; slot < kTile / 1024; slot += NW) {      // wave-contiguous KiB
      const int p = slot * 64 + lane;
      const int r = p / (kD / 8), cc = p % (kD / 8);
      dma16_to_lds(rk, r * row + ((cc ^ swz_rows<kLo>(r)) << 4), sK + slot * 1024);
      dma16_to_lds(rq, r * row + ((cc ^ swz_rows<kLo>(r)) << 4), sQ + slot * 1024);
    }
    gates(0);
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm<0>());
  __syncthreads();

  auto row_chunk = [&](const unsigned char* tile, int r, int cs) __attribute__((always_inline)) {
    return *reinterpret_cast<const u32x4*>(tile + r * kRB + ((cs ^ swz_rows<kLo>(r)) << 4));
  };
  // ---- 2. raw products: jobs 0..9 (K K^T), 10..19 (Q K^T), tile (ti, tj), both
  //      transposed (rows s of tile tj, columns t of tile ti), so that a lane
  //      holds four consecutive s of one t.
  constexpr int kJobs = 20, JP = (kJobs + NW - 1) / NW;
  f32x4 prod[JP];
#pragma unroll
  for (int i = 0; i < JP; ++i) {
    const int job = wave + NW * i;
    prod[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (job < kJobs) {
      int tj = job < 10 ? job : job - 10, ti = 0;
      while (tj > ti) { tj -= ti + 1; ++ti; }
      const unsigned char* X = job < 10 ? sK : sQ;
      const unsigned char* Xl = job < 10 ? sKl : sQl;
#pragma unroll
      for (int ks = 0; ks < kD / 32; ++ks) {
        const bf16x8_t ka = as_bf16x8(row_chunk(sK, tj * 16 + m16, ks * 4 + g4));
        const bf16x8_t xb = as_bf16x8(row_chunk(X, ti * 16 + m16, ks * 4 + g4));
        prod[i] = mfma16x16x32(ka, xb, prod[i]);
        if constexpr (kLo) {
          prod[i] = mfma16x16x32(as_bf16x8(row_chunk(sKl, tj * 16 + m16, ks * 4 + g4)), xb, prod[i]);
          prod[i] = mfma16x16x32(ka, as_bf16x8(row_chunk(Xl, ti * 16 + m16, ks * 4 + g4)), prod[i]);
        }
      }
    }
  }
  // ---- 3. row norms: 4 threads per row of the K and the Q tile -------------------
  for (int it = tid; it < 2 * 4 * kC; it += kThr) {
    const int r = (it & 255) >> 2, part = it & 3;
    const unsigned char* X = it < 256 ? sK : sQ;
    const unsigned char* Xl = it < 256 ? sKl : sQl;
    float ss = 0.f;
#pragma unroll
    for (int cc = 0; cc < kD / 32; ++cc) {
      float x[8];
      unpack8(row_chunk(X, r, part * (kD / 32) + cc), x);
      if constexpr (kLo) {
        float l[8];
        unpack8(row_chunk(Xl, r, part * (kD / 32) + cc), l);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] += l[e];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf(x[e], x[e], ss);
    }
    ss += __shfl_xor(ss, 1);
    ss += __shfl_xor(ss, 2);
    if (part == 0) (it < 256 ? sIk : sIq)[r] = 1.0f / sqrtf(ss + eps);
  }
  // ---- 4. key-head record (first share): K tile image(s), Q in register order -----
  for (int o = tid; share == 0 && o < kTile / 16; o += kThr) {
    __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(sK + o * 16), reinterpret_cast<u32x4*>(krec + RK::kK) + o);
    if constexpr (kLo)
      __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(sKl + o * 16), reinterpret_cast<u32x4*>(krec + RK::kKLo) + o);
    // [token tile][k-step][lane]
    const int l = o & 63;
    __builtin_nontemporal_store(__builtin_bit_cast(u32x4, row_operand<kLo>(sQ, (o >> 6) & 3, (o >> 8) * 16 + (l & 15), l >> 4)),
                                reinterpret_cast<u32x4*>(krec + RK::kQ) + o);
  }
  __syncthreads();   // the tiles are read: their space becomes the raw products, A and To
  f32x4* const raw = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int i = 0; i < JP; ++i)
    if (wave + NW * i < kJobs) raw[(wave + NW * i) * 64 + lane] = prod[i];
  __syncthreads();

  float* const sA = reinterpret_cast<float*>(smem + kRaw + grp * 2 * kTri);
  float* const sT = sA + kTri / 4;
  for (int pass = 0; pass * GP < nv; ++pass) {
    const bool live = pass * GP + grp < nv;
    const int hv = hv0 + min(pass * GP + grp, nv - 1);
    unsigned char* rec = ws + ((static_cast<size_t>(b) * Hv + hv) * nch + c) * R::kBytes;
    // ---- 5. A (LDS, packed tiles) and P (register order) with this head's gates --
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int job = w4 + 4 * i;
      if (job < 10) {
        int tj = job, ti = 0;
        while (tj > ti) { tj -= ti + 1; ++ti; }
        const int t = ti * 16 + m16, s0 = tj * 16 + 4 * g4;
        const f32x4 x = raw[job * 64 + lane];
        const f32x4 iks = *reinterpret_cast<const f32x4*>(sIk + s0), g2s = *reinterpret_cast<const f32x4*>(sG2[grp] + s0);
        const float f = sBeta[grp][t] * sIk[t], g2t = sG2[grp][t];
        f32x4 r;
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] = (s0 + j < t) ? f * iks[j] * fast_exp2(g2t - g2s[j]) * x[j] : 0.f;
        *reinterpret_cast<f32x4*>(sA + job * 256 + m16 * 16 + 4 * g4) = r;
      } else if (live) {
        // P jobs (ti, s2): (0,0) (1,0) (2,0) (2,1) (3,0) (3,1)
        const int pj = job - 10, ti = pj < 2 ? pj : 2 + ((pj - 2) >> 1), s2 = pj < 2 ? 0 : (pj & 1);
        const int t = ti * 16 + m16;
        const float iqt = sIq[t], g2t = sG2[grp][t];
        float pv[8];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int tj = 2 * s2 + h, s0 = tj * 16 + 4 * g4;
          const f32x4 x = raw[(10 + tri(ti, min(tj, ti))) * 64 + lane];
          const f32x4 iks = *reinterpret_cast<const f32x4*>(sIk + s0), g2s = *reinterpret_cast<const f32x4*>(sG2[grp] + s0);
#pragma unroll
          for (int j = 0; j < 4; ++j)
            pv[4 * h + j] = (s0 + j <= t) ? iqt * iks[j] * fast_exp2(g2t - g2s[j]) * x[j] : 0.f;
        }
        __builtin_nontemporal_store(u32x4{pack_bf16x2(pv[0], pv[1]), pack_bf16x2(pv[2], pv[3]),
                                          pack_bf16x2(pv[4], pv[5]), pack_bf16x2(pv[6], pv[7])},
                                    reinterpret_cast<u32x4*>(rec + R::kP) + (ti * 2 + s2) * 64 + lane);
      }
    }
    // row factors
    if (live && w4 == 3) {
      float* F = reinterpret_cast<float*>(rec + R::kF);
      const float Gt = sGn[grp][lane], Glast = sGn[grp][n - 1], ik = sIk[lane], beta = sBeta[grp][lane];
      F[lane] = (lane < n) ? expf(Gt) * sIq[lane] : 0.f;                   // fq
      F[kC + lane] = (lane < n) ? expf(Glast - Gt) * ik : 0.f;             // fk
      F[2 * kC + lane] = beta;
      F[3 * kC + lane] = beta * expf(Gt) * ik;                             // sw
      F[4 * kC + lane] = expf(Glast);                                      // gamma
    }
    __syncthreads();

    // ---- 6. To = (I + A)^-1 - I -----------------------------------------------
    // 6a. diagonal block w4 by substitution: lane (g4, m16) owns column m16 and
    //     the partial sums over rows m = 4*g4 .. 4*g4+3 of the block.
    {
      const float* At = sA + tri(w4, w4) * 256;
      const int j = m16;
      float xl[4];
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) xl[kk] = (4 * g4 + kk == j) ? 1.f : 0.f;
#pragma unroll
      for (int i = 1; i < 16; ++i) {
        const f32x4 arow = *reinterpret_cast<const f32x4*>(At + i * 16 + 4 * g4);
        float part = arow[0] * xl[0];
#pragma unroll
        for (int kk = 1; kk < 4; ++kk) part = fmaf(arow[kk], xl[kk], part);   // A[i][m] = 0 for m >= i
        const float sum = xrow4_sum(part);
        const float xi = (i > j) ? -sum : ((i == j) ? 1.f : 0.f);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
          if (4 * g4 + kk == i) xl[kk] = xi;
      }
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        sT[tri(w4, w4) * 256 + (4 * g4 + kk) * 16 + j] = (4 * g4 + kk > j) ? xl[kk] : 0.f;
    }
    __syncthreads();
    // 6b. off-diagonal blocks by distance d on the fp32 matrix cores:
    //     T_IJ = -(I + To_II) R,  R = sum_{M=J}^{I-1} A_IM T_MJ,  T_JJ = I + To_JJ.
    // 16x16x16 products on v_mfma_f32_16x16x4f32 with the k index permuted so
    // that at step kk lane group g supplies k = 4g + kk: the A operand of the
    // four steps is one float4 of row m16, and a 16x16 block held in C layout
    // (lane (g, m16) has rows 4g..4g+3 of column m16) is directly the B
    // operand of the four steps.
    auto mul = [&](f32x4 acc, const float* X, const f32x4& yb) __attribute__((always_inline)) {
      const f32x4 xa = *reinterpret_cast<const f32x4*>(X + m16 * 16 + 4 * g4);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[kk], yb[kk], acc, 0, 0, 0);
      return acc;
    };
    auto cblock = [&](const float* Y) __attribute__((always_inline)) {   // C layout of a block
      f32x4 r;
#pragma unroll
      for (int j = 0; j < 4; ++j) r[j] = Y[(4 * g4 + j) * 16 + m16];
      return r;
    };
    for (int d = 1; d < 4; ++d) {
      if (w4 < 4 - d) {
        const int J = w4, I = J + d;
        f32x4 r = cblock(sA + tri(I, J) * 256);                             // A_IJ (identity part of T_JJ)
        for (int M = J; M < I; ++M) r = mul(r, sA + tri(I, M) * 256, cblock(sT + tri(M, J) * 256));
        const f32x4 tr = mul(r, sT + tri(I, I) * 256, r);                   // R + To_II R
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) sT[tri(I, J) * 256 + (4 * g4 + jj) * 16 + m16] = -tr[jj];
      }
      __syncthreads();
    }
    // ---- 7. To as a hi + lo pair in register order -------------------------------
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      if (live && ks <= (w4 >> 1)) {
        float f[8];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int J = 2 * ks + h;
          const f32x4 x = *reinterpret_cast<const f32x4*>(sT + tri(w4, min(J, w4)) * 256 + m16 * 16 + 4 * g4);
#pragma unroll
          for (int j = 0; j < 4; ++j) f[4 * h + j] = J <= w4 ? x[j] : 0.f;
        }
        u32x4 hi, lo;
        split8(f, hi, lo);
        __builtin_nontemporal_store(hi, reinterpret_cast<u32x4*>(rec + R::kT) + (w4 * 2 + ks) * 64 + lane);
        __builtin_nontemporal_store(lo, reinterpret_cast<u32x4*>(rec + R::kTLo) + (w4 * 2 + ks) * 64 + lane);
      }
    }
    if ((pass + 1) * GP < nv) {
      __syncthreads();   // the gates and A of this pass are no longer read
      gates(pass + 1);
      __syncthreads();
    }
  }
}

// ---------------------------------------------------------------------------
// Per-chunk operands in registers, by wave role.
struct StateOps {
  u32x4 th[2], tl[2];    // To rows of token tile w4, token k-steps 0..1, and their residual
};
template <int NT, int RAW>
struct OutOps {
  u32x4 q[4];        // Q rows of token tile w4, k-steps 0..3 (slot order)
  u32x4 p[2];        // P rows, token k-steps 0..1
  u32x2 v[RAW];      // V input rows (NT = 1: 4 columns, else this lane's NT)
};

// One workgroup = 8 waves (12 at NT = 1, with four helpers) on NT 16-column tiles
// of one (value head, sequence).
// Waves 0-3 ("state" waves) carry the recurrence: each holds 32 key rows of
// the slab's state. Waves 4-7 ("output" waves) form the outputs of token tile
// w4, V of the next chunk, and the DMAs that bring later chunks' K tiles.
// With two waves per SIMD the output path runs beside the state path; three
// barriers per chunk order both:
//   A: state: R = beta V - sw (K S), publish R       | output: Q S
//   B: state: D = R + To R, publish D and fk D       | output: V of the next chunk
//   C: state: S' = gamma S + K^T (fk D), publish S'  | output: + P D, store
// K tiles and register operands run NS - 1 chunks ahead.
// Bound by the chunk's dependent chain (NT = 1: 62 of the scan's 85 us remain
// with every load, DMA and V row taken out), then by its ~90 vector memory
// instructions and the LDS traffic of the exchanges. Hence: row factors by DMA
// instead of one load per wave and factor, V input in 4 loads of 8 bytes, not
// 7 of 2 (103 -> 97 us together with it), and with one column tile the DMAs and
// V on four helper waves (97 -> 89) whose DMAs follow V, since the wait the
// compiler places for V's rows would cover them.
template <bool kLo, int NT>
__global__ __launch_bounds__(scan_threads(NT), 1) void deltanet_chunk_scan_kernel(
    const bf16* __restrict__ v, ConvIn cv, const unsigned char* __restrict__ ws, float* __restrict__ state,
    bf16* __restrict__ out, int T, int Hk, int Hv, float scale) {
  using R = ChunkRec;
  using RK = KeyRec<kLo>;
  constexpr int NS = NT <= 2 ? 3 : 2;            // chunks in flight (LDS stages, register sets)
  constexpr int kSlabs = kD / (16 * NT);
  // V input rows per lane: with one column tile a lane forms four columns of
  // one token, else the four tokens of its C-layout registers (conv: + 3 rows)
  constexpr int RAW = NT == 1 ? (kLo ? 4 : 1) : (kLo ? 7 : 4);
  constexpr int kDma = (kLo ? 2 : 1) * kTile / 1024 / 4;   // DMA instructions per output wave and chunk
  // XCD-aware placement: workgroups are dispatched round-robin over the 8
  // XCDs, so linear id i runs on XCD i % 8. The slabs of a head are put on
  // the same XCD, where they share the head's chunk records in L2 (otherwise
  // every XCD fetches them from HBM), and each XCD takes a contiguous range
  // of heads, so that the value heads of a key head also share its key-head
  // records there.
  const int nwg = static_cast<int>(gridDim.x * gridDim.y * gridDim.z);
  int lin = blockIdx.x + kSlabs * (blockIdx.y + static_cast<int>(gridDim.y) * blockIdx.z);
  if (nwg % kNumXcd == 0) lin = (lin % kNumXcd) * (nwg / kNumXcd) + lin / kNumXcd;
  const int slab = lin % kSlabs, headlin = lin / kSlabs;
  const int hv = headlin % Hv, b = headlin / Hv;
  const int nch = (T + kC - 1) / kC;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w4 = wave & 3;
  const int m16 = lane & 15, g4 = lane >> 4;
  // Column m16 of the NT tiles is column m16 * NT + nt of the slab, so that a
  // lane's columns are contiguous in the state, the V rows and the outputs.
  const int col = (slab * 16 + m16) * NT;

  __shared__ __attribute__((aligned(1024))) unsigned char sK[NS][kTile];
  __shared__ __attribute__((aligned(1024))) unsigned char sKl[kLo ? NS : 1][kLo ? kTile : 16];
  __shared__ u32x4 sS[NT][4][64];            // S B-operands, one per 32-row k-step
  __shared__ u32x4 sSl[NT][4][64];           // residual of S
  __shared__ u32x2 sRh[NT][2][2][64], sRl[NT][2][2][64];   // R hi, lo: [k-step][half][lane]
  __shared__ u32x2 sD[NT][2][2][64];         // D (bf16)
  __shared__ u32x2 sDh[NT][2][2][64], sDl[NT][2][2][64];   // (fk D) hi, lo
  __shared__ __attribute__((aligned(256))) float sF[NS][5][kC];   // row factors of the record
  // V rows. One column tile: [token][column], rows padded to 20 floats; else C
  // layout. By chunk parity where the next chunk's V is formed in phase A.
  constexpr int kVRow = 20;
  __shared__ __attribute__((aligned(16))) float sV1[NT == 1 ? 2 : 1][NT == 1 ? kC * kVRow : 4];
  __shared__ f32x4 sV[NT == 2 ? 2 : 1][NT == 1 ? 1 : NT][4][64];

  const unsigned char* recs = ws + (static_cast<size_t>(b) * Hv + hv) * nch * R::kBytes;
  auto rec_of = [&](int c) __attribute__((always_inline)) { return recs + static_cast<size_t>(c) * R::kBytes; };
  const unsigned char* krecs =
      ws + key_rec_offset<kLo>(b, hv / (Hv / Hk), 0, static_cast<int>(gridDim.z), Hk, Hv, nch);
  auto krec_of = [&](int c) __attribute__((always_inline)) { return krecs + static_cast<size_t>(c) * RK::kBytes; };

  if (wave < 4) {
    // ------------------------------------------------------------ state waves
    auto load = [&](int c, StateOps& o) __attribute__((always_inline)) {
      const unsigned char* rec = rec_of(c);
      const u32x4* Th = reinterpret_cast<const u32x4*>(rec + R::kT) + w4 * 128 + lane;
      const u32x4* Tl = reinterpret_cast<const u32x4*>(rec + R::kTLo) + w4 * 128 + lane;
      o.th[0] = Th[0];
      o.tl[0] = Tl[0];
      if (w4 >= 2) {
        o.th[1] = Th[64];
        o.tl[1] = Tl[64];
      }
    };
    auto factor = [&](const float (&f)[5][kC], int which) __attribute__((always_inline)) {
      return *reinterpret_cast<const f32x4*>(&f[which][w4 * 16 + g4 * 4]);
    };
    // state slab in C layout: rows 32*w4 + 16*tt + 4*g4 + j, column col + nt
    float* Sg = state + (static_cast<size_t>(b) * Hv + hv) * kD * kD + static_cast<size_t>(w4 * 32 + g4 * 4) * kD + col;
    float s_reg[NT][8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) s_reg[nt][e] = Sg[((e >> 2) * 16 + (e & 3)) * kD + nt];
    u32x4 s_hi[NT], s_lo[NT];   // this wave's own k-step of the S operand
    auto publish_state = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        split8(s_reg[nt], s_hi[nt], s_lo[nt]);
        sS[nt][w4][lane] = s_hi[nt];
        sSl[nt][w4][lane] = s_lo[nt];
      }
    };
    const int s2w = w4 >> 1, halfw = w4 & 1;
    // `active` is uniform; an inactive chunk (past the last one, padding the
    // rotation) computes on repeated operands but keeps its state (a select,
    // so the chunk body stays one basic block for the schedule).
    // K rows of token tile w4, read a phase ahead; k-step (w4 + i) % 4 at i, so
    // that the first products take the wave's own state rows from registers
    bf16x8_t kh[4], kl[4];
    auto read_k = [&](const unsigned char* kt, const unsigned char* klt) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        kh[i] = row_operand<kLo>(kt, (w4 + i) & 3, w4 * 16 + m16, g4);
        if constexpr (kLo) kl[i] = row_operand<kLo>(klt, (w4 + i) & 3, w4 * 16 + m16, g4);
      }
    };
    auto chunk = [&](auto pos, bool active, int c, const StateOps& o, StateOps& on) __attribute__((always_inline)) {
      constexpr int st = decltype(pos)::value, stn = (st + 1) % NS;
      // A: R = beta V - sw (K S) of token tile w4
      const f32x4 beta = factor(sF[st], 2), sw = factor(sF[st], 3), fk = factor(sF[st], 1);
      const float gam = sF[st][4][lane];
      f32x4 r[NT];
      bf16x8_t kth[2][2], ktl[2][2];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f}, acl = {0.f, 0.f, 0.f, 0.f}, acm = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int ks = (w4 + i) & 3;
          const bf16x8_t sh = as_bf16x8(i == 0 ? s_hi[nt] : sS[nt][ks][lane]);
          const bf16x8_t sl = as_bf16x8(i == 0 ? s_lo[nt] : sSl[nt][ks][lane]);
          acc = mfma16x16x32(kh[i], sh, acc);
          acl = mfma16x16x32(kh[i], sl, acl);
          if constexpr (kLo) acm = mfma16x16x32(kl[i], sh, acm);
        }
        if (nt == 0) {   // the K^T operands of phase C, read under the arithmetic
#pragma unroll
          for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2) {
              kth[tt][s2] = tr_operand<kLo>(sK[st], s2, w4 * 2 + tt, m16, g4);
              if constexpr (kLo) ktl[tt][s2] = tr_operand<kLo>(sKl[st], s2, w4 * 2 + tt, m16, g4);
            }
        }
        if constexpr (kLo) acl += acm;
        f32x4 vr;
        if constexpr (NT == 1) {
#pragma unroll
          for (int j = 0; j < 4; ++j) vr[j] = sV1[c & 1][(w4 * 16 + g4 * 4 + j) * kVRow + m16];
        } else {
          vr = sV[NT == 2 ? c & 1 : 0][nt][w4][lane];
        }
        r[nt] = beta * vr - sw * (acc + acl);
        u32x2 hi, lo;
        split4(r[nt], hi, lo);
        sRh[nt][s2w][halfw][lane] = hi;
        sRl[nt][s2w][halfw][lane] = lo;
      }
      phase_barrier();
      // B: D = R + To R
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        f32x4 d = r[nt], dl = {0.f, 0.f, 0.f, 0.f}, dm = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2)
          if (s2 <= s2w) {
            const bf16x8_t rh = cat8x2(sRh[nt][s2][0][lane], sRh[nt][s2][1][lane]);
            const bf16x8_t rl = cat8x2(sRl[nt][s2][0][lane], sRl[nt][s2][1][lane]);
            d = mfma16x16x32(as_bf16x8(o.th[s2]), rh, d);
            dl = mfma16x16x32(as_bf16x8(o.th[s2]), rl, dl);
            dm = mfma16x16x32(as_bf16x8(o.tl[s2]), rh, dm);
          }
        d += dl + dm;
        sD[nt][s2w][halfw][lane] = u32x2{pack_bf16x2(d[0], d[1]), pack_bf16x2(d[2], d[3])};
        u32x2 hi, lo;
        split4(fk * d, hi, lo);
        sDh[nt][s2w][halfw][lane] = hi;
        sDl[nt][s2w][halfw][lane] = lo;
      }
      phase_barrier();
      // C: S = gamma S + K^T (fk D) for the key rows of this wave
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        f32x4 a2[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const bf16x8_t dh = cat8x2(sDh[nt][s2][0][lane], sDh[nt][s2][1][lane]);
          const bf16x8_t dl = cat8x2(sDl[nt][s2][0][lane], sDl[nt][s2][1][lane]);
#pragma unroll
          for (int tt = 0; tt < 2; ++tt) {
            a2[tt] = mfma16x16x32(kth[tt][s2], dh, a2[tt]);
            a2[tt] = mfma16x16x32(kth[tt][s2], dl, a2[tt]);
            if constexpr (kLo) a2[tt] = mfma16x16x32(ktl[tt][s2], dh, a2[tt]);
          }
        }
        if (NS == 3 && nt == 0) read_k(sK[stn], sKl[kLo ? stn : 0]);   // of the next chunk (landed since barrier 2)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          s_reg[nt][e] = active ? gam * s_reg[nt][e] + a2[e >> 2][e & 3] : s_reg[nt][e];
      }
      publish_state();
      load(min(c + NS - 1, nch - 1), on);
      phase_barrier();
      if constexpr (NS == 2) read_k(sK[stn], sKl[kLo ? stn : 0]);
    };
    publish_state();
    // Register sets rotate; loads are unconditional (clamped to the last
    // chunk) so that the compiler's wait counts stay exact.
    StateOps o[NS];
#pragma unroll
    for (int i = 0; i < NS - 1; ++i) load(min(i, nch - 1), o[i]);
    __syncthreads();
    read_k(sK[0], sKl[0]);
    for (int c = 0; c < nch; c += NS) {
      chunk(std::integral_constant<int, 0>{}, true, c, o[0], o[NS - 1]);
      chunk(std::integral_constant<int, 1>{}, c + 1 < nch, c + 1, o[1], o[0]);
      if constexpr (NS == 3) chunk(std::integral_constant<int, NS - 1>{}, c + 2 < nch, c + 2, o[NS - 1], o[1]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) Sg[((e >> 2) * 16 + (e & 3)) * kD + nt] = s_reg[nt][e];
  } else {
    // ------------------------------------------------- output and helper waves
    constexpr bool kHelp = NT == 1;
    const bool outw = wave < 8;   // else helper
    using Ops = OutOps<NT, RAW>;
    const int trow = w4 * 16 + g4 * 4;             // first of this lane's 4 token rows
    // first token and V channel this lane forms, and its number of channels
    const int vtok = NT == 1 ? w4 * 16 + (lane >> 2) : trow;
    const int vch = (kLo ? 2 * Hk * kD : 0) + hv * kD + (NT == 1 ? slab * 16 + (lane & 3) * 4 : col);
    constexpr int NV = NT == 1 ? 4 : NT;
    float cw[NV][4];                               // conv taps
    if constexpr (kLo) {
#pragma unroll
      for (int e = 0; e < NV; ++e) {
        const u32x2 w = *reinterpret_cast<const u32x2*>(cv.w + static_cast<size_t>(vch + e) * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) cw[e][i] = bf_at(w, i);
      }
    }
    auto load_v = [&](int c, Ops& o) __attribute__((always_inline)) {
      // V input rows, through a resource that ends at the chunk's last token
      // (rows past it read as zeros). The rows a lane needs start at its first
      // token, less the conv's three (`lead` of which lie before the chunk; in
      // the first chunk those come from the ring, in form_v).
      const int t0 = c * kC, lead = kLo && c > 0 ? 3 : 0, back = kLo ? 3 : 0;
      const int stride = kLo ? cv.stride : Hv * kD;
      const bf16* base = (kLo ? cv.qkv : v) + (static_cast<size_t>(b) * T + t0 - lead) * stride;
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<bf16*>(base), 0, (min(kC, T - t0) + lead) * stride * 2, kBufferRsrcWord3);
#pragma unroll
      for (int i = 0; i < RAW; ++i) {
        const int at = (max(vtok - back + i + lead, 0) * stride + vch) * 2;
        if constexpr (NT == 2) o.v[i][0] = __builtin_amdgcn_raw_buffer_load_b32(rs, at, 0, 0);
        else o.v[i] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, at, 0, 0));
      }
    };
    auto load_qp = [&](int c, Ops& o) __attribute__((always_inline)) {
      const unsigned char* rec = rec_of(c);
      const u32x4* Q = reinterpret_cast<const u32x4*>(krec_of(c) + RK::kQ) + w4 * 256 + lane;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) o.q[ks] = Q[ks * 64];
      const u32x4* P = reinterpret_cast<const u32x4*>(rec + R::kP) + w4 * 128 + lane;
      o.p[0] = P[0];
      if (w4 >= 2) o.p[1] = P[64];
    };
    // V of chunk c (the layer: conv + SiLU of its raw rows), published for the
    // state waves; `first`: chunk 0, whose first rows reach into the ring
    auto form_v = [&](int c, const Ops& o, bool first) __attribute__((always_inline)) {
      constexpr int TOK = NT == 1 ? 1 : 4;         // tokens per lane
      float y[NV][TOK];
#pragma unroll
      for (int e = 0; e < NV; ++e) {
        float x[RAW];
#pragma unroll
        for (int i = 0; i < RAW; ++i) x[i] = bf_at(o.v[i], e);
        if constexpr (kLo) {
          if (first && vtok < 3) {
            const int head = ((cv.head % 3) + 3) % 3;
#pragma unroll
            for (int i = 0; i < 3; ++i)
              if (vtok - 3 + i < 0)
                x[i] = cv.ring[(static_cast<size_t>(b) * 3 + (head + vtok + i) % 3) * cv.ch + vch + e];
          }
#pragma unroll
          for (int j = 0; j < TOK; ++j) {
            float acc = x[j] * cw[e][0];
            acc += x[j + 1] * cw[e][1];
            acc += x[j + 2] * cw[e][2];
            acc += x[j + 3] * cw[e][3];
            const float sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-acc * kLog2e));
            y[e][j] = (c * kC + vtok + j < T) ? acc * sg : 0.f;
          }
        } else {
#pragma unroll
          for (int j = 0; j < TOK; ++j) y[e][j] = x[j];
        }
      }
      if constexpr (NT == 1) {
        *reinterpret_cast<f32x4*>(&sV1[c & 1][vtok * kVRow + (lane & 3) * 4]) = f32x4{y[0][0], y[1][0], y[2][0], y[3][0]};
      } else {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) sV[NT == 2 ? c & 1 : 0][nt][w4][lane] = f32x4{y[nt][0], y[nt][1], y[nt][2], y[nt][3]};
      }
    };
    // K tile(s) and row factors of chunk c -> LDS stage, the wave's share of
    // wave-contiguous KiB. (The DMA builtin makes the compiler wait for every load in flight
    // before the next LDS read; the wrapper's DMAs are ordered by hand below.)
    auto dma_k = [&](int c, unsigned char* kt, unsigned char* klt, float* ft) __attribute__((always_inline)) {
      const u32x4 src = buffer_rsrc(krec_of(c), static_cast<int>(RK::kBytes));
#pragma unroll
      for (int i = 0; i < kTile / 1024 / 4; ++i) {
        const int slot = (i * 4 + w4) * 1024;
        dma16_to_lds(src, static_cast<int>(RK::kK) + slot + lane * 16, kt + slot);
        if constexpr (kLo) dma16_to_lds(src, static_cast<int>(RK::kKLo) + slot + lane * 16, klt + slot);
      }
      const u32x4 fsrc = buffer_rsrc(rec_of(c), 5 * kC * 4);
      if (w4 == 0) dma16_to_lds(fsrc, lane * 16, ft);
      if (w4 == 1 && lane < 16) dma16_to_lds(fsrc, 1024 + lane * 16, ft + 256);
    };
    // Output rows go out through a buffer resource bounded at the chunk's
    // last token, so the stores need no per-row branch (rows past T drop).
    const int rs2 = Hv * kD * 2;   // bytes per token row
    const int lane_off = trow * rs2 + (hv * kD + col) * 2;
    // Three stages: the K tile of chunk cn = c + 2 goes out, V of chunk c + 1 is
    // formed. The K tile of chunk c + 1 must have landed: its DMAs were issued
    // a chunk ago, and the vector memory operations since then (for an output
    // wave also its stores, Q and P, at least one of it) may stay in flight.
    // (V first: its wait for the rows, which the compiler places, would
    // otherwise cover the DMAs just issued.)
    auto supply = [&](int c, int cn, int nst, const Ops& ov, Ops& on) __attribute__((always_inline)) {
      form_v(c + 1, ov, false);
      load_v(cn, on);
      dma_k(cn, sK[nst], sKl[kLo ? nst : 0], &sF[nst][0][0]);
      __builtin_amdgcn_s_waitcnt(vmcnt_imm<(kHelp ? 0 : 4 + 4 + 1) + RAW + kDma>());
    };
    auto helper = [&](auto pos, int c, const Ops& ov, Ops& on) __attribute__((always_inline)) {
      supply(c, min(c + NS - 1, nch - 1), (decltype(pos)::value + NS - 1) % NS, ov, on);
      phase_barrier();
      phase_barrier();
      phase_barrier();
    };
    auto chunk = [&](auto pos, bool active, int c, const Ops& o, const Ops& ov, Ops& on) __attribute__((always_inline)) {
      constexpr int cst = decltype(pos)::value;
      constexpr int nst = (decltype(pos)::value + NS - 1) % NS;   // stage of chunk c + NS - 1 (free since chunk c - 1)
      const int cn = min(c + NS - 1, nch - 1);
      if constexpr (NS == 2) {
        load_v(cn, on);
        dma_k(cn, sK[nst], sKl[kLo ? nst : 0], &sF[nst][0][0]);
        load_qp(cn, on);
      }
      f32x4 acc[NT];
      auto q_s = [&]() __attribute__((always_inline)) {   // Q S with the state of this chunk
        const f32x4 fq = *reinterpret_cast<const f32x4*>(&sF[cst][0][trow]);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
          f32x4 acl = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) {
            acc[nt] = mfma16x16x32(as_bf16x8(o.q[ks]), as_bf16x8(sS[nt][ks][lane]), acc[nt]);
            // split inputs: S as hi + lo (the residual of Q adds ~15% to the
            // scan's operand bytes for no measurable gain: P carries it)
            if constexpr (kLo) acl = mfma16x16x32(as_bf16x8(o.q[ks]), as_bf16x8(sSl[nt][ks][lane]), acl);
          }
          if constexpr (kLo) acc[nt] += acl;
          acc[nt] *= fq;
        }
      };
      // A and B: Q S and the loads of a later chunk. Q S goes first with one
      // column tile; with more, the state waves first have the LDS to themselves
      // for their reads of S (4 tiles, 96 heads: 150 against 157 us a layer).
      if constexpr (kHelp) q_s();
      else if constexpr (NS == 3) supply(c, cn, nst, ov, on);
      phase_barrier();
      if constexpr (NS == 3) load_qp(cn, on);
      if constexpr (!kHelp) q_s();
      phase_barrier();
      // C: + P D, store (an inactive chunk's resource holds no bytes)
      const int t0 = min(c, nch - 1) * kC;
      const __amdgpu_buffer_rsrc_t orsrc = __builtin_amdgcn_make_buffer_rsrc(
          out + (static_cast<size_t>(b) * T + t0) * Hv * kD, 0, active ? min(kC, T - t0) * rs2 : 0, kBufferRsrcWord3);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2)
          if (s2 <= (w4 >> 1))
            acc[nt] = mfma16x16x32(as_bf16x8(o.p[s2]), cat8x2(sD[nt][s2][0][lane], sD[nt][s2][1][lane]), acc[nt]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int at = lane_off + j * rs2;
        if constexpr (NT == 1)
          __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(pack_bf16x2(scale * acc[0][j], 0.f)), orsrc, at, 0, 0);
        else if constexpr (NT == 2)
          __builtin_amdgcn_raw_buffer_store_b32(pack_bf16x2(scale * acc[0][j], scale * acc[1][j]), orsrc, at, 0, 0);
        else
          __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack_bf16x2(scale * acc[0][j], scale * acc[1][j]),
                                                      pack_bf16x2(scale * acc[2][j], scale * acc[3][j])}, orsrc, at, 0, 0);
      }
      if constexpr (NS == 2) {
        // With two stages the K tile of chunk c + 1 was issued in this chunk:
        // only the stores after it may stay in flight.
        form_v(c + 1, ov, false);
        __builtin_amdgcn_s_waitcnt(vmcnt_imm<4>());
      }
      phase_barrier();
    };
    Ops o[NS];
    if (!kHelp || !outw) {
#pragma unroll
      for (int i = 0; i < NS - 1; ++i) {
        dma_k(min(i, nch - 1), sK[i], sKl[kLo ? i : 0], &sF[i][0][0]);
        load_v(min(i, nch - 1), o[i]);
      }
      form_v(0, o[0], true);
    }
    if (outw) {
#pragma unroll
      for (int i = 0; i < NS - 1; ++i) load_qp(min(i, nch - 1), o[i]);
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm<0>());
    __syncthreads();
    if (outw) {
      for (int c = 0; c < nch; c += NS) {
        chunk(std::integral_constant<int, 0>{}, true, c, o[0], o[1], o[NS - 1]);
        chunk(std::integral_constant<int, 1>{}, c + 1 < nch, c + 1, o[1], o[2 % NS], o[0]);
        if constexpr (NS == 3) chunk(std::integral_constant<int, NS - 1>{}, c + 2 < nch, c + 2, o[NS - 1], o[0], o[1]);
      }
    } else if constexpr (kHelp) {
      for (int c = 0; c < nch; c += NS) {
        helper(std::integral_constant<int, 0>{}, c, o[1], o[2]);
        helper(std::integral_constant<int, 1>{}, c + 1, o[2], o[0]);
        helper(std::integral_constant<int, 2>{}, c + 2, o[0], o[1]);
      }
    }
  }
}

template <bool kLo>
void launch_prep(const bf16* q, const bf16* k, const ConvIn& cv, const bf16* a, const bf16* b, int ab_stride,
                 const bf16* dt_bias, const float* A_log, unsigned char* records, int B, int T, int Hk, int Hv,
                 float eps, hipStream_t st) {
  // Value heads per workgroup: all of the key head's, more than four in passes, or
  // shares of two (each forms the key head's tiles and products again). Shares are
  // faster while each finds one of the 256 CUs, and where they replace passes until
  // the whole key heads fill 5/8 of the CUs by themselves. Whole key head / shares,
  // us at n workgroups of whole key heads: recurrence, ratio 16, n = 1 46.0 / 16.6,
  // 64 81.8 / 56.8, 128 94.5 / 79.6, 192 115.8 / 112.3, 256 142.4 / 146.6; ratio 4, 1
  // 19.7 / 16.4, 128 55.5 / 52.5; layer, ratio 16, 1 55.5 / 26.8, 128 134.7 / 127.8,
  // 192 171.7 / 177.4; ratio 8, 128 88.2 / 82.8, 192 111.1 / 114.2, 512 224 / 241;
  // ratio 4, 128 73.4 / 71.5, 192 94.4 / 97.0; ratio 3, 128 69.5 / 69.8, 160 44.7 / 50.0.
  const int G = Hv / Hk, nch = (T + kC - 1) / kC;
  const long whole = static_cast<long>(nch) * Hk * B;
  const int per = whole * ((G + 1) / 2) <= 256 || (G > 4 && whole < 160) ? std::min(G, 2) : G;
  auto go = [&](auto gp) {
    constexpr int GP = decltype(gp)::value;
    hipLaunchKernelGGL((deltanet_chunk_prep_kernel<kLo, GP>), dim3(nch, Hk * ((G + per - 1) / per), B),
                       dim3(kHeadThreads * GP), 0, st, q, k, cv, a, b, ab_stride, dt_bias, A_log, records, T, Hk, Hv,
                       per, eps);
  };
  switch (per) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    default: go(std::integral_constant<int, 4>{}); break;   // in passes of four
  }
}

template <bool kLo>
void launch_scan(const bf16* v, const ConvIn& cv, const unsigned char* records, float* state, bf16* out, int B, int T,
                 int Hk, int Hv, float scale, hipStream_t st) {
  auto go = [&](auto nt) {
    constexpr int NT = decltype(nt)::value;
    hipLaunchKernelGGL((deltanet_chunk_scan_kernel<kLo, NT>), dim3(kD / (16 * NT), Hv, B), dim3(scan_threads(NT)), 0, st,
                       v, cv, records, state, out, T, Hk, Hv, scale);
  };
  // One workgroup per CU; a chunk of 32 or 64 columns takes about 1.25 or 1.75
  // times one of 16. So the narrowest slab that fits one round of 256 CUs wins
  // (layer, us at 16 / 32 / 64 columns: 32 heads, T = 4096 152 / 191 / 261; 48
  // heads, T = 2048 140 / 117 / 152; 64 heads, T = 2048 157 / 131 / 165; 80
  // heads, T = 1024 148 / 141 / 120; 128 heads, T = 1024 173 / 142 / 120).
  const long heads = static_cast<long>(B) * Hv;
  if (heads <= 32) go(std::integral_constant<int, 1>{});
  else if (heads <= 64) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 4>{});
}

}  // namespace

// Records of the chunked prefill.
size_t deltanet_chunk_records_bytes(int B, int T, int Hk, int Hv, bool split) {
  const size_t nch = (static_cast<size_t>(T) + kC - 1) / kC;
  return static_cast<size_t>(B) * nch *
         (Hv * ChunkRec::kBytes + Hk * (split ? KeyRec<true>::kBytes : KeyRec<false>::kBytes));
}

// Chunk records + launches of the two kernels; shared by the recurrence
// entry point (bf16 inputs) and the full layer (split fp32 inputs).
// conv == nullptr: q, k, v planes (bf16 inputs). Otherwise the layer: q, k,
// v are formed from conv->qkv by the kernels (q, k, v unused).
void launch_deltanet_chunked(const bf16* q, const bf16* k, const bf16* v, const ConvIn* conv, const bf16* a,
                             const bf16* b, int ab_stride, const bf16* dt_bias, const float* A_log, float* state,
                             bf16* out, unsigned char* records, int B, int T, int Hk, int Hv, float eps, float scale,
                             hipStream_t st) {
  if (conv) {
    launch_prep<true>(q, k, *conv, a, b, ab_stride, dt_bias, A_log, records, B, T, Hk, Hv, eps, st);
    launch_scan<true>(v, *conv, records, state, out, B, T, Hk, Hv, scale, st);
  } else {
    launch_prep<false>(q, k, ConvIn{}, a, b, ab_stride, dt_bias, A_log, records, B, T, Hk, Hv, eps, st);
    launch_scan<false>(v, ConvIn{}, records, state, out, B, T, Hk, Hv, scale, st);
  }
}
}  // namespace aila

extern "C" size_t aila_hip_deltanet_prefill_workspace_size(int B, int T, int Hv, int dk, int dv) {
  // 0 also for the shapes that run the sequential general-shape kernel
  if (B <= 0 || T <= 0 || Hv <= 0 || dk != 128 || dv != 128) return 0;
  return aila::deltanet_chunk_records_bytes(B, T, Hv, Hv, false);   // at most one key head per value head
}

extern "C" int aila_hip_deltanet_prefill(const void* q, const void* k, const void* v, const void* a,
                                         const void* b, const void* dt_bias, const float* A_log,
                                         float* state, void* out, void* workspace,
                                         size_t workspace_bytes, int B, int T, int Hk, int Hv,
                                         int dk, int dv, float eps, float scale, void* stream) {
  using namespace aila;
  AILA_REQUIRE(q && k && v && a && b && state && out, "deltanet_prefill: null pointer");
  AILA_REQUIRE(B > 0 && B <= 65535 && T > 0 && Hk > 0 && Hv > 0 && Hv <= 65535,
               "deltanet_prefill: bad shape (B=%d T=%d Hk=%d Hv=%d)", B, T, Hk, Hv);
  if (dk != 128 || dv != 128 || Hv % Hk != 0) {
    // general shapes: the token-sequential kernel (no workspace)
    GenericDeltaNet g{};
    g.q = static_cast<const bf16*>(q);
    g.k = static_cast<const bf16*>(k);
    g.v = static_cast<const bf16*>(v);
    g.a = static_cast<const bf16*>(a);
    g.b = static_cast<const bf16*>(b);
    g.ab_stride = Hv;
    g.dt_bias = static_cast<const bf16*>(dt_bias);
    g.A_log = A_log;
    g.state = state;
    g.out = static_cast<bf16*>(out);
    g.B = B, g.T = T, g.Hk = Hk, g.Hv = Hv, g.dk = dk, g.dv = dv, g.K = 1;
    g.eps = eps, g.scale = scale;
    return deltanet_generic_launch(g, static_cast<hipStream_t>(stream), "deltanet_prefill");
  }
  const size_t need = aila_hip_deltanet_prefill_workspace_size(B, T, Hv, dk, dv);
  if (!workspace || workspace_bytes < need)
    return set_error(AILA_HIP_EWORKSPACE, "deltanet_prefill: workspace %zu < %zu bytes", workspace_bytes, need);
  launch_deltanet_chunked(static_cast<const bf16*>(q), static_cast<const bf16*>(k), static_cast<const bf16*>(v),
                          nullptr, static_cast<const bf16*>(a), static_cast<const bf16*>(b), Hv,
                          static_cast<const bf16*>(dt_bias), A_log, state, static_cast<bf16*>(out),
                          static_cast<unsigned char*>(workspace), B, T, Hk, Hv, eps, scale,
                          static_cast<hipStream_t>(stream));
  return check_launch("deltanet_prefill");
}
