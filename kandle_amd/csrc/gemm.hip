// GEMM for the projections: C = alpha * A * B' + beta * Cin (+ bias), fp32 accumulate.
//
//  * bf16 weights, trans_b = 1 (nn.Linear weight [n, k]), m > 8: MFMA tile kernel
//    (v_mfma_f32_32x32x16_bf16); so are most bf16 products of two to eight rows (tile_min_rows: all with bf16
//    results but two short rows against few columns, and those with fp32 results whose rows do not fit LDS).
//  * bf16 weights, m = 1: one-row kernel that reads each weight row once (decode, lm_head); fp32 rows, two to
//    eight, too long for LDS go through it one by one.
//  * otherwise m <= 8, trans_b = 1: skinny kernel, the rows in LDS as fp32.
//  * anything else: LDS-tiled fp32-math kernel.
// The output (and Cin / bias) may be bf16 or fp32 independently of bf16 inputs, e.g. fp32 logits.
//
// Reference semantics: out = alpha * op(A) op(B) + beta * C (packages/core/src/dispatch/matmulOps.ts:32-125;
// epilogue packages/backend-webgpu/src/kernels/matrix/builder.ts:152-218); linear = x W^T + b
// (packages/core/src/dispatch/handlers/composite.ts:55-77).
#include <type_traits>

#include "common.h"
#include "gemv.h"
#include "qk_rope.h"

using namespace kh;
using namespace kh::gemv;

namespace {

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// Four consecutive outputs of one row, vectorised when the row start allows it.
template <typename TO>
__device__ __forceinline__ void store4(TO* C, int64_t off, const float (&v)[4], bool vec, int valid) {
  if (vec && valid == 4) {
    if constexpr (sizeof(TO) == 2) {
      uint2 w;
      w.x = pack_bf16x2(v[0], v[1]);
      w.y = pack_bf16x2(v[2], v[3]);
      *reinterpret_cast<uint2*>(C + off) = w;
    } else {
      *reinterpret_cast<float4*>(C + off) = make_float4(v[0], v[1], v[2], v[3]);
    }
  } else {
    for (int e = 0; e < valid; ++e) Elem<TO>::store(C, off + e, v[e]);
  }
}

// =============================================================================================
// MFMA tile kernel: C = A B^T of K-contiguous rows, a workgroup per GM x GN output tile (and k range).
// The product is formed as C^T = B A^T so that each lane owns one m row and 4 consecutive n per
// register group: A-operand = B rows (n), B-operand = A rows (m), both k-contiguous 16-byte LDS
// reads.  Every output is summed over k in the same 16-wide MFMA steps, in the same order, so the
// tile that holds it does not change its bits.
//
// SPLIT: S workgroups share one output tile, each summing its K range (kchunk columns, a multiple
// of 128) of the products into fp32 partials part[split][m][n] (row-major, leading dimension N);
// gemm_splitk_reduce_kernel -- or a consumer such as kh_add_rms_norm -- then adds the S partials
// in split order (deterministic whichever workgroup finished last) and applies the epilogue.
// SWIGLU (no split): B's rows interleave the gate and up projections in blocks of 8 (rows 16i ..
// 16i + 7: gate rows 8i .. 8i + 7; rows 16i + 8 .. 16i + 15: the matching up rows), so every lane
// holds each gate accumulator and its up partner, and the epilogue stores
// C[m, f] = bf16(silu(bf16(gate)) * bf16(up)) over N / 2 features f -- the values the separate
// GEMM (bf16 store) and silu*mul kernel produce, without the [M, N] intermediate.
// QKNR (no split): the QKV projection of a prefill, whose output columns are head rows of 128 (the
// q heads, then the k heads, then the v heads).  The epilogue stages the tile, rounded to bf16 as
// the plain GEMM stores it, in LDS and reads it back one head row per group of 8 lanes --
// qk_norm_rope_kernel's layout -- to apply qk-norm + RoPE to q and k rows with the same arithmetic
// (qk_norm_rope_row) and write q rows to q_out and k / v rows into the KV cache, so the [M, N]
// projection output is never written.
// =============================================================================================
constexpr int kMaxSplits = 8;

struct QknrArgs {
  const uint16_t* wq = nullptr;       // q_norm / k_norm weights [128], bf16
  const uint16_t* wk = nullptr;
  const float* inv_freq = nullptr;    // [64]
  const int32_t* positions = nullptr; // [M]: RoPE position (and, with kv_cache_len > 0, cache row)
  void* q_out = nullptr;              // the activations' type: bf16, or fp32 with fp32 activations
  void* k_out = nullptr;
  void* v_out = nullptr;
  int64_t s[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};  // (batch, seq, head) element strides of q_out, k_out, v_out
  int hq = 0, hkv = 0;
  uint32_t seq_len = 1;               // token m is (batch m / seq_len, index m % seq_len)
  float eps = 0.f;
  int64_t kv_cache_len = 0;           // > 0: K/V rows at positions[m] (outside [0, len): not written)
  // Optional [M][64][2] (cos, sin) of float(positions[m]) * inv_freq[i] (rope_table_kernel, the same
  // expression): read instead of evaluating sincosf in every head tile.
  const float* rope_cs = nullptr;
};

// The QKNR epilogue of a GM x GN tile (m0, n0) of NW waves: acc[a][b] holds, per lane, output row
// m0 + wm + 32b + r and columns n0 + wn + 32a + 8(j/4) + 4g + j%4 (r = lane & 31, g = lane >> 5).
// smem: the k loop's LDS; the caller has passed a barrier since the loop's last LDS read.
template <typename TA, int AM, int AN, int GM, int GN, int NW>
__device__ __forceinline__ void gemm_qknr_store(const f32x16 (&acc)[AN][AM], uint16_t* smem, int m0, int n0, int wm,
                                                int wn, int M, int N, const QknrArgs& qa) {
  constexpr bool AF = std::is_same<TA, float>::value;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 31, g = lane >> 5;
  static_assert(GN % 128 == 0 && GM % (8 * NW) == 0, "whole head rows of 128");
  // Staged row stride (elements of TA): 272 B (bf16) or 528 B (fp32), 16-byte aligned rows.
  constexpr int TSTR = 128 + 16 / (int)sizeof(TA);
  // The tile is staged as the plain GEMM would store it: rounded to bf16, or fp32 with fp32
  // activations; one head row of 128 columns at a time.
  TA* tile = reinterpret_cast<TA*>(smem);
  // 8 elements of TA at p (16 or 32 bytes) <-> 8 floats
  auto ld8 = [](const TA* p, float (&v)[8]) {
    if constexpr (AF) {
      const float4 x0 = reinterpret_cast<const float4*>(p)[0], x1 = reinterpret_cast<const float4*>(p)[1];
      v[0] = x0.x; v[1] = x0.y; v[2] = x0.z; v[3] = x0.w; v[4] = x1.x; v[5] = x1.y; v[6] = x1.z; v[7] = x1.w;
    } else {
      unpack_bf16x8(*reinterpret_cast<const uint4*>(p), v);
    }
  };
  auto st8 = [](TA* p, const float (&v)[8]) {
    if constexpr (AF) {
      reinterpret_cast<float4*>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
      reinterpret_cast<float4*>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
    } else {
      *reinterpret_cast<uint4*>(p) = pack_bf16x8(v);
    }
  };
  const int t8 = lane & 7, rs = lane >> 3;      // 8 lanes per head row, 8 rows per wave step
  const bool cache_mode = qa.kv_cache_len > 0;
#pragma unroll 1
  for (int hh = 0; hh < GN / 128; ++hh) {
    if (hh > 0) __syncthreads();
    if (wn / 128 == hh) {
#pragma unroll
      for (int a = 0; a < AN; ++a)
#pragma unroll
        for (int b = 0; b < AM; ++b)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            TA* dst = tile + (wm + 32 * b + r) * TSTR + wn % 128 + 32 * a + 8 * q + 4 * g;
            if constexpr (AF) {
              *reinterpret_cast<float4*>(dst) =
                  make_float4(acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2], acc[a][b][4 * q + 3]);
            } else {
              uint2 w;
              w.x = pack_bf16x2(acc[a][b][4 * q], acc[a][b][4 * q + 1]);
              w.y = pack_bf16x2(acc[a][b][4 * q + 2], acc[a][b][4 * q + 3]);
              *reinterpret_cast<uint2*>(dst) = w;
            }
          }
    }
    __syncthreads();
    const int hd = n0 / 128 + hh;               // q heads, then k heads, then v heads
    if (hd * 128 >= N) continue;                // a tile column past the last head
    const bool is_q = hd < qa.hq, is_k = !is_q && hd < qa.hq + qa.hkv;
    float wa[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, wb[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float f[8];
    if (is_q || is_k) {
      const uint16_t* wn8 = is_q ? qa.wq : qa.wk;
      unpack_bf16x8(*reinterpret_cast<const uint4*>(wn8 + 8 * t8), wa);
      unpack_bf16x8(*reinterpret_cast<const uint4*>(wn8 + 64 + 8 * t8), wb);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = qa.inv_freq[8 * t8 + j];
    }
#pragma unroll
    for (int st = 0; st < GM / (8 * NW); ++st) {
      const int row = wave * (GM / NW) + st * 8 + rs;
      const int m = m0 + row;
      const bool live = m < M;
      float a8[8], c8[8];
      ld8(tile + row * TSTR + 8 * t8, a8);
      ld8(tile + row * TSTR + 64 + 8 * t8, c8);
      const int32_t ipos = live ? qa.positions[m] : 0;
      const uint32_t bi = live ? (uint32_t)m / qa.seq_len : 0u, si = live ? (uint32_t)m - bi * qa.seq_len : 0u;
      const int64_t kv_row = cache_mode ? (int64_t)ipos : (int64_t)si;
      const bool kv_ok = !cache_mode || (ipos >= 0 && (int64_t)ipos < qa.kv_cache_len);
      if (is_q || is_k) {
        float cs[8], sn[8], oa[8], oc[8];
        if (qa.rope_cs != nullptr) {
          const float4* t4 = reinterpret_cast<const float4*>(qa.rope_cs + ((int64_t)(live ? m : 0) * 64 + 8 * t8) * 2);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float4 v = t4[j];
            cs[2 * j] = v.x;
            sn[2 * j] = v.y;
            cs[2 * j + 1] = v.z;
            sn[2 * j + 1] = v.w;
          }
        } else {
          const float pos = (float)ipos;
#pragma unroll
          for (int j = 0; j < 8; ++j) sincosf(pos * f[j], &sn[j], &cs[j]);
        }
        qk_norm_rope_row<128>(a8, c8, wa, wb, cs, sn, qa.eps, oa, oc);
        if (live && (is_q || kv_ok)) {
          TA* dst = is_q ? (TA*)qa.q_out + bi * qa.s[0] + si * qa.s[1] + (int64_t)hd * qa.s[2]
                         : (TA*)qa.k_out + bi * qa.s[3] + kv_row * qa.s[4] + (int64_t)(hd - qa.hq) * qa.s[5];
          st8(dst + 8 * t8, oa);
          st8(dst + 64 + 8 * t8, oc);
        }
      } else if (live && kv_ok) {
        TA* dst = (TA*)qa.v_out + bi * qa.s[6] + kv_row * qa.s[7] + (int64_t)(hd - qa.hq - qa.hkv) * qa.s[8];
        st8(dst + 8 * t8, a8);
        st8(dst + 64 + 8 * t8, c8);
      }
    }
  }
}

// The other epilogues, wave by wave, each with its own WLDS bytes of LDS: a register group holds 16
// bytes of a row, so stored as they are the 64 lanes write 32-byte pieces of 32 rows; instead the
// finished blocks of 32 rows are turned in LDS and stored as whole row segments (2000 x 19456 fp32
// outputs, K = 2560, 256 x 128 tiles: 251.7 -> 238.5 us).  (mw, nw): the wave's first output; acc as in
// gemm_qknr_store.  The caller has passed a barrier since the k loop's last LDS read.
template <typename TO, bool AF, int AM, int AN, bool SPLIT, bool SWIGLU>
__device__ __forceinline__ void gemm_wave_store(const f32x16 (&acc)[AN][AM], char* wlds, int mw, int nw,
                                                float* __restrict__ part, TO* C, int64_t ldc, const TO* cin,
                                                int64_t ldcin, const TO* __restrict__ bias, int M, int N, float alpha,
                                                float beta) {
  using TS = std::conditional_t<SWIGLU, TO, float>;          // what is staged
  constexpr int COLS = SWIGLU ? 16 * AN : 32 * AN;           // staged (output) columns of the wave
  constexpr int ROW = COLS * (int)sizeof(TS) + 16;           // bytes per staged row
  constexpr int E = SWIGLU ? 16 / (int)sizeof(TO) : 4;       // outputs per 16-byte chunk
  constexpr int CH = COLS / E, STEPS = 32 * CH / 64;         // chunks per row, chunks per lane
  const int lane = threadIdx.x & 63, r = lane & 31, g = lane >> 5;
  const int NO = SWIGLU ? N / 2 : N, n0 = SWIGLU ? nw / 2 : nw;
  const bool vec = SPLIT || (((reinterpret_cast<uintptr_t>(C) | (cin ? reinterpret_cast<uintptr_t>(cin) : 0) |
                               (bias ? reinterpret_cast<uintptr_t>(bias) : 0)) & 15) == 0 &&
                             ((ldc | (cin ? ldcin : 0)) & 7) == 0);
#pragma unroll
  for (int b = 0; b < AM; ++b) {
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int a = 0; a < AN; ++a)
#pragma unroll
      for (int q = 0; q < 4; q += SWIGLU ? 2 : 1) {
        if constexpr (SWIGLU) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v[e] = AF ? silu_ref(acc[a][b][4 * q + e]) * acc[a][b][4 * q + 4 + e]
                      : silu_ref(round_bf16(acc[a][b][4 * q + e])) * round_bf16(acc[a][b][4 * q + 4 + e]);
          TO* dst = reinterpret_cast<TO*>(wlds + r * ROW) + 16 * a + 4 * q + 4 * g;
          if constexpr (sizeof(TO) == 2)
            *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
          else
            *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
          *reinterpret_cast<float4*>(reinterpret_cast<float*>(wlds + r * ROW) + 32 * a + 8 * q + 4 * g) =
              make_float4(acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2], acc[a][b][4 * q + 3]);
        }
      }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int st = 0; st < STEPS; ++st) {
      const int l = st * 64 + lane, row = l / CH, c = l % CH * E;
      const int m = mw + 32 * b + row, n = n0 + c;
      const uint4 x = *reinterpret_cast<const uint4*>(wlds + row * ROW + c * (int)sizeof(TS));
      if (m >= M || n >= NO) continue;
      if constexpr (SPLIT) {
        *reinterpret_cast<uint4*>(part + (int64_t)m * N + n) = x;   // N % 4 == 0
      } else if constexpr (SWIGLU) {
        TO* dst = C + (int64_t)m * ldc + n;                         // N / 2 is a multiple of 8
        if (vec) {
          *reinterpret_cast<uint4*>(dst) = x;
        } else {
          const TO* xe = reinterpret_cast<const TO*>(&x);
#pragma unroll
          for (int e = 0; e < E; ++e) dst[e] = xe[e];
        }
      } else {
        const float f[4] = {__uint_as_float(x.x), __uint_as_float(x.y), __uint_as_float(x.z), __uint_as_float(x.w)};
        float v[4];
        if (vec && n + 4 <= N) {
          float ci[4] = {0.f, 0.f, 0.f, 0.f}, bi[4] = {0.f, 0.f, 0.f, 0.f};
          auto ld4 = [](const TO* p, float (&o)[4]) {
            if constexpr (sizeof(TO) == 2) {
              const uint2 u = *reinterpret_cast<const uint2*>(p);
              o[0] = lo_bf16(u.x); o[1] = hi_bf16(u.x); o[2] = lo_bf16(u.y); o[3] = hi_bf16(u.y);
            } else {
              const float4 u = *reinterpret_cast<const float4*>(p);
              o[0] = u.x; o[1] = u.y; o[2] = u.z; o[3] = u.w;
            }
          };
          const bool has_c = cin != nullptr && beta != 0.f;
          if (has_c) ld4(cin + (int64_t)m * ldcin + n, ci);
          if (bias != nullptr) ld4(bias + n, bi);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = alpha * f[e];
            if (has_c) v[e] += beta * ci[e];
            if (bias != nullptr) v[e] += bi[e];
          }
          store4<TO>(C, (int64_t)m * ldc + n, v, true, 4);
        } else {
          const int valid = min(4, N - n);
          for (int e = 0; e < valid; ++e)
            Elem<TO>::store(C, (int64_t)m * ldc + n + e,
                            epilogue<TO>(f[e], alpha, beta, cin, ldcin, bias, m, n + e));
        }
      }
    }
  }
}

// TA = float (fp32 activations, the reference's float32 arithmetic): A stays fp32 in LDS, and each value
// a of a fragment is split into bf16 hi = bf16(a) and lo = bf16(a - hi) (a - hi is exact in fp32); every
// 16-wide step then runs two MFMAs into the same accumulator, W * hi and W * lo.  The weights are exactly
// bf16, so each product is W * a up to the 2^-17 relative error of hi + lo, fp32 accumulate; the
// epilogues keep their fp32 values (no bf16 rounding of the SwiGLU operands or of the qk-norm + RoPE
// input) and store fp32.
//
// What bounds it: for a few hundred rows, the latency of the loads and of the LDS and MFMA chain of each
// k-step; for thousands of rows, the matrix cores and the power they draw.  So A and B rows go from
// memory straight to LDS (buffer_load ... lds, 16 bytes a lane): a stage of the k loop costs no registers,
// up to five of them are in flight, and there is one barrier per stage.  A wave's copy writes 1 KiB of
// consecutive LDS bytes, so rows are stored without padding and the 16-byte chunks of a row are permuted
// instead (chunk c of row i at place c ^ swz(i)): the 16 lanes that one cycle of a fragment read serves
// then fall on 16 different bank groups (no bank conflicts counted in the k loop).  Measured against the register-staged
// kernel before it (two LDS buffers, 64 x 64 to 128 x 128 tiles), one call, weights from HBM:
//   bf16  512 x 4096 x 1024  13.0 ->  9.4 us     fp32  512 x 4096 x 1024  19.3 -> 14.8 us
//   bf16 1000 x 4096 x 1024  19.9 -> 14.4 us     fp32 1000 x 4096 x 1024  30.4 -> 23.1 us
//   bf16 1000 x 6144 x 1024  30.9 -> 20.1 us     fp32 1000 x 6144 x 1024  55.1 -> 33.0 us
//   bf16 2000 x 19456 x 2560  339 ->  240 us     fp32 2000 x 19456 x 2560  600 -> 405 us
// Rows past M or N repeat the last one and are never stored; columns past the k range read as zero.
//
// PARTS (bf16 activations, long fp32 sums of few tiles): each of a stage's four 16-wide steps has an
// accumulator of its own, added at the end: the chains of fp32 additions are those of a product split in
// four.  A chain of n steps is about 2^-24 sqrt(n / 6) of the result off: 640 x 1024 x 2048 1.3e-7 against
// 64 bits (one accumulator 2.7e-7), 256 x 2560 x 9728 3.0e-7 (6.3e-7), 128 x 4096 x 1024 split in two
// 8e-8 (1.3e-7).  The additions at the end take 0.2-0.3 us (640 x 1024 x 2048 8.8 -> 9.1).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// 64 lanes x 16 bytes from rsrc at byte voff (per lane) + soff to LDS byte address lds + 16 lane.
// Asynchronous: complete once a later s_waitcnt vmcnt says so.  (Inline asm rather than the builtin,
// after which the compiler waits for every copy in flight before it reads any LDS.  m0 is reserved:
// the compiler sets it anew before each use of its own.)
__device__ __forceinline__ void copy_to_lds16(u32x4 rsrc, uint32_t voff, uint32_t soff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff)
               : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vmem() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
// Wait until at most `left` stages of LPS copies each are in flight (left <= MAX).
template <int LPS, int MAX>
__device__ __forceinline__ void wait_stages(int left) {
  if constexpr (MAX <= 0) {
    wait_vmem<0>();
  } else {
    if (left >= MAX)
      wait_vmem<LPS * MAX>();
    else
      wait_stages<LPS, MAX - 1>(left);
  }
}
__device__ __forceinline__ u32x4 raw_rsrc(const void* base, uint32_t bytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  u32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane((uint32_t)p);
  r[1] = __builtin_amdgcn_readfirstlane((uint32_t)(p >> 32));
  r[2] = __builtin_amdgcn_readfirstlane(bytes);
  r[3] = 0x00020000u;
  return r;
}

// A workgroup of WM x WN waves, each 32 AM x 32 AN outputs; NST stages of KS columns in LDS.
template <typename TA, int AM, int AN, int WM, int WN, int KS>
struct DmaTile {
  static constexpr int GM = 32 * AM * WM, GN = 32 * AN * WN, NW = WM * WN;
  static constexpr int CA = KS * (int)sizeof(TA) / 16, CB = KS * 2 / 16;   // 16-byte chunks per row
  static constexpr int ABYTES = GM * CA * 16, BBYTES = GN * CB * 16, STAGE = ABYTES + BBYTES;
  static constexpr int LA = GM * CA / (64 * NW), LB = GN * CB / (64 * NW); // copies per wave and stage
  static_assert(GM * CA % (64 * NW) == 0 && GN * CB % (64 * NW) == 0, "whole copies");
};
// Rows that share one place of a chunk: 16 / C rows fill the 256 bytes of the 64 banks.
template <int C>
__device__ __forceinline__ int lds_swz(int row) {
  static_assert(C == 4 || C == 8 || C == 16, "4, 8 or 16 chunks per row");
  return (row / (16 / C)) & (C - 1);
}

template <typename TO, int AM, int AN, int WM, int WN, int KS, int NST, bool SPLIT, bool SWIGLU, bool QKNR,
          bool PARTS, typename TA>
__global__ __launch_bounds__(64 * WM * WN) void gemm_tile_kernel(
    const TA* __restrict__ A, int64_t lda, const uint16_t* __restrict__ B, int64_t ldb, TO* C, int64_t ldc,
    const TO* cin, int64_t ldcin, const TO* __restrict__ bias, int M, int N, int K, float alpha, float beta,
    int splits, int kchunk, float* __restrict__ part, QknrArgs qa) {
  using T = DmaTile<TA, AM, AN, WM, WN, KS>;
  constexpr bool AF = std::is_same<TA, float>::value;
  constexpr int GM = T::GM, GN = T::GN, NW = T::NW, LPS = T::LA + T::LB;
  constexpr int WLDS = 32 * (32 * AN * 4 + 16);  // a wave's 32 output rows, fp32 (gemm_wave_store)
  constexpr int EPI = QKNR ? GM * (128 + 16 / (int)sizeof(TA)) * (int)sizeof(TA) : NW * WLDS;
  constexpr int BYTES = NST * T::STAGE > EPI ? NST * T::STAGE : EPI;
  __shared__ __attribute__((aligned(1024))) uint16_t smem[BYTES / 2];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int r = lane & 31, g = lane >> 5;
  int bid = blockIdx.x;
  if ((gridDim.x & 7) == 0) bid = (bid & 7) * (gridDim.x >> 3) + (bid >> 3);
  const int tiles_m = (M + GM - 1) / GM;
  const int tile = SPLIT ? bid / splits : bid, split = SPLIT ? bid % splits : 0;
  const int m0 = tile % tiles_m * GM, n0 = tile / tiles_m * GN;
  const int wm = wave / WN * 32 * AM, wn = wave % WN * 32 * AN;
  const int kbeg = split * kchunk, klen = min(K, kbeg + kchunk) - kbeg, nk = (klen + KS - 1) / KS;

  const int mrows = min(GM, M - m0), nrows = min(GN, N - n0);
  const u32x4 ra = raw_rsrc(A + (int64_t)m0 * lda + kbeg, (uint32_t)(((int64_t)(mrows - 1) * lda + klen) * sizeof(TA)));
  const u32x4 rb = raw_rsrc(B + (int64_t)n0 * ldb + kbeg, (uint32_t)(((int64_t)(nrows - 1) * ldb + klen) * 2));
  // (128 rows of either operand fit 2 GiB, so the up to 256 of a tile fit 32-bit byte offsets.)
  // Copy i of a stage holds chunk (i NW + wave) 64 + lane of its rows.  The copies of a wave are a
  // multiple of 16 rows apart, so the lane's place in the row -- and its first column ka, kb -- is the
  // same in each.
  uint32_t va[T::LA], vb[T::LB];
  const int l0 = wave * 64 + lane;
  static_assert(NW * 64 / T::CA % 16 == 0 && NW * 64 / T::CB % 16 == 0, "copies whole swizzle periods apart");
  const int ca = (l0 % T::CA) ^ lds_swz<T::CA>(l0 / T::CA), cb = (l0 % T::CB) ^ lds_swz<T::CB>(l0 / T::CB);
  const int ka = ca * (16 / (int)sizeof(TA)), kb = cb * 8;
#pragma unroll
  for (int i = 0; i < T::LA; ++i)
    va[i] = (uint32_t)min((i * NW * 64 + l0) / T::CA, mrows - 1) * (uint32_t)(lda * sizeof(TA)) + 16u * ca;
#pragma unroll
  for (int i = 0; i < T::LB; ++i)
    vb[i] = (uint32_t)min((i * NW * 64 + l0) / T::CB, nrows - 1) * (uint32_t)(ldb * 2) + 16u * cb;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem;
  // Copy i of this wave's LPS copies of stage t into buffer buf.  A chunk past the k range (K % 8 == 0:
  // all in or all out) takes an offset past the buffer's, which reads zero.
  auto issue_one = [&](int t, int buf, int i) {
    const uint32_t base = lds0 + (uint32_t)(buf * T::STAGE + wave * 1024);
    if (i < T::LA)
      copy_to_lds16(ra, t * KS + ka < klen ? va[i < T::LA ? i : 0] : 0xffffffffu,
                    (uint32_t)(t * KS * (int)sizeof(TA)), base + i * NW * 1024);
    else
      copy_to_lds16(rb, t * KS + kb < klen ? vb[i < T::LA ? 0 : i - T::LA] : 0xffffffffu, (uint32_t)(t * KS * 2),
                    base + T::ABYTES + (i - T::LA) * NW * 1024);
  };

  constexpr int KC = KS / 16, ALL = KC * AN;  // 16-wide steps of a stage, and places between its products
  constexpr int SETS = PARTS ? KC : 1;
  f32x16 sums[SETS][AN][AM];
#pragma unroll
  for (int s = 0; s < SETS; ++s)
#pragma unroll
    for (int a = 0; a < AN; ++a)
#pragma unroll
      for (int b = 0; b < AM; ++b)
#pragma unroll
        for (int j = 0; j < 16; ++j) sums[s][a][b][j] = 0.f;
  auto& acc = sums[0];
  // Fragments of one 16-wide k step: B rows, and A rows as stored (fp32: two 16-byte halves) until
  // split_a makes them bf16 (fp32: hi and lo).
  constexpr int AW = AF ? 2 : 1;
  struct Frag {
    uint4 b[AN], a[AM][AW];
  };
  auto read_frag = [&](Frag& f, int buf, int kc) {
    const char* as = reinterpret_cast<const char*>(smem) + buf * T::STAGE;
    const char* bs = as + T::ABYTES;
#pragma unroll
    for (int b = 0; b < AM; ++b) {
      const int row = wm + 32 * b + r;
#pragma unroll
      for (int h = 0; h < AW; ++h)
        f.a[b][h] = *reinterpret_cast<const uint4*>(as + row * (T::CA * 16) +
                                                    (((AW * (2 * kc + g) + h) ^ lds_swz<T::CA>(row)) * 16));
    }
#pragma unroll
    for (int a = 0; a < AN; ++a) {
      const int row = wn + 32 * a + r;
      f.b[a] = *reinterpret_cast<const uint4*>(bs + row * (T::CB * 16) + (((2 * kc + g) ^ lds_swz<T::CB>(row)) * 16));
    }
  };
  auto split_a = [&](Frag& f) {
    if constexpr (AF) {
#pragma unroll
      for (int b = 0; b < AM; ++b) {
        const float4 x = __builtin_bit_cast(float4, f.a[b][0]), y = __builtin_bit_cast(float4, f.a[b][AW - 1]);
        const uint32_t h0 = pack_bf16x2(x.x, x.y), h1 = pack_bf16x2(x.z, x.w), h2 = pack_bf16x2(y.x, y.y),
                       h3 = pack_bf16x2(y.z, y.w);
        f.a[b][0] = make_uint4(h0, h1, h2, h3);
        f.a[b][AW - 1] = make_uint4(pack_bf16x2(x.x - lo_bf16(h0), x.y - hi_bf16(h0)),
                                    pack_bf16x2(x.z - lo_bf16(h1), x.w - hi_bf16(h1)),
                                    pack_bf16x2(y.x - lo_bf16(h2), y.y - hi_bf16(h2)),
                                    pack_bf16x2(y.z - lo_bf16(h3), y.w - hi_bf16(h3)));
      }
    }
  };
  // kc: the step of its stage that f holds
  auto multiply = [&](const Frag& f, int kc, int pl, auto&& between) {
    auto& to = sums[PARTS ? kc : 0];
#pragma unroll
    for (int a = 0; a < AN; ++a) {
#pragma unroll
      for (int b = 0; b < AM; ++b)
        to[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(f.b[a]), as_bf16x8(f.a[b][pl]), to[a][b], 0, 0, 0);
      between(a);
    }
  };
  auto nothing = [](int) {};
  // One 16-wide step: read the next step's (kc) fragments, multiply this one's (kc - 1, or the last); with fp32 activations the
  // next fragments are split in the shadow of the second plane's products.
  auto step = [&](Frag& cur, Frag& nxt, int buf, int kc, auto&& between) {
    read_frag(nxt, buf, kc);
    __builtin_amdgcn_sched_barrier(0);
    multiply(cur, (kc + KC - 1) % KC, 0, between);
    if constexpr (AF) {
      __builtin_amdgcn_sched_barrier(0);
      split_a(nxt);
      multiply(cur, (kc + KC - 1) % KC, AW - 1, nothing);
#pragma unroll
      for (int i = 0; i < AN * AM; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                            // one MFMA
        __builtin_amdgcn_sched_group_barrier(0x2, (24 + AN - 1) / AN, 0);           // its share of the split
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // The fragments of the next 16-wide step are read before the current one is multiplied.  The last
  // step of a stage is multiplied after the barrier that opens the next stage: there every wave's
  // copies of that stage are complete, and every wave has read all of this stage, whose buffer takes
  // the copies of the stage NST later.  Those are issued one by one between the products of the steps
  // that follow, up to the next stage's barrier: issued together they keep the matrix cores waiting
  // for the address unit (64 bytes per cycle).
  Frag fr[2];
  if (nk > 0) {
#pragma unroll
    for (int s = 0; s < NST; ++s)
      if (s < nk) {
#pragma unroll
        for (int i = 0; i < LPS; ++i) issue_one(s, s, i);
      }
    wait_stages<LPS, NST - 1>(nk - 1);
    __builtin_amdgcn_s_barrier();
    read_frag(fr[0], 0, 0);
    split_a(fr[0]);
    int buf = 0;
    // Slots sl0 .. sl0 + AN - 1 of the ALL between two barriers: the copies of stage it.
    auto copies = [&](int sl0, int it, int ibuf) {
      return [&, sl0, it, ibuf](int i) {
        const int k0 = (sl0 + i) * LPS / ALL, k1 = (sl0 + i + 1) * LPS / ALL;
        if (k1 > k0) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int k = 0; k < LPS; ++k)
            if (k >= k0 && k < k1) issue_one(it, ibuf, k);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
    };
    constexpr int kLgkm0 = 0xc07f;  // s_waitcnt lgkmcnt(0)
#pragma unroll
    for (int kc = 0; kc + 1 < KC; ++kc) step(fr[kc & 1], fr[(kc + 1) & 1], 0, kc + 1, nothing);
    int t = 0;
    // Entering an iteration: stage t is read, its last step not yet multiplied, and stages up to
    // t + NST - 1 are requested.
    for (; t + NST < nk; ++t) {
      __builtin_amdgcn_s_waitcnt(kLgkm0);
      wait_vmem<LPS*(NST - 2)>();
      const int ibuf = buf;
      buf = buf == NST - 1 ? 0 : buf + 1;
      __builtin_amdgcn_s_barrier();
      step(fr[1], fr[0], buf, 0, copies(0, t + NST, ibuf));
#pragma unroll
      for (int kc = 0; kc + 1 < KC; ++kc)
        step(fr[kc & 1], fr[(kc + 1) & 1], buf, kc + 1, copies((kc + 1) * AN, t + NST, ibuf));
    }
    for (; t + 1 < nk; ++t) {  // nothing left to request
      __builtin_amdgcn_s_waitcnt(kLgkm0);
      wait_stages<LPS, NST - 2>(nk - 2 - t);
      buf = buf == NST - 1 ? 0 : buf + 1;
      __builtin_amdgcn_s_barrier();
      step(fr[1], fr[0], buf, 0, nothing);
#pragma unroll
      for (int kc = 0; kc + 1 < KC; ++kc) step(fr[kc & 1], fr[(kc + 1) & 1], buf, kc + 1, nothing);
    }
    multiply(fr[1], KC - 1, 0, nothing);
    if constexpr (AF) multiply(fr[1], KC - 1, AW - 1, nothing);
    if constexpr (PARTS) {
      static_assert(!AF && KC == 4, "four steps per stage");
#pragma unroll
      for (int a = 0; a < AN; ++a)
#pragma unroll
        for (int b = 0; b < AM; ++b)
#pragma unroll
          for (int j = 0; j < 16; ++j)
            acc[a][b][j] = (acc[a][b][j] + sums[1][a][b][j]) + (sums[SETS - 2][a][b][j] + sums[SETS - 1][a][b][j]);
    }
  }
  __syncthreads();  // the tile is stored by way of the loop's LDS
  if constexpr (QKNR) {
    gemm_qknr_store<TA, AM, AN, GM, GN, NW>(acc, smem, m0, n0, wm, wn, M, N, qa);
  } else {
    gemm_wave_store<TO, AF, AM, AN, SPLIT, SWIGLU>(acc, reinterpret_cast<char*>(smem) + wave * WLDS, m0 + wm, n0 + wn,
                                                   SPLIT ? part + (int64_t)split * M * N : nullptr, C, ldc, cin, ldcin,
                                                   bias, M, N, alpha, beta);
  }
}

// Split-K reduction: one thread per four consecutive outputs (N % 4 == 0), so every partial of the
// whole output is in flight at once; the splits are added in split order from 0, then the epilogue.
template <typename TO>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(const float* __restrict__ part, int splits,
                                                                  TO* C, int64_t ldc, const TO* cin, int64_t ldcin,
                                                                  const TO* __restrict__ bias, int M, int N,
                                                                  float alpha, float beta) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t mn = (int64_t)M * N;
  if (gid * 4 >= mn) return;
  const int m = (int)(gid * 4 / N), n = (int)(gid * 4 % N);
  const float* tp = part + gid * 4;
  float4 pv[kMaxSplits];
#pragma unroll
  for (int s2 = 0; s2 < kMaxSplits; ++s2)
    pv[s2] = s2 < splits ? *reinterpret_cast<const float4*>(tp + s2 * mn) : make_float4(0.f, 0.f, 0.f, 0.f);
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s2 = 0; s2 < kMaxSplits; ++s2) {
    v[0] += pv[s2].x;
    v[1] += pv[s2].y;
    v[2] += pv[s2].z;
    v[3] += pv[s2].w;
  }
  const bool vec = ((reinterpret_cast<uintptr_t>(C) & (4 * sizeof(TO) - 1)) == 0) && ((ldc & 3) == 0);
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = epilogue<TO>(v[e], alpha, beta, cin, ldcin, bias, m, n + e);
  store4<TO>(C, (int64_t)m * ldc + n, v, vec, 4);
}

// =============================================================================================
// Skinny kernel for m <= 8 (trans_b = 1, rows that fit 64 KiB of LDS; bf16 ones mostly take the tiles,
// tile_min_rows): each wave owns output columns n and streams weight row n
// once with 16-byte loads; the m rows of A are kept in LDS as fp32.
// =============================================================================================
constexpr int SK_MAXM = 8;
constexpr int SK_ROWS_PER_WAVE = 4;  // weight rows in flight per wave step

template <typename TA, typename T, typename TO>
__global__ __launch_bounds__(256) void gemv_nt_kernel(const TA* __restrict__ A, int64_t lda, const T* __restrict__ B,
                                                      int64_t ldb, TO* C, int64_t ldc, const TO* cin, int64_t ldcin,
                                                      const TO* __restrict__ bias, int M, int N, int K, float alpha,
                                                      float beta) {
  extern __shared__ float xs[];  // [M][K] fp32
  for (int i = threadIdx.x; i < M * K; i += blockDim.x) {
    const int mm = i / K, kk = i % K;
    xs[i] = Elem<TA>::load(A, (int64_t)mm * lda + kk);
  }
  __syncthreads();
  constexpr int EPL = 16 / sizeof(T);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int waves_total = gridDim.x * (blockDim.x >> 6);
  const int wid = blockIdx.x * (blockDim.x >> 6) + w;
  const bool vec = (K % EPL == 0) && (ldb % EPL == 0);
  for (int n0 = wid * SK_ROWS_PER_WAVE; n0 < N; n0 += waves_total * SK_ROWS_PER_WAVE) {
    float acc[SK_ROWS_PER_WAVE][SK_MAXM];
#pragma unroll
    for (int rr = 0; rr < SK_ROWS_PER_WAVE; ++rr)
#pragma unroll
      for (int mm = 0; mm < SK_MAXM; ++mm) acc[rr][mm] = 0.f;
    if (vec) {
      for (int k0 = lane * EPL; k0 < K; k0 += 64 * EPL) {
        uint4 wv[SK_ROWS_PER_WAVE];
#pragma unroll
        for (int rr = 0; rr < SK_ROWS_PER_WAVE; ++rr) {
          const int n = n0 + rr;
          wv[rr] = n < N ? *reinterpret_cast<const uint4*>(B + (int64_t)n * ldb + k0) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int rr = 0; rr < SK_ROWS_PER_WAVE; ++rr) {
          float wf[EPL];
          if constexpr (sizeof(T) == 2) {
            const uint32_t u[4] = {wv[rr].x, wv[rr].y, wv[rr].z, wv[rr].w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              wf[2 * e] = lo_bf16(u[e]);
              wf[2 * e + 1] = hi_bf16(u[e]);
            }
          } else {
            wf[0] = __uint_as_float(wv[rr].x); wf[1] = __uint_as_float(wv[rr].y);
            wf[2] = __uint_as_float(wv[rr].z); wf[3] = __uint_as_float(wv[rr].w);
          }
#pragma unroll
          for (int mm = 0; mm < SK_MAXM; ++mm) {
            if (mm < M) {
              float s = 0.f;
#pragma unroll
              for (int e = 0; e < EPL; ++e) s += wf[e] * xs[mm * K + k0 + e];
              acc[rr][mm] += s;
            }
          }
        }
      }
    } else {
      for (int kk = lane; kk < K; kk += 64)
#pragma unroll
        for (int rr = 0; rr < SK_ROWS_PER_WAVE; ++rr) {
          const int n = n0 + rr;
          const float wf = n < N ? Elem<T>::load(B, (int64_t)n * ldb + kk) : 0.f;
#pragma unroll
          for (int mm = 0; mm < SK_MAXM; ++mm)
            if (mm < M) acc[rr][mm] += wf * xs[mm * K + kk];
        }
    }
#pragma unroll
    for (int rr = 0; rr < SK_ROWS_PER_WAVE; ++rr)
#pragma unroll
      for (int mm = 0; mm < SK_MAXM; ++mm) {
        if (mm < M) {
          const float s = wave_sum(acc[rr][mm]);
          const int n = n0 + rr;
          if (lane == 0 && n < N)
            Elem<TO>::store(C, (int64_t)mm * ldc + n, epilogue<TO>(s, alpha, beta, cin, ldcin, bias, mm, n));
        }
      }
  }
}

// =============================================================================================
// One-row GEMV (decode: m = 1, bf16 weight [n, k], trans_b = 1) with an optional fused prologue
// that forms the activation row the way the unfused ops would have stored it (bf16):
//   PRO_NONE      x' = x                               (x bf16)
//   PRO_RMSNORM   x' = bf16(rms_norm(x, norm_w, eps))  (x fp32 residual row, norm_w bf16)
//   PRO_SILU_MUL  x' = bf16(silu(x) * x2)              (x, x2 bf16: gate and up halves)
//   PRO_SILU_MUL_IL x'[i] = bf16(silu(x[16(i/8) + i%8]) * x[16(i/8) + 8 + i%8])  (x bf16 [2k]: the
//                 gate/up row of a projection whose weight interleaves gate and up rows in blocks of 8)
//   PRO_ATTN_MERGE x' = bf16(split-K decode attention merged)  (x: the fp32 partials of one sequence,
//                 o[h][chunk][128] then (m, l)[h][chunk]; see AttnMerge)
// Each workgroup forms x' once in LDS (fp32, zero past k); each wave then owns U weight rows and
// streams them with raw 16-byte buffer loads, CB chunks of 512 columns per row in flight (rows past
// n read as zero), and reduces each row across the wave.  Every weight byte is read once.
// =============================================================================================
template <int U, int PRO, typename TO, bool PAIR8 = false, bool EX = false>
__global__ __launch_bounds__(256) void gemv1_kernel(const void* __restrict__ x, const void* __restrict__ x2,
                                                    const uint16_t* __restrict__ nw, float eps,
                                                    const uint16_t* __restrict__ W, int64_t ldw, uint32_t w_bytes,
                                                    TO* C, const TO* cin, const TO* __restrict__ bias, int N, int K,
                                                    int nch, float alpha, float beta, AttnMerge am) {
  extern __shared__ float xs[];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  GemvRows<U, PAIR8, EX> g;
  g.init(W, ldw, w_bytes, N, K, nch, (int64_t)blockIdx.x * (blockDim.x >> 6) + w,
         (int64_t)gridDim.x * (blockDim.x >> 6));
  GemvPrologue<PRO, EX> pro;
  pro.load(x, nw, K, nch * GV_CHUNK, am);
  __builtin_amdgcn_sched_barrier(0);
  // The first batch is in flight while the workgroup forms x'.
  g.issue_first();
  __builtin_amdgcn_sched_barrier(0);
  pro.finish(xs, x, x2, nw, eps, K, nch * GV_CHUNK, am);
  g.template run<TO>(xs, C, cin, bias, alpha, beta);
}

// x' is staged in LDS as fp32: k <= 32768 (128 KiB of the CU's 160 KiB; above 64 KiB one
// workgroup per CU, the size of the down projections of 14B- and 32B-class models).
constexpr size_t kGemvMaxLds = 128 * 1024;

// Launches gemv1_kernel; returns false (nothing launched) when the operands do not fit its
// assumptions (16-byte aligned weight rows, 32-bit byte offsets, x' within kGemvMaxLds of LDS) or
// the runtime refuses the workgroup's LDS size.
template <int U, int PRO, typename TO, bool PAIR8 = false, bool EX = false>
bool gemv1_go(const void* x, const void* x2, const void* nw, float eps, const uint16_t* W, int64_t ldw,
              uint32_t w_bytes, TO* C, const TO* cin, const TO* bias, int N, int K, int nch, float alpha, float beta,
              const AttnMerge& am) {
  const int64_t waves = (N + U - 1) / U;
  int64_t grid = (waves + 3) / 4;
  // Waves stride over the rows past the first grid: lm_head (151936 rows, 8 per wave) at most 2048
  // workgroups: 69.5 -> 59.9 us graph-replayed with 4 rows per wave and 8192 workgroups before.
  if (grid > 2048) grid = 2048;
  const size_t shm = (size_t)nch * GV_CHUNK * sizeof(float);
  if (shm > 64 * 1024) {
    // dynamic LDS above 64 KiB is opted into once per kernel instantiation
    static const bool raised = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemv1_kernel<U, PRO, TO, PAIR8, EX>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   (int)kGemvMaxLds) == hipSuccess;
    if (!raised) return false;
  }
  gemv1_kernel<U, PRO, TO, PAIR8, EX><<<(int)grid, 256, shm, stream()>>>(x, x2, (const uint16_t*)nw, eps, W, ldw,
                                                                         w_bytes, C, cin, bias, N, K, nch, alpha,
                                                                         beta, am);
  return true;
}

// The weight rows a one-row projection may address fit 32-bit byte offsets: row groups start below
// N and hold U rows, so the largest row index formed is N - 1 + U - 1 (rows at or past N are never
// stored, and the buffer range reads them as zero).
inline bool gemv_offsets_fit(int N, int U, int64_t ldw) {
  return ((int64_t)(N + U) * ldw) * 2 < (int64_t(1) << 32);
}

// SwiGLU one-row projection: h[f] = bf16(silu(bf16(gate_f)) * bf16(up_f)) (EX: silu(gate_f) * up_f in
// fp32, TO float) from the interleaved gate/up weight (2 * n_half rows, blocks of 8), one wave per
// (gate, up) row pair.  False when the operands do not fit (as launch_gemv1).
template <int PRO, bool EX = false, typename TO = uint16_t>
bool launch_gemv_swiglu(const void* x, const void* nw, float eps, const uint16_t* W, int64_t ldw, TO* H,
                        int n_half, int K) {
  const int N = 2 * n_half;
  if (n_half <= 0 || n_half % 8 != 0 || K <= 0) return false;
  const int nch = (K + GV_CHUNK - 1) / GV_CHUNK;
  const int64_t w_bytes = ((int64_t)(N - 1) * ldw + K) * 2;
  // a pair of row group q addresses rows up to 16 (q / 8) + q % 8 + 8 < N + 8
  if (K % 8 != 0 || ldw % 8 != 0 || !aligned16(W) || !gemv_offsets_fit(N, 8, ldw) ||
      (size_t)nch * GV_CHUNK * sizeof(float) > kGemvMaxLds)
    return false;
  return gemv1_go<2, PRO, TO, true, EX>(x, nullptr, nw, eps, W, ldw, (uint32_t)w_bytes, H, nullptr, nullptr, N, K, nch,
                                        1.f, 0.f, AttnMerge{});
}

template <int PRO, typename TO, bool EX = false>
bool launch_gemv1(const void* x, const void* x2, const void* nw, float eps, const uint16_t* W, int64_t ldw, TO* C,
                  const TO* cin, const TO* bias, int N, int K, float alpha, float beta, const AttnMerge& am = {}) {
  if (N <= 0 || K <= 0) return false;
  const int nch = (K + GV_CHUNK - 1) / GV_CHUNK;
  const int64_t w_bytes = ((int64_t)(N - 1) * ldw + K) * 2;
  const int U = N >= 16384 ? 8 : (N >= 2048 ? 2 : 1);
  if (K % 8 != 0 || ldw % 8 != 0 || !aligned16(W) || !gemv_offsets_fit(N, U, ldw) ||
      (size_t)nch * GV_CHUNK * sizeof(float) > kGemvMaxLds)
    return false;
  const uint32_t wb = (uint32_t)w_bytes;
  if (U == 8) return gemv1_go<8, PRO, TO, false, EX>(x, x2, nw, eps, W, ldw, wb, C, cin, bias, N, K, nch, alpha, beta, am);
  if (U == 2) return gemv1_go<2, PRO, TO, false, EX>(x, x2, nw, eps, W, ldw, wb, C, cin, bias, N, K, nch, alpha, beta, am);
  return gemv1_go<1, PRO, TO, false, EX>(x, x2, nw, eps, W, ldw, wb, C, cin, bias, N, K, nch, alpha, beta, am);
}

// =============================================================================================
// Generic tiled kernel (f32 or bf16 storage, trans_b 0/1): 16 x 16 threads, 64 x 64 tile, each
// thread 4 x 4 outputs, fp32 math.
// =============================================================================================
template <typename TA, typename T, typename TO>
__global__ __launch_bounds__(256) void gemm_generic_kernel(const TA* __restrict__ A, int64_t lda,
                                                           const T* __restrict__ B, int64_t ldb, TO* C, int64_t ldc,
                                                           const TO* cin, int64_t ldcin, const TO* __restrict__ bias,
                                                           int M, int N, int K, float alpha, float beta, int trans_b) {
  __shared__ float As[16][64 + 1];
  __shared__ float Bs[16][64 + 1];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += 16) {
    for (int i = threadIdx.x; i < 16 * 64; i += 256) {
      const int kk = i / 64, mm = i % 64;
      const int gm = m0 + mm, gk = k0 + kk;
      As[kk][mm] = (gm < M && gk < K) ? Elem<TA>::load(A, (int64_t)gm * lda + gk) : 0.f;
      const int gn = n0 + mm;
      float bv = 0.f;
      if (gn < N && gk < K)
        bv = trans_b ? Elem<T>::load(B, (int64_t)gn * ldb + gk) : Elem<T>::load(B, (int64_t)gk * ldb + gn);
      Bs[kk][mm] = bv;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += As[kk][ty * 4 + i] * Bs[kk][tx * 4 + j];
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = m0 + ty * 4 + i, n = n0 + tx * 4 + j;
      if (m < M && n < N)
        Elem<TO>::store(C, (int64_t)m * ldc + n, epilogue<TO>(acc[i][j], alpha, beta, cin, ldcin, bias, m, n));
    }
}

// The tiles, and what the choice among them rests on: microseconds of one 64-wide k-step with every CU
// busy (from calls of 200 to 2000 rows; bf16 and fp32 activations) and of a tile's prologue and
// epilogue.  Per output the large tiles cost the least, but a call takes as many rounds of 256
// workgroups as its tiles need, so the choice is the smallest ceil(tiles / CUs) * (steps * step + ends).
// For example 512 x 4096 x 1024 (fp32): 256 tiles of 64 x 128 14.8 us, 128 of 128 x 128 18.9, 512 of
// 64 x 64 16.7; 1000 x 6144 x 1024: 256 of 128 x 192 32.0 us, 192 of 128 x 256 34.2, 96 of 256 x 256 42,
// 384 of 128 x 128 40; 512 x 6144 x 1024: 256 of 64 x 192 19.8 us, 192 of 128 x 128 21.5.
struct TileCost {
  int gm, gn;
  float step, ends;
};
constexpr int kTiles = 7;
constexpr TileCost kTileBf16[kTiles] = {
    {64, 64, .20f, 1.f}, {64, 128, .38f, 1.5f}, {128, 128, .65f, 2.f}, {256, 128, .98f, 3.f}, {256, 256, 1.7f, 5.f}, {0, 0, 0.f, 0.f}, {0, 0, 0.f, 0.f}};
constexpr TileCost kTileF32[kTiles] = {
    {64, 64, .50f, 1.f}, {64, 128, .71f, 1.5f}, {128, 128, 1.19f, 2.f}, {128, 256, 1.75f, 3.f}, {256, 256, 3.2f, 5.f},
    {64, 192, .95f, 2.f}, {128, 192, 1.6f, 2.5f}};  // (not whole head rows: no QKNR)
// The compute units a plan fills: the device's, or an undivided card's before kh_init (the split count may be
// asked for then).
inline int cus() { return cu_count() > 0 ? cu_count() : 256; }

inline float tile_cost(const TileCost& t, int64_t M, int64_t N, int64_t K, int splits) {
  const int64_t blocks = ((M + t.gm - 1) / t.gm) * ((N + t.gn - 1) / t.gn) * splits;
  const float steps = (float)((K + 63) / 64) / (float)splits;
  return (float)((blocks + cus() - 1) / cus()) * (steps * t.step + t.ends);
}
// The tile of a product split `splits` ways; its cost in *cost if given.  heads: tiles of whole head rows.
inline int choose_tile(bool f32, int M, int N, int K, int splits, bool heads = false, float* cost = nullptr) {
  const int first = heads ? 1 : 0, end = heads || !f32 ? 5 : kTiles;
  int best = first;
  float low = 0.f;
  for (int i = first; i < end; ++i) {
    const float c = tile_cost(f32 ? kTileF32[i] : kTileBf16[i], M, N, K, splits);
    if (i == first || c < low) {
      low = c;
      best = i;
    }
  }
  if (cost) *cost = low;
  return best;
}

// The skinny kernel's fp32 rows fit its LDS.
inline bool fits_skinny(int64_t M, int64_t K) { return M <= SK_MAXM && M * K * (int64_t)sizeof(float) <= 64 * 1024; }

// Two to SK_MAXM rows.  bf16 results come from the tiles, which read the weights once whatever the rows,
// where the skinny kernel re-reads its fp32 rows from LDS for every four weight rows: 5 x 1024 x 1024
// 17.9 -> 8.3 us, 2 x 6144 x 2560 28.5 -> 11.3, 8 x 151936 x 1024 541 -> 58; two short rows against few
// columns stay (2 x 4096 x 1024: 11.0 there, 12.3 on tiles).  fp32 results keep the
// skinny kernel's 64-way sums (error against 64 bits 7e-8 at K = 1024, the tiles' 8e-8) as long as its rows
// fit LDS; beyond, the generic kernel's one sum over K (1e-6 at K = 9728) was both slower and less
// exact: bf16 rows take the tiles there (8 x 2560 x 9728 1529 -> 13.9 us, error 1.3e-7), fp32 rows the
// one-row kernel row by row (1542 -> 141 us, 2.3e-7; its exact products, which the tiles' split of
// fp32 rows into two bf16 would not keep).
inline int tile_min_rows(int a_bytes, int out_bytes, int M, int N, int K) {
  const bool few_tiles = out_bytes == 2 && (M > 2 || K > 1024 || N > 4096);
  return a_bytes == 2 && (few_tiles || !fits_skinny(M, K)) ? 2 : SK_MAXM + 1;
}

// Launch plan of the MFMA tile kernel for a bf16 (or fp32) [M, K] x bf16 [N, K]^T product.
struct GemmPlan {
  bool mfma = false;  // the MFMA tile kernel applies (else the skinny or generic kernel)
  int tile = 0, splits = 1, kchunk = 0;
  bool parts = false;  // fp32 results of bf16 products are summed in PARTS
};

// The split that puts two 64 x 64 tiles on every CU (t64 of them unsplit, fewer than CUs); its k ranges.
inline int wide_splits(int64_t t64, int K, int* kchunk) {
  const int want = 2 * cus() / t64 > kMaxSplits ? kMaxSplits : (int)(2 * cus() / t64);
  *kchunk = ((K + want - 1) / want + 127) / 128 * 128;
  return (K + *kchunk - 1) / *kchunk;
}
// Long fp32 sums of bf16 products whose 64 x 64 tiles leave CUs idle, split in fewer ways than
// wide_splits, are taken in PARTS: the wider split can cost more than it gains (the partials' way through
// memory), but its shorter chains are worth keeping.
inline bool narrow_split(int64_t M, int64_t N, int K, int splits) {
  const int64_t t64 = ((M + 63) / 64) * ((N + 63) / 64);
  int kchunk;
  return K >= 1024 && N % 4 == 0 && t64 > 0 && t64 < cus() && splits < wide_splits(t64, K, &kchunk);
}

// aligned: both operands start on 16 bytes.  bf16: bf16 weights B with bf16 (a_bytes 2) or fp32
// (a_bytes 4, split into hi + lo) activations A.
GemmPlan gemm_plan(bool aligned, int64_t lda, int64_t ldb, int M, int N, int K, bool bf16, int trans_b,
                   int a_bytes, int min_rows) {
  GemmPlan p;
  const int64_t lim = int64_t(1) << 31;
  if (!(bf16 && trans_b && M >= min_rows && K % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && aligned &&
        128 * lda * a_bytes < lim && 128 * ldb * 2 < lim))
    return p;
  p.mfma = true;
  p.kchunk = K;
  // The K split: a split adds the partials' way through memory (0.35 us a MB) and about 1 us, and pays
  // where the tiles of whole sums leave CUs idle.  1000 x 1024 x 3072 fp32: 64 x 64 tiles unsplit 26.8 us,
  // 64 x 128 split in two 19.9; 512 x 1024 x 3072: 23.7 us unsplit, 13.3 split in four.  bf16 products
  // (half the work per step) take the same split while 64 x 64 tiles fill less than five eighths of the
  // CUs, none from there on: 1000 x 1024 x 2048 split in two 10.1 us and 4.7 for the sum, unsplit 9.5;
  // 1500 x 1024 x 3072 18.5 and 11.4 against 18.6; 2000 x 2560 x 9728 102 and 22 against 125.
  // From 6144 columns on five eighths to all of the CUs do better with two tiles each: 256 x 2560 x 9728 whole
  // 43.6 us, in three (64 x 128 tiles) 29.7; 800 x 1024 x 9728 (208 tiles) 42.6 and 38.1; 150 x 5120 x 17408 (240)
  // 73 and 63; 180 x 4096 x 6144 (192) 29.1 and 27.6; shorter sums go either way (256 x 2560 x 4096 20.8 and
  // 16.8, 800 x 1024 x 4096 14.6 and 17.1) and stay whole.
  // So do a few fp32 rows, which stream weights: 9 x 2560 x 4096 in six 12.4 us, in eight 11.3.
  // Sums shorter than 1024 are split only while the tiles are few for their length: 512 x 1024 x 640 (128
  // tiles) bf16 split in two 8.2 us, whole 4.9, fp32 10.4 and 8.1; 128 x 1024 x 640 (32) bf16 6.6 and 4.7, fp32
  // 7.5 and 7.7; 300 x 1024 x 1000 (80) fp32 10.2 and 10.9.  (fp32 results of bf16 products keep the short
  // chains: 512 x 512 x 512 is 1.2e-7 off 64 bits in one chain, 6.3e-8 in PARTS.)
  const int64_t t64 = (int64_t)((M + 63) / 64) * ((N + 63) / 64);
  const bool wide = a_bytes == 2 ? K >= 6144 && t64 >= cus() * 5 / 8 : K >= 2048 && M <= 32;
  if (wide && N % 4 == 0 && t64 > 0 && t64 < cus()) {
    p.splits = wide_splits(t64, K, &p.kchunk);
  } else if (K >= 512 && N % 4 == 0 && (a_bytes == 4 || t64 < cus() * 5 / 8)) {
    float low = 0.f;
    for (int sp = 1; sp <= kMaxSplits; ++sp) {
      const int kchunk = ((K + sp - 1) / sp + 127) / 128 * 128;
      if (sp > 1 && (K + kchunk - 1) / kchunk != sp) continue;
      float c;
      choose_tile(true, M, N, K, sp, false, &c);
      if (sp > 1) c += 1.f + 0.35e-6f * 4.f * (float)sp * (float)M * (float)N;
      if (sp == 1 || c < low) {
        low = c;
        p.splits = sp;
        p.kchunk = sp > 1 ? kchunk : K;
      }
    }
  }
  if (p.splits > 1 && K < 1024 && t64 * (a_bytes == 4 ? 12 : 20) >= K) {
    p.splits = 1;
    p.kchunk = K;
    p.parts = a_bytes == 2;
  } else {
    p.parts = a_bytes == 2 && narrow_split(M, N, K, p.splits);
  }
  p.tile = choose_tile(a_bytes == 4, M, N, K, p.splits);
  return p;
}

enum TileUse { USE_PLAIN, USE_SPLIT, USE_SWIGLU, USE_QKNR };

// One launch of the tile kernel: AM x AN blocks of 32 x 32 outputs per wave, WM x WN waves, NST stages
// of KS columns in LDS.
template <typename TO, typename TA, TileUse USE, bool PARTS, int AM, int AN, int WM, int WN, int KS, int NST>
int go_tile(const TA* A, int64_t lda, const uint16_t* B, int64_t ldb, TO* C, int64_t ldc, const TO* CI, int64_t ldcin,
            const TO* BI, int M, int N, int K, float alpha, float beta, int splits, int kchunk, float* part,
            const QknrArgs& qa) {
  using T = DmaTile<TA, AM, AN, WM, WN, KS>;
  const int64_t blocks = (int64_t)((M + T::GM - 1) / T::GM) * ((N + T::GN - 1) / T::GN) * splits;
  KH_REQUIRE(blocks <= INT32_MAX, "kh_gemm: grid too large");
  gemm_tile_kernel<TO, AM, AN, WM, WN, KS, NST, USE == USE_SPLIT, USE == USE_SWIGLU, USE == USE_QKNR, PARTS, TA>
      <<<(int)blocks, 64 * WM * WN, 0, stream()>>>(A, lda, B, ldb, C, ldc, CI, ldcin, BI, M, N, K, alpha, beta, splits,
                                                   kchunk, part, qa);
  KH_CHECK_LAUNCH();
  return KH_OK;
}

// The tile kernel with tile `tile` of kTileBf16 / kTileF32.  k-steps of 64 columns; of 32 where two or
// three stages of 64 do not fit the CU's 160 KiB of LDS.  64 x 128 fp32 tiles run four waves of 32 x 64
// (each A fragment split by two waves, not four: 16.6 -> 14.8 us at 512 x 4096 x 1024).
template <typename TO, typename TA, TileUse USE>
int launch_tile(int tile, const TA* A, int64_t lda, const uint16_t* B, int64_t ldb, TO* C, int64_t ldc, const TO* CI,
                int64_t ldcin, const TO* BI, int M, int N, int K, float alpha, float beta, int splits, int kchunk,
                float* part, const QknrArgs& qa = QknrArgs{}, bool parts = false) {
  constexpr bool AF = std::is_same<TA, float>::value;
  constexpr bool F32SUM = !AF && sizeof(TO) == 4 && (USE == USE_PLAIN || USE == USE_SPLIT);
  auto go = [&](auto am, auto an, auto wm, auto wn, auto ks, auto nst) {
    constexpr int AM = decltype(am)::value, AN = decltype(an)::value, WM = decltype(wm)::value, WN = decltype(wn)::value,
                  KS = decltype(ks)::value, NST = decltype(nst)::value;
    if constexpr (F32SUM && AM * AN <= 2)  // the tiles that a plan with parts takes
      if (parts)
        return go_tile<TO, TA, USE, true, AM, AN, WM, WN, KS, NST>(A, lda, B, ldb, C, ldc, CI, ldcin, BI, M, N, K,
                                                                   alpha, beta, splits, kchunk, part, qa);
    return go_tile<TO, TA, USE, false, AM, AN, WM, WN, KS, NST>(A, lda, B, ldb, C, ldc, CI, ldcin, BI, M, N, K, alpha,
                                                                beta, splits, kchunk, part, qa);
  };
  auto c = [](auto v) { return v; };
#define KH_I(v) c(std::integral_constant<int, (v)>{})
  if constexpr (USE != USE_QKNR)
    if (tile == 0) return go(KH_I(1), KH_I(1), KH_I(2), KH_I(2), KH_I(64), KH_I(AF ? 3 : 4));
  if (tile <= 1) {
    if constexpr (AF)
      return go(KH_I(1), KH_I(2), KH_I(2), KH_I(2), KH_I(64), KH_I(4));
    else
      return go(KH_I(1), KH_I(1), KH_I(2), KH_I(4), KH_I(64), KH_I(6));
  }
  if (tile == 2) return go(KH_I(1), KH_I(2), KH_I(4), KH_I(2), KH_I(64), KH_I(AF ? 3 : 4));
  if (tile == 3) {
    if constexpr (AF)
      return go(KH_I(1), KH_I(4), KH_I(4), KH_I(2), KH_I(32), KH_I(4));
    else
      return go(KH_I(2), KH_I(2), KH_I(4), KH_I(2), KH_I(64), KH_I(3));
  }
  if constexpr (AF && USE != USE_QKNR) {
    if (tile == 5) return go(KH_I(1), KH_I(3), KH_I(2), KH_I(2), KH_I(64), KH_I(3));
    if (tile == 6) return go(KH_I(1), KH_I(3), KH_I(4), KH_I(2), KH_I(64), KH_I(2));
  }
  return go(KH_I(2), KH_I(4), KH_I(4), KH_I(2), KH_I(32), KH_I(AF ? 3 : 4));
#undef KH_I
}

// A has element type TA, B has T (bf16 weights may meet fp32 activations: TA float, T uint16_t).
template <typename TA, typename T, typename TO>
int launch_gemm(const void* a, int64_t lda, const void* b, int64_t ldb, void* c, int64_t ldc, const void* cin,
                int64_t ldcin, const void* bias, int M, int N, int K, float alpha, float beta, int trans_b) {
  const TA* A = (const TA*)a;
  const T* B = (const T*)b;
  TO* C = (TO*)c;
  const TO* CI = (const TO*)cin;
  const TO* BI = (const TO*)bias;
  constexpr bool w_bf16 = sizeof(T) == 2;
  const bool skinny_fits = fits_skinny(M, K);
  const int min_rows = tile_min_rows((int)sizeof(TA), (int)sizeof(TO), M, N, K);
  const GemmPlan p =
      gemm_plan(aligned16(a) && aligned16(b), lda, ldb, M, N, K, w_bf16, trans_b, (int)sizeof(TA), min_rows);
  if constexpr (w_bf16) {
    if (p.mfma) {
      if (p.splits > 1) {
        float* part = (float*)scratch_alloc((size_t)p.splits * M * N * sizeof(float));
        if (part != nullptr) {
          const int rc = launch_tile<float, TA, USE_SPLIT>(p.tile, A, lda, (const uint16_t*)B, ldb, nullptr, 0, nullptr,
                                                           0, nullptr, M, N, K, alpha, beta, p.splits, p.kchunk, part,
                                                           QknrArgs{}, sizeof(TO) == 4 && p.parts);
          if (rc == KH_OK)
            gemm_splitk_reduce_kernel<TO><<<(int)(((int64_t)M * N / 4 + 255) / 256), 256, 0, stream()>>>(
                part, p.splits, C, ldc, CI, ldcin, BI, M, N, alpha, beta);
          scratch_free(part);  // stream-ordered reuse only
          if (rc != KH_OK) return rc;
          KH_CHECK_LAUNCH();
          return KH_OK;
        }
      }
      return launch_tile<TO, TA, USE_PLAIN>(choose_tile(sizeof(TA) == 4, M, N, K, 1), A, lda, (const uint16_t*)B, ldb, C,
                                            ldc, CI, ldcin, BI, M, N, K, alpha, beta, 1, K, nullptr, QknrArgs{},
                                            p.parts);
    }
    if (trans_b && M == 1) {
      constexpr bool EX = std::is_same<TA, float>::value;
      if (launch_gemv1<PRO_NONE, TO, EX>(a, nullptr, nullptr, 0.f, (const uint16_t*)B, ldb, C, CI, BI, N, K, alpha,
                                         beta)) {
        KH_CHECK_LAUNCH();
        return KH_OK;
      }
    }
    if constexpr (std::is_same<TA, float>::value) {
      if (trans_b && M > 1 && M <= SK_MAXM && !skinny_fits) {
        int m = 0;
        while (m < M && launch_gemv1<PRO_NONE, TO, true>(A + m * lda, nullptr, nullptr, 0.f, (const uint16_t*)B, ldb,
                                                         C + m * ldc, CI ? CI + m * ldcin : nullptr, BI, N, K, alpha, beta))
          ++m;
        KH_CHECK_LAUNCH();
        if (m == M) return KH_OK;
        KH_REQUIRE(m == 0, "kh_gemm: row %d of %d was refused", m, M);
      }
    }
  }
  if (trans_b && skinny_fits && aligned16(b)) {
    const int waves_needed = (N + SK_ROWS_PER_WAVE - 1) / SK_ROWS_PER_WAVE;
    int grid = (waves_needed + 3) / 4;
    if (grid > 4096) grid = 4096;
    const size_t shm = (size_t)M * K * sizeof(float);
    gemv_nt_kernel<TA, T, TO><<<grid, 256, shm, stream()>>>(A, lda, B, ldb, C, ldc, CI, ldcin, BI, M, N, K, alpha,
                                                            beta);
    KH_CHECK_LAUNCH();
    return KH_OK;
  }
  dim3 grid((N + 63) / 64, (M + 63) / 64);
  KH_REQUIRE(grid.y <= 65535, "kh_gemm: m too large for the generic kernel");
  gemm_generic_kernel<TA, T, TO><<<grid, 256, 0, stream()>>>(A, lda, B, ldb, C, ldc, CI, ldcin, BI, M, N, K, alpha,
                                                             beta, trans_b);
  KH_CHECK_LAUNCH();
  return KH_OK;
}

// The fused SwiGLU projection: the MFMA tile kernel with the SWIGLU epilogue, never split over K (the
// epilogue needs whole sums).  TA = TO: bf16, or fp32 activations in and out.
template <typename TA>
int launch_gemm_swiglu(const TA* X, int64_t ldx, const uint16_t* W, int64_t ldw, TA* H, int64_t ldh, int M, int N,
                       int K) {
  return launch_tile<TA, TA, USE_SWIGLU>(choose_tile(sizeof(TA) == 4, M, N, K, 1), X, ldx, W, ldw, H, ldh, nullptr, 0,
                                         nullptr, M, N, K, 1.f, 0.f, 1, K, nullptr);
}

// The fused QKV projection: tiles of whole head rows of 128, never split.
template <typename TA>
int launch_gemm_qk_norm_rope(const TA* X, int64_t ldx, const uint16_t* W, int64_t ldw, int M, int N, int K,
                             const QknrArgs& qa) {
  return launch_tile<TA, TA, USE_QKNR>(choose_tile(sizeof(TA) == 4, M, N, K, 1, true), X, ldx, W, ldw, (TA*)nullptr, 0,
                                       nullptr, 0, nullptr, M, N, K, 1.f, 0.f, 1, K, nullptr, qa);
}

}  // namespace

namespace kh {
// o_proj of the decode attention block: C = alpha * merge(part) W^T + beta * cin (fp32 out), with
// the split-K partials merged in every workgroup's prologue (exact: the merged row kept in fp32,
// else rounded to bf16 as the unfused path stores it).  False when the shapes do not fit.
bool launch_gemv_attn_merge(const float* part, const AttnMerge& am, const uint16_t* W, int64_t ldw, float* C,
                            const float* cin, int N, int K, float alpha, float beta, bool exact) {
  if (am.max_chunks > kAttnMergeMaxChunks || K != am.hq * 128) return false;
  if (exact)
    return launch_gemv1<PRO_ATTN_MERGE, float, true>(part, nullptr, nullptr, 0.f, W, ldw, C, cin, nullptr, N, K,
                                                     alpha, beta, am);
  return launch_gemv1<PRO_ATTN_MERGE, float>(part, nullptr, nullptr, 0.f, W, ldw, C, cin, nullptr, N, K, alpha, beta,
                                             am);
}
}  // namespace kh

extern "C" {

int kh_gemm_ex(const void* a, int64_t lda, int a_dtype, const void* b, int64_t ldb, int b_dtype, void* c,
               int64_t ldc, const void* cin, int64_t ldcin, const void* bias, int64_t m, int64_t n, int64_t k,
               float alpha, float beta, int trans_b, int out_dtype) {
  KH_REQUIRE_INIT();
  KH_REQUIRE(m >= 0 && n >= 0 && k >= 0, "kh_gemm: negative extent");
  KH_REQUIRE(m <= INT32_MAX && n <= INT32_MAX && k <= INT32_MAX, "kh_gemm: extent too large");
  KH_REQUIRE(a_dtype == KH_BF16 || a_dtype == KH_F32, "kh_gemm: unsupported dtype %d", a_dtype);
  KH_REQUIRE(b_dtype == KH_BF16 || b_dtype == KH_F32, "kh_gemm: unsupported dtype %d", b_dtype);
  KH_REQUIRE(!(a_dtype == KH_BF16 && b_dtype == KH_F32),
             "kh_gemm: a bfloat16 A with a float32 B is not supported (float32 A with bfloat16 B is)");
  KH_REQUIRE(out_dtype == KH_BF16 || out_dtype == KH_F32, "kh_gemm: unsupported output dtype %d", out_dtype);
  KH_REQUIRE(!(a_dtype == KH_F32 && out_dtype == KH_BF16),
             "kh_gemm: fp32 inputs with a bf16 output are not supported");
  if (m == 0 || n == 0) return KH_OK;
  KH_REQUIRE(a && b && c, "kh_gemm: null pointer");
  KH_REQUIRE(lda >= k && ldc >= n && (trans_b ? ldb >= k : ldb >= n), "kh_gemm: leading dimension too small");
  KH_REQUIRE(cin == nullptr || ldcin >= n, "kh_gemm: ldcin too small");
  const int M = (int)m, N = (int)n, K = (int)k;
  if (a_dtype == KH_BF16 && out_dtype == KH_BF16)
    return launch_gemm<uint16_t, uint16_t, uint16_t>(a, lda, b, ldb, c, ldc, cin, ldcin, bias, M, N, K, alpha, beta,
                                                     trans_b);
  if (a_dtype == KH_BF16)
    return launch_gemm<uint16_t, uint16_t, float>(a, lda, b, ldb, c, ldc, cin, ldcin, bias, M, N, K, alpha, beta,
                                                  trans_b);
  if (b_dtype == KH_BF16)
    return launch_gemm<float, uint16_t, float>(a, lda, b, ldb, c, ldc, cin, ldcin, bias, M, N, K, alpha, beta,
                                               trans_b);
  return launch_gemm<float, float, float>(a, lda, b, ldb, c, ldc, cin, ldcin, bias, M, N, K, alpha, beta, trans_b);
}

int kh_gemm(const void* a, int64_t lda, const void* b, int64_t ldb, void* c, int64_t ldc, const void* cin,
            int64_t ldcin, const void* bias, int64_t m, int64_t n, int64_t k, float alpha, float beta, int trans_b,
            int dtype, int out_dtype) {
  return kh_gemm_ex(a, lda, dtype, b, ldb, dtype, c, ldc, cin, ldcin, bias, m, n, k, alpha, beta, trans_b, out_dtype);
}

int kh_gemm_split_count(int64_t m, int64_t n, int64_t k, int* splits) {
  KH_REQUIRE(splits != nullptr, "kh_gemm_split_count: null pointer");
  KH_REQUIRE(m >= 0 && n >= 0 && k >= 0 && m <= INT32_MAX && n <= INT32_MAX && k <= INT32_MAX,
             "kh_gemm_split_count: bad extents");
  return kh_gemm_split_count_for(m, n, k, KH_BF16, splits);
}

int kh_gemm_split_count_for(int64_t m, int64_t n, int64_t k, int a_dtype, int* splits) {
  KH_REQUIRE(splits != nullptr, "kh_gemm_split_count_for: null pointer");
  KH_REQUIRE(m >= 0 && n >= 0 && k >= 0 && m <= INT32_MAX && n <= INT32_MAX && k <= INT32_MAX,
             "kh_gemm_split_count_for: bad extents");
  KH_REQUIRE(a_dtype == KH_BF16 || a_dtype == KH_F32, "kh_gemm_split_count_for: unsupported dtype %d", a_dtype);
  // bf16 weights, fp32 results, contiguous and 16-byte aligned operands
  const int ab = a_dtype == KH_F32 ? 4 : 2;
  const GemmPlan p = gemm_plan(true, k, k, (int)m, (int)n, (int)k, true, 1, ab,
                               tile_min_rows(ab, 4, (int)m, (int)n, (int)k));
  *splits = p.mfma ? p.splits : 1;
  return KH_OK;
}

int kh_gemm_splitk_partials(const void* a, int64_t lda, const void* b, int64_t ldb, float* part, int64_t m,
                            int64_t n, int64_t k, int splits, int a_dtype) {
  KH_REQUIRE_INIT();
  KH_REQUIRE(m > 0 && n > 0 && k > 0 && m <= INT32_MAX && n <= INT32_MAX && k <= INT32_MAX,
             "kh_gemm_splitk_partials: bad extents");
  KH_REQUIRE(a && b && part, "kh_gemm_splitk_partials: null pointer");
  KH_REQUIRE(lda >= k && ldb >= k, "kh_gemm_splitk_partials: leading dimension too small");
  KH_REQUIRE(a_dtype == KH_BF16 || a_dtype == KH_F32, "kh_gemm_splitk_partials: unsupported dtype %d", a_dtype);
  const int ab = a_dtype == KH_F32 ? 4 : 2;
  GemmPlan p = gemm_plan(aligned16(a) && aligned16(b), lda, ldb, (int)m, (int)n, (int)k, true, 1, ab,
                         tile_min_rows(ab, 4, (int)m, (int)n, (int)k));
  int other = 1;  // the other type's count is taken too: a caller may have asked for it without a type
  if (kh_gemm_split_count_for(m, n, k, ab == 4 ? KH_BF16 : KH_F32, &other) != KH_OK) return KH_ERR_INVALID;
  if (splits > 1 && splits == other && splits != p.splits) {
    p.splits = splits;
    p.kchunk = (((int)k + splits - 1) / splits + 127) / 128 * 128;
    p.tile = choose_tile(ab == 4, (int)m, (int)n, (int)k, splits);
    p.parts = ab == 2 && narrow_split(m, n, (int)k, splits);
  }
  KH_REQUIRE(p.mfma && p.splits > 1 && p.splits == splits,
             "kh_gemm_splitk_partials: this product is not split %d ways (kh_gemm_split_count_for gives the count; "
             "operands must be 16-byte aligned with k and the leading dimensions multiples of 8)", splits);
  if (a_dtype == KH_F32)
    return launch_tile<float, float, USE_SPLIT>(p.tile, (const float*)a, lda, (const uint16_t*)b, ldb, nullptr, 0,
                                                nullptr, 0, nullptr, (int)m, (int)n, (int)k, 1.f, 0.f, p.splits, p.kchunk,
                                                part);
  return launch_tile<float, uint16_t, USE_SPLIT>(p.tile, (const uint16_t*)a, lda, (const uint16_t*)b, ldb, nullptr, 0,
                                                 nullptr, 0, nullptr, (int)m, (int)n, (int)k, 1.f, 0.f, p.splits,
                                                 p.kchunk, part, QknrArgs{}, p.parts);
}

int kh_gemm_swiglu(const void* x, int64_t ldx, const void* w_gu, int64_t ldw, void* h, int64_t ldh, int64_t m,
                   int64_t n_half, int64_t k, int x_dtype) {
  KH_REQUIRE_INIT();
  KH_REQUIRE(m >= 0 && n_half >= 0 && k > 0 && m <= INT32_MAX && 2 * n_half <= INT32_MAX && k <= INT32_MAX,
             "kh_gemm_swiglu: bad extents");
  KH_REQUIRE(x_dtype == KH_BF16 || x_dtype == KH_F32, "kh_gemm_swiglu: unsupported dtype %d", x_dtype);
  if (m == 0 || n_half == 0) return KH_OK;
  KH_REQUIRE(x && w_gu && h, "kh_gemm_swiglu: null pointer");
  KH_REQUIRE(n_half % 8 == 0, "kh_gemm_swiglu: the intermediate size %lld is not a multiple of 8", (long long)n_half);
  KH_REQUIRE(k % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && ldx >= k && ldw >= k && ldh >= n_half,
             "kh_gemm_swiglu: k and the row strides must be multiples of 8 elements (ldx, ldw >= k, ldh >= n_half)");
  KH_REQUIRE(aligned16(x) && aligned16(w_gu), "kh_gemm_swiglu: x and w_gu must be 16-byte aligned");
  const int64_t lim = int64_t(1) << 31;
  const int xb = x_dtype == KH_F32 ? 4 : 2;
  KH_REQUIRE(128 * ldx * xb < lim && 128 * ldw * 2 < lim,
             "kh_gemm_swiglu: row stride too large");
  if (x_dtype == KH_F32)
    return launch_gemm_swiglu<float>((const float*)x, ldx, (const uint16_t*)w_gu, ldw, (float*)h, ldh, (int)m,
                                     (int)(2 * n_half), (int)k);
  return launch_gemm_swiglu<uint16_t>((const uint16_t*)x, ldx, (const uint16_t*)w_gu, ldw, (uint16_t*)h, ldh, (int)m,
                                      (int)(2 * n_half), (int)k);
}

// cos / sin of float(positions[t]) * inv_freq[i] for n tokens and `half` frequencies, interleaved
// (cos, sin) per (t, i): the angles of every qk-norm + RoPE head tile of a prefill, evaluated once.
__global__ __launch_bounds__(256) void rope_table_kernel(const int32_t* __restrict__ positions, int64_t n,
                                                         const float* __restrict__ inv_freq, int half,
                                                         float* __restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n * half; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = i / half;
    const float pos = (float)positions[t];
    float sn, cs;
    sincosf(pos * inv_freq[i - t * half], &sn, &cs);
    out[2 * i] = cs;
    out[2 * i + 1] = sn;
  }
}

int kh_rope_table(const int32_t* positions, int64_t n, const float* inv_freq, int half, float* out) {
  KH_REQUIRE_INIT();
  KH_REQUIRE(n >= 0 && half > 0 && half <= 4096, "kh_rope_table: bad extents");
  if (n == 0) return KH_OK;
  KH_REQUIRE(positions && inv_freq && out, "kh_rope_table: null pointer");
  const int64_t total = n * half;
  const int64_t want = (total + 255) / 256;
  const int grid = (int)(want < 4096 ? want : 4096);
  rope_table_kernel<<<grid, 256, 0, stream()>>>(positions, n, inv_freq, half, out);
  KH_CHECK_LAUNCH();
  return KH_OK;
}

int kh_gemm_qk_norm_rope(const void* x, int64_t ldx, const void* w_qkv, int64_t ldw, int64_t n_batch,
                         int64_t seq_len, int64_t k, int n_q_heads, int n_kv_heads, int head_dim, const void* wq,
                         const void* wk, const float* inv_freq, const int32_t* positions, void* q_out, void* k_out,
                         void* v_out, const int64_t* strides, float eps, int64_t kv_cache_len, int dtype) {
  return kh_gemm_qk_norm_rope_table(x, ldx, w_qkv, ldw, n_batch, seq_len, k, n_q_heads, n_kv_heads, head_dim, wq, wk,
                                    inv_freq, positions, q_out, k_out, v_out, strides, eps, kv_cache_len, dtype,
                                    nullptr);
}

int kh_gemm_qk_norm_rope_table(const void* x, int64_t ldx, const void* w_qkv, int64_t ldw, int64_t n_batch,
                               int64_t seq_len, int64_t k, int n_q_heads, int n_kv_heads, int head_dim, const void* wq,
                               const void* wk, const float* inv_freq, const int32_t* positions, void* q_out,
                               void* k_out, void* v_out, const int64_t* strides, float eps, int64_t kv_cache_len,
                               int dtype, const float* rope_table) {
  KH_REQUIRE_INIT();
  KH_REQUIRE(n_batch >= 0 && seq_len >= 0 && k > 0 && k <= INT32_MAX && kv_cache_len >= 0,
             "kh_gemm_qk_norm_rope: bad extents");
  KH_REQUIRE(head_dim == 128, "kh_gemm_qk_norm_rope: head_dim %d (the fused projection takes 128)", head_dim);
  KH_REQUIRE(n_q_heads > 0 && n_kv_heads > 0, "kh_gemm_qk_norm_rope: head counts must be positive");
  KH_REQUIRE(dtype == KH_BF16 || dtype == KH_F32, "kh_gemm_qk_norm_rope: unsupported dtype %d", dtype);
  const int64_t M = n_batch * seq_len, N = (int64_t)(n_q_heads + 2 * n_kv_heads) * 128;
  KH_REQUIRE(M <= INT32_MAX && N <= INT32_MAX && seq_len <= (int64_t)UINT32_MAX, "kh_gemm_qk_norm_rope: too large");
  if (M == 0) return KH_OK;
  KH_REQUIRE(x && w_qkv && wq && wk && inv_freq && positions && q_out && k_out && v_out && strides,
             "kh_gemm_qk_norm_rope: null pointer");
  KH_REQUIRE(k % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && ldx >= k && ldw >= k,
             "kh_gemm_qk_norm_rope: k and the row strides must be multiples of 8 elements (ldx, ldw >= k)");
  const void* al[] = {x, w_qkv, wq, wk, q_out, k_out, v_out};
  for (const void* p : al) KH_REQUIRE(aligned16(p), "kh_gemm_qk_norm_rope: operands must be 16-byte aligned");
  const int64_t lim = int64_t(1) << 31;
  const int xb = dtype == KH_F32 ? 4 : 2;
  KH_REQUIRE(128 * ldx * xb < lim && 128 * ldw * 2 < lim,
             "kh_gemm_qk_norm_rope: row stride too large");
  QknrArgs qa;
  const int64_t vec = 16 / xb;
  for (int i = 0; i < 9; ++i) {
    KH_REQUIRE(strides[i] % vec == 0, "kh_gemm_qk_norm_rope: stride %d (%lld) breaks 16-byte alignment", i,
               (long long)strides[i]);
    qa.s[i] = strides[i];
  }
  qa.wq = (const uint16_t*)wq;
  qa.wk = (const uint16_t*)wk;
  qa.inv_freq = inv_freq;
  qa.positions = positions;
  qa.q_out = q_out;
  qa.k_out = k_out;
  qa.v_out = v_out;
  qa.hq = n_q_heads;
  qa.hkv = n_kv_heads;
  qa.seq_len = (uint32_t)(seq_len > 0 ? seq_len : 1);
  qa.eps = eps;
  qa.kv_cache_len = kv_cache_len;
  KH_REQUIRE(rope_table == nullptr || aligned16(rope_table), "kh_gemm_qk_norm_rope: rope_table must be 16-byte aligned");
  qa.rope_cs = rope_table;
  if (dtype == KH_F32)
    return launch_gemm_qk_norm_rope<float>((const float*)x, ldx, (const uint16_t*)w_qkv, ldw, (int)M, (int)N, (int)k,
                                           qa);
  return launch_gemm_qk_norm_rope<uint16_t>((const uint16_t*)x, ldx, (const uint16_t*)w_qkv, ldw, (int)M, (int)N,
                                            (int)k, qa);
}

int kh_gemv_swiglu(int prologue, const void* x, const void* norm_w, float eps, const void* w_gu, int64_t ldw,
                   void* h, int64_t n_half, int64_t k, int x_dtype) {
  KH_REQUIRE_INIT();
  KH_REQUIRE(prologue == PRO_NONE || prologue == PRO_RMSNORM, "kh_gemv_swiglu: prologue must be 0 (none) or 1 (RMSNorm)");
  KH_REQUIRE(x_dtype == KH_BF16 || x_dtype == KH_F32, "kh_gemv_swiglu: unsupported dtype %d", x_dtype);
  KH_REQUIRE(n_half > 0 && k > 0 && 2 * n_half <= INT32_MAX && k <= INT32_MAX, "kh_gemv_swiglu: bad extents");
  KH_REQUIRE(n_half % 8 == 0, "kh_gemv_swiglu: the intermediate size %lld is not a multiple of 8", (long long)n_half);
  KH_REQUIRE(x && w_gu && h, "kh_gemv_swiglu: null pointer");
  KH_REQUIRE(prologue != PRO_RMSNORM || norm_w != nullptr, "kh_gemv_swiglu: the RMSNorm prologue needs norm_w");
  KH_REQUIRE(ldw >= k, "kh_gemv_swiglu: ldw < k");
  const uint16_t* W = (const uint16_t*)w_gu;
  const int NH = (int)n_half, K = (int)k;
  bool ok;
  if (x_dtype == KH_F32)
    ok = prologue == PRO_RMSNORM ? launch_gemv_swiglu<PRO_RMSNORM, true, float>(x, norm_w, eps, W, ldw, (float*)h, NH, K)
                                 : launch_gemv_swiglu<PRO_NONE, true, float>(x, norm_w, eps, W, ldw, (float*)h, NH, K);
  else
    ok = prologue == PRO_RMSNORM ? launch_gemv_swiglu<PRO_RMSNORM>(x, norm_w, eps, W, ldw, (uint16_t*)h, NH, K)
                                 : launch_gemv_swiglu<PRO_NONE>(x, norm_w, eps, W, ldw, (uint16_t*)h, NH, K);
  KH_REQUIRE(ok, "kh_gemv_swiglu: unsupported operands (need k %% 8 == 0, ldw %% 8 == 0, a 16-byte aligned weight, "
                 "k <= 32768 and byte offsets below 4 GiB)");
  KH_CHECK_LAUNCH();
  return KH_OK;
}

int kh_gemv_fused(int prologue, const void* x, const void* x2, const void* norm_w, float eps, const void* w,
                  int64_t ldw, void* c, const void* cin, const void* bias, int64_t n, int64_t k, float alpha,
                  float beta, int out_dtype, int x_dtype) {
  KH_REQUIRE_INIT();
  KH_REQUIRE(prologue >= PRO_NONE && prologue <= PRO_SILU_MUL_IL, "kh_gemv_fused: unknown prologue %d", prologue);
  KH_REQUIRE(prologue != PRO_SILU_MUL_IL || k % 8 == 0, "kh_gemv_fused: the interleaved silu*mul prologue needs k %% 8 == 0");
  KH_REQUIRE(n >= 0 && k > 0 && n <= INT32_MAX && k <= INT32_MAX, "kh_gemv_fused: bad extents");
  KH_REQUIRE(out_dtype == KH_BF16 || out_dtype == KH_F32, "kh_gemv_fused: unsupported output dtype %d", out_dtype);
  KH_REQUIRE(x_dtype == KH_BF16 || x_dtype == KH_F32, "kh_gemv_fused: unsupported activation dtype %d", x_dtype);
  if (n == 0) return KH_OK;
  KH_REQUIRE(x && w && c, "kh_gemv_fused: null pointer");
  KH_REQUIRE(prologue != PRO_RMSNORM || norm_w != nullptr, "kh_gemv_fused: the RMSNorm prologue needs norm_w");
  KH_REQUIRE(prologue != PRO_SILU_MUL || x2 != nullptr, "kh_gemv_fused: the silu*mul prologue needs x2");
  KH_REQUIRE(ldw >= k, "kh_gemv_fused: ldw < k");
  const int N = (int)n, K = (int)k;
  const uint16_t* W = (const uint16_t*)w;
  bool ok = false;
  auto run = [&](auto* C, auto* CI, auto* BI, auto ex) {
    using TO = std::remove_const_t<std::remove_pointer_t<decltype(CI)>>;
    constexpr bool EX = decltype(ex)::value;
    if (prologue == PRO_RMSNORM)
      ok = launch_gemv1<PRO_RMSNORM, TO, EX>(x, x2, norm_w, eps, W, ldw, C, CI, BI, N, K, alpha, beta);
    else if (prologue == PRO_SILU_MUL)
      ok = launch_gemv1<PRO_SILU_MUL, TO, EX>(x, x2, norm_w, eps, W, ldw, C, CI, BI, N, K, alpha, beta);
    else if (prologue == PRO_SILU_MUL_IL)
      ok = launch_gemv1<PRO_SILU_MUL_IL, TO, EX>(x, x2, norm_w, eps, W, ldw, C, CI, BI, N, K, alpha, beta);
    else
      ok = launch_gemv1<PRO_NONE, TO, EX>(x, x2, norm_w, eps, W, ldw, C, CI, BI, N, K, alpha, beta);
  };
  const bool exact = x_dtype == KH_F32;
  if (out_dtype == KH_F32 && exact)
    run((float*)c, (const float*)cin, (const float*)bias, std::true_type{});
  else if (out_dtype == KH_F32)
    run((float*)c, (const float*)cin, (const float*)bias, std::false_type{});
  else if (exact)
    run((uint16_t*)c, (const uint16_t*)cin, (const uint16_t*)bias, std::true_type{});
  else
    run((uint16_t*)c, (const uint16_t*)cin, (const uint16_t*)bias, std::false_type{});
  KH_REQUIRE(ok, "kh_gemv_fused: unsupported operands (need k %% 8 == 0, ldw %% 8 == 0, a 16-byte aligned weight, "
                 "k <= 32768 and byte offsets below 4 GiB)");
  KH_CHECK_LAUNCH();
  return KH_OK;
}

}  // extern "C"
