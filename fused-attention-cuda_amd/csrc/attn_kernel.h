// attn_kernel.h -- the fp32-compute correctness rung of the fused SDPA forward (stage 3).
//
// Included by attn_f32.hip, which instantiates it for fp16 inputs, and by attn_split32.h, whose fp32
// kernel falls back to it (Attn<float, ...>) on magnitudes that it does not split:
//   fa_s3_fused<T>   (stage 3)  operands are held in LDS as fp32 and multiplied on
//                               v_mfma_f32_32x32x2_f32, so no operand is rounded below fp32
//                               (fp32 or fp16 I/O, ref:src/stage3_fused.cu:142-160). K/V tiles are
//                               double-buffered in LDS with register-staged prefetch.
// The 16-bit matrix-core stages (4 and 5) live in attn_mfma16.h.
//
// Algorithm (FlashAttention-2 loop order, the reference's recurrence ref:include/fa/softmax_math.cuh):
// a workgroup owns BR = 32*WAVES query rows of one (b, h); each wave owns 32 rows for the whole
// kernel; K/V tiles of BC keys stream through LDS; per tile a wave computes S^T = K Q^T on MFMA,
// masks (causal diagonal block only), updates the running max m (raw score units), rescales
// (alpha = exp2((m_old - m_new) c), c = scale*log2 e), exponentiates p = exp2(s c - m c), sums l,
// and accumulates O^T += V^T P^T on MFMA. Epilogue: O = acc / l, lse = m*scale + ln l. Causal key
// tiles beyond the workgroup's last row are never loaded; per wave, key blocks beyond the wave's
// last row are skipped and only the diagonal 32x32 block is masked.
//
// WHY S^T = K Q^T (not S = Q K^T): the 32x32 MFMA accumulator gives lane l the column n = l % 32
// and 16 rows m = 8(r/4) + 4(l/32) + r%4 (r = register). With M = keys and N = query rows, every
// lane owns ONE query row and 16 of its keys, so (a) the row max/sum needs a single cross-lane
// step (lane l with l ^ 32), (b) alpha is one scalar per lane, and (c) the probabilities are
// already in the B-operand layout of the second product O^T = V^T P^T (lane l supplies column
// n = l % 32 = its row; its 8 k-slots are 8 of its own keys). P never leaves registers -- the
// smem round trips the reference's WMMA kernels need (ref:src/stage5_tuned.cu:63-76) do not exist.
// The price is that V must be read "transposed" (keys of one head-dim column per lane): V^T is
// therefore what the tile loader writes to LDS, so every PV operand is one 16-byte LDS read.
//
// LDS layout (per buffer): Ks[BC][D + pad] row-major (A operand of S^T: lane reads 16 contiguous
// bytes of key row l % 32), then Vt[D][BC + pad]. pad = 16 bytes: rows shift by 4 banks, so the
// 32 lanes reading 32 different rows at the same column hit distinct banks (16 lanes x 16 B per
// LDS cycle).
//
// Work distribution: grid = (N / BR) * B * H workgroups on a 1-D grid, mapped by layout::grid_item as
// in the 16-bit kernels. Hardware hands workgroup i to XCD (i + c) % 8, c fixed for the launch (8
// XCDs, each with its own L2), so the workgroups of one residue i % 8 take a contiguous range of
// (head, q-tile) pairs and a head's K/V is fetched into one L2. Causal grids issue the longest walks
// first, of all heads of an XCD where it has whole ones: measured on MI355X, fp16, against head by
// head, B8 H12 N1024 D64 209.5 -> 145.6 us, B16 H32 Hkv8 N512 D64 273 -> 172, B1 H16 N4096 D128 1082
// -> 791. On other grids the order is the same as head by head (B2 H8 N2048 D64 162.9 and 163.6, B7
// H7 N992 142.1 and 144.6).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <type_traits>

#include "fa_internal.h"
#include "tile_layout.h"
#include "wave_halves.h"

namespace fa {
namespace kern {

using ::fa::KArgs;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kLn2 = 0.69314718055994531f;
// Lazy rescaling threshold, in exp2 units: probabilities may reach 2^8 before m is moved.
constexpr float kLazyLog2 = 8.0f;

// 2^x on the transcendental unit (v_exp_f32). exp2(-inf) = 0, which the masking relies on.
__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }
// log2(x) on the transcendental unit (v_log_f32).
__device__ __forceinline__ float log2_hw(float x) { return __builtin_amdgcn_logf(x); }

// 32x32x2 MFMA on fp32 operands (one element per lane in a/b).
__device__ __forceinline__ f32x16 mma32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// The work item of this workgroup (layout::grid_item): its head and query tile.
struct Where {
  int b, h, hk, qt;
};
__device__ __forceinline__ Where where(const KArgs& a) {
  auto div = [](int n, const FastDiv& f) {
    return f.d == 1 ? n
                    : __builtin_amdgcn_readfirstlane(static_cast<int>(
                          __umulhi(static_cast<uint32_t>(n), f.m) >> f.s));
  };
  const layout::Item it = layout::grid_item(
      static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x), a.n_qtiles, 1, a.causal != 0,
      a.xcd_heads, 0, [](int x) { return x; }, [&](int x) { return div(x, a.fd_qtiles); },
      [&](int x) { return div(x, a.fd_xcd_heads); }, [](int x) { return x; });
  const int b = div(it.bh, a.fd_h);
  const int h = it.bh - b * a.H;
  return Where{b, h, div(h, a.fd_group), it.qt};
}
// Host side of where(): the grid's divisors, once n_qtiles is set.
inline void fill_grid(KArgs& a) {
  a.fd_qtiles = make_fastdiv(static_cast<uint32_t>(a.n_qtiles));
  a.xcd_heads = layout::xcd_heads_for(a.B * a.H, a.causal != 0);
  a.fd_xcd_heads = make_fastdiv(static_cast<uint32_t>(a.xcd_heads > 0 ? a.xcd_heads : 1));
}

// Tio: element type in HBM (q/k/v/o: fp32 or fp16); LDS and the MFMA operands are fp32 (Tc).
// WAVES: 32-row query groups per workgroup (BR = 32*WAVES). BC: keys per K/V tile. PREFETCH:
// double-buffered LDS + register-staged next-tile loads. THREADS: the workgroup's threads; waves
// past the first WAVES own no rows and only help to stage the tiles.
template <typename Tio, int D_, int WAVES, int BC_, bool PREFETCH, int THREADS = 64 * WAVES>
struct Attn {
  using Tc = float;
  static constexpr int D = D_;
  static constexpr int BC = BC_;
  static constexpr int kThreads = THREADS;
  static constexpr int kBr = 32 * WAVES;
  static constexpr int kPad = 16 / static_cast<int>(sizeof(Tc));
  static constexpr int kLdK = D + kPad;  // Ks row stride (elements)
  static constexpr int kLdV = BC + kPad;  // Vt row stride (elements)
  static constexpr int kKElems = BC * kLdK;
  static constexpr int kBufElems = kKElems + D * kLdV;
  static constexpr int kBufs = PREFETCH ? 2 : 1;
  static constexpr int kLdsElems = kBufs * kBufElems;
  static constexpr size_t kLdsBytes = static_cast<size_t>(kLdsElems) * sizeof(Tc);
  static constexpr int kKB = BC / 32;  // 32-key blocks per tile
  static constexpr int kDB = D / 32;   // 32-wide head-dim blocks of O^T
  // Global -> register staging: 16-byte vectors of Tio.
  static constexpr int kVec = 16 / static_cast<int>(sizeof(Tio));
  static constexpr int kRowVecs = D / kVec;                 // 16-byte vectors per K/V row
  static constexpr int kKChunks = BC * kRowVecs;             // one vector per chunk
  static constexpr int kVChunks = (BC / 4) * kRowVecs;       // 4 keys x one vector per chunk
  static constexpr int kNK = (kKChunks + kThreads - 1) / kThreads;
  static constexpr int kNV = (kVChunks + kThreads - 1) / kThreads;
  // Per-lane Q operand storage: D/2 floats as D/8 vectors of 4.
  static constexpr int kQVecs = D / 8;

  static_assert(BC % 32 == 0 && BC >= 32 && BC <= 128, "BC must be 32, 64 or 128");
  static_assert(D == 64 || D == 128, "D must be 64 or 128");
  static_assert(WAVES >= 1 && WAVES <= 8, "1..8 waves");
  static_assert(kLdsBytes <= 160 * 1024, "gfx950 LDS is 160 KiB per workgroup");
  static_assert(__is_same(Tio, float) || __is_same(Tio, _Float16), "fp32 or fp16 I/O");

  struct Staging {
    u32x4 kv[kNK];
    u32x4 vv[kNV][4];
  };

  // Issue the global loads of K/V tile starting at key k0 into registers. Rows of keys >= N
  // (only in a partial last tile) are never read back from LDS -- their whole 32-key blocks are
  // skipped by the math -- so instead of zero-filling, the row index is clamped to N-1: every
  // address stays inside the tensor and the loads need no per-lane branch.
  __device__ static void load_tile(Staging& st, const Tio* kb, const Tio* vb, int k0, int N,
                                   int ksn, int vsn, int tid) {
    const Tio* kt = kb + static_cast<ptrdiff_t>(k0) * ksn;
    const Tio* vt = vb + static_cast<ptrdiff_t>(k0) * vsn;
    const int last = N - 1 - k0;  // last valid tile-local key row (>= BC - 1 for a full tile)
#pragma unroll
    for (int i = 0; i < kNK; ++i) {
      const int c = tid + i * kThreads;
      if ((kKChunks % kThreads == 0) || c < kKChunks) {
        const int row = min(c / kRowVecs, last);
        st.kv[i] = *reinterpret_cast<const u32x4*>(kt + row * ksn + (c % kRowVecs) * kVec);
      }
    }
#pragma unroll
    for (int i = 0; i < kNV; ++i) {
      const int c = tid + i * kThreads;
      if ((kVChunks % kThreads == 0) || c < kVChunks) {
        const int row = 4 * (c / kRowVecs);
        const Tio* src = vt + (c % kRowVecs) * kVec;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          st.vv[i][j] = *reinterpret_cast<const u32x4*>(src + min(row + j, last) * vsn);
        }
      }
    }
  }

  // Write the staged tile into one LDS buffer: K row-major, V transposed (see header).
  __device__ static void store_tile(const Staging& st, Tc* buf, int tid) {
    Tc* Ks = buf;
    Tc* Vt = buf + kKElems;
#pragma unroll
    for (int i = 0; i < kNK; ++i) {
      const int c = tid + i * kThreads;
      if ((kKChunks % kThreads == 0) || c < kKChunks) {
        const int key = c / kRowVecs;
        const int col = (c % kRowVecs) * kVec;
        Tc* dst = Ks + key * kLdK + col;
        if constexpr (__is_same(Tio, Tc)) {
          *reinterpret_cast<u32x4*>(dst) = st.kv[i];
        } else {  // fp16 in HBM, fp32 in LDS: 8 values -> two 16-byte writes
          const f16x8 h = __builtin_bit_cast(f16x8, st.kv[i]);
          *reinterpret_cast<f32x4*>(dst) = f32x4{(float)h[0], (float)h[1], (float)h[2], (float)h[3]};
          *reinterpret_cast<f32x4*>(dst + 4) =
              f32x4{(float)h[4], (float)h[5], (float)h[6], (float)h[7]};
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kNV; ++i) {
      const int c = tid + i * kThreads;
      if ((kVChunks % kThreads == 0) || c < kVChunks) {
        const int key0 = 4 * (c / kRowVecs);  // first of the 4 keys (tile-local)
        const int d0 = (c % kRowVecs) * kVec;
        if constexpr (__is_same(Tio, float)) {
          // 4 keys x 4 head-dim fp32 values -> 4 rows of V^T (natural key order), 16 bytes each.
          const f32x4 r0 = __builtin_bit_cast(f32x4, st.vv[i][0]);
          const f32x4 r1 = __builtin_bit_cast(f32x4, st.vv[i][1]);
          const f32x4 r2 = __builtin_bit_cast(f32x4, st.vv[i][2]);
          const f32x4 r3 = __builtin_bit_cast(f32x4, st.vv[i][3]);
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            *reinterpret_cast<f32x4*>(Vt + (d0 + d) * kLdV + key0) =
                f32x4{r0[d], r1[d], r2[d], r3[d]};
          }
        } else {
          // fp16 in HBM, fp32 in LDS: 4 keys x 8 head-dim values -> 8 rows of V^T.
          const f16x8 h0 = __builtin_bit_cast(f16x8, st.vv[i][0]);
          const f16x8 h1 = __builtin_bit_cast(f16x8, st.vv[i][1]);
          const f16x8 h2 = __builtin_bit_cast(f16x8, st.vv[i][2]);
          const f16x8 h3 = __builtin_bit_cast(f16x8, st.vv[i][3]);
#pragma unroll
          for (int d = 0; d < 8; ++d) {
            *reinterpret_cast<f32x4*>(Vt + (d0 + d) * kLdV + key0) =
                f32x4{(float)h0[d], (float)h1[d], (float)h2[d], (float)h3[d]};
          }
        }
      }
    }
  }

  // Per-wave running state: Q operand, O^T accumulator, row max (raw units) and partial row sum
  // (this lane's half of the row's keys; the two halves are added in the epilogue).
  struct WaveState {
    f32x4 qf[kQVecs];
    f32x16 o[kDB];
    float m;   // running row max, raw score units (may lag the true max: lazy rescaling)
    float mc;  // m * c with the -inf guard applied (0 while m == -inf)
    float l;   // this lane's partial row sum, relative to m
  };

  __device__ static void load_q(WaveState& ws, const Tio* qb, int row, int qsn, bool valid, int g) {
    // fp32 MFMA k-slot mapping: lane half g covers head-dim [g*D/2, (g+1)*D/2).
    const Tio* src = qb + row * qsn + g * (D / 2);
#pragma unroll
    for (int j = 0; j < kQVecs; ++j) {
      if (!valid) {
        ws.qf[j] = f32x4{0.f, 0.f, 0.f, 0.f};
      } else if constexpr (__is_same(Tio, float)) {
        ws.qf[j] = *reinterpret_cast<const f32x4*>(src + 4 * j);
      } else {
        const f16x4 h = *reinterpret_cast<const f16x4*>(src + 4 * j);
        ws.qf[j] = f32x4{(float)h[0], (float)h[1], (float)h[2], (float)h[3]};
      }
    }
  }

  // One K/V tile for one wave: nvalid leading 32-key blocks take part; `diag` is the index of
  // the block on the causal diagonal (-1 if none).
  __device__ static void compute_tile(WaveState& ws, const Tc* buf, int nvalid, int diag, float c,
                                      float lazy_raw, int lane) {
    const Tc* Ks = buf;
    const Tc* Vt = buf + kKElems;
    const int g = lane >> 5;
    const int r32 = lane & 31;
    f32x16 s[kKB];
    // ---- S^T = K Q^T ---------------------------------------------------------------------------
#pragma unroll
    for (int kb = 0; kb < kKB; ++kb) {
      if (kb < nvalid) {
        f32x16 acc = {};
        const Tc* krow = Ks + (32 * kb + r32) * kLdK;
#pragma unroll
        for (int j = 0; j < kQVecs; ++j) {
          const f32x4 a = *reinterpret_cast<const f32x4*>(krow + g * (D / 2) + 4 * j);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc = mma32(a[e], ws.qf[j][e], acc);
        }
        s[kb] = acc;
      }
    }
    // ---- causal diagonal block: key (8(r/4) + 4g + r%4) > row (r32) is masked ---------------
    if (diag >= 0) {
#pragma unroll
      for (int kb = 0; kb < kKB; ++kb) {
        if (kb == diag) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = 8 * (r >> 2) + 4 * g + (r & 3);
            if (key > r32) s[kb][r] = -__builtin_inff();
          }
        }
      }
    }
    // ---- online softmax with lazy rescaling (ref:include/fa/softmax_math.cuh:25-71) --------
    // Row max of this tile: the lane's 16*nvalid scores, then the partner lane (l ^ 32), which
    // holds the row's other keys.
    float mx = -__builtin_inff();
#pragma unroll
    for (int kb = 0; kb < kKB; ++kb) {
      if (kb < nvalid) {
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kb][r]);
      }
    }
    mx = halves_max(mx);
    // The reference recurrence moves m to the row max on every tile and rescales acc and l by
    // alpha = exp2((m_old - m_new) c). Here m moves only when some row of the wave sees a max
    // more than kLazyLog2 (exp2 units) above its current m; otherwise p = exp2(s c - m c)
    // stays <= 2^kLazyLog2 and nothing is rescaled. acc, l and lse are all taken relative to the same m,
    // so the function is unchanged, and p stays far inside the fp32 range. The decision
    // is one ballot per tile (wave-uniform), so a skipped rescale costs a scalar branch.
    if (__builtin_amdgcn_ballot_w64(mx > ws.m + lazy_raw) != 0) {
      const float m_new = fmaxf(ws.m, mx);
      // Guard: a row with no visible key so far keeps m = -inf; using 0 in the exponent keeps
      // every masked p = exp2(-inf) = 0 and alpha = 0 (acc and l are still 0), never NaN.
      const float m_use = (m_new == -__builtin_inff()) ? 0.f : m_new;
      const float alpha = exp2_hw((ws.m - m_use) * c);
      ws.l *= alpha;
#pragma unroll
      for (int db = 0; db < kDB; ++db) ws.o[db] *= alpha;
      ws.m = m_new;
      ws.mc = m_use * c;
    }
#pragma unroll
    for (int kb = 0; kb < kKB; ++kb) {
      if (kb < nvalid) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[kb][r] = exp2_hw(__builtin_fmaf(s[kb][r], c, -ws.mc));
      }
    }
    // ---- O^T += V^T P^T, and the row sum ---------------------------------------------------
    float rs = 0.f;
#pragma unroll
    for (int kb = 0; kb < kKB; ++kb) {
      if (kb < nvalid) {
#pragma unroll
        for (int r = 0; r < 16; ++r) rs += s[kb][r];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
          for (int db = 0; db < kDB; ++db) {
            const f32x4 a = *reinterpret_cast<const f32x4*>(Vt + (32 * db + r32) * kLdV +
                                                            32 * kb + 8 * j + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) ws.o[db] = mma32(a[e], s[kb][4 * j + e], ws.o[db]);
          }
        }
      }
    }
    ws.l += rs;
  }

  // `lds`: kLdsBytes of the workgroup's LDS, 16-byte aligned.
  __device__ static void run(const KArgs& a, const Where& w, Tc* lds) {
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    // readfirstlane makes the wave index (and everything derived from it: the wave's rows, key
    // range, diagonal block) provably wave-uniform, so per-wave decisions are scalar branches.
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 5;
    const int b = w.b, h = w.h, hk = w.hk, qt = w.qt;
    const int N = a.N;

    const Tio* qb = static_cast<const Tio*>(a.q) + b * a.qsb + h * a.qsh;
    const Tio* kb = static_cast<const Tio*>(a.k) + b * a.ksb + hk * a.ksh;
    const Tio* vb = static_cast<const Tio*>(a.v) + b * a.vsb + hk * a.vsh;

    const int i0 = qt * kBr;
    const int r0 = i0 + 32 * wave;  // this wave's first row
    const bool wave_valid = wave < WAVES && r0 < N;
    const int row = r0 + (lane & 31);

    // Key range of the workgroup: causal stops at its last row (tiles beyond are never loaded).
    const int kv_end = a.causal ? min(N, i0 + kBr) : N;
    const int n_tiles = (kv_end + BC - 1) / BC;
    // Key range of this wave (exclusive end), in whole 32-key blocks.
    const int wave_end = wave_valid ? (a.causal ? min(N, r0 + 32) : N) : 0;

    WaveState ws;
    load_q(ws, qb, row, a.qsn, wave_valid, g);
#pragma unroll
    for (int db = 0; db < kDB; ++db) ws.o[db] = f32x16{};
    ws.m = -__builtin_inff();
    ws.mc = 0.f;
    ws.l = 0.f;

    const float lazy_raw = kLazyLog2 / a.c;  // lazy-rescale threshold, raw score units
    Staging st;
    if constexpr (PREFETCH) {
      load_tile(st, kb, vb, 0, N, a.ksn, a.vsn, tid);
      store_tile(st, lds, tid);
      __syncthreads();
      for (int t = 0; t < n_tiles; ++t) {
        const int k0 = t * BC;
        if (t + 1 < n_tiles) load_tile(st, kb, vb, k0 + BC, N, a.ksn, a.vsn, tid);
        const int nvalid = max(0, min(kKB, (wave_end - k0 + 31) / 32));
        if (nvalid > 0) {
          const int diag = a.causal ? (r0 - k0) / 32 : -1;  // r0, k0 multiples of 32
          compute_tile(ws, lds + (t & 1) * kBufElems, nvalid,
                       (diag >= 0 && diag < nvalid) ? diag : -1, a.c, lazy_raw, lane);
        }
        if (t + 1 < n_tiles) store_tile(st, lds + ((t + 1) & 1) * kBufElems, tid);
        __syncthreads();
      }
    } else {
      for (int t = 0; t < n_tiles; ++t) {
        const int k0 = t * BC;
        load_tile(st, kb, vb, k0, N, a.ksn, a.vsn, tid);
        store_tile(st, lds, tid);
        __syncthreads();
        const int nvalid = max(0, min(kKB, (wave_end - k0 + 31) / 32));
        if (nvalid > 0) {
          const int diag = a.causal ? (r0 - k0) / 32 : -1;
          compute_tile(ws, lds, nvalid, (diag >= 0 && diag < nvalid) ? diag : -1, a.c, lazy_raw,
                       lane);
        }
        __syncthreads();
      }
    }

    // ---- epilogue: O = acc / l, lse = m*scale + ln l (ref:include/fa/softmax_math.cuh:58-71) --
    const float lt = halves_sum(ws.l);
    if (!wave_valid) return;
    const float inv = (lt > 0.f) ? 1.f / lt : 0.f;
    // With helper waves the lane again: kept over the walk it costs registers that the fp32 split kernel,
    // which falls back to this one, does not have.
    const int out_lane =
        THREADS == 64 * WAVES
            ? lane
            : static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
    const int out_g = out_lane >> 5;
    const int out_row = r0 + (out_lane & 31);
    Tio* orow = static_cast<Tio*>(a.o) + b * a.osb + h * a.osh + out_row * a.osn;
#pragma unroll
    for (int db = 0; db < kDB; ++db) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = 32 * db + 8 * j + 4 * out_g;
        const float x0 = ws.o[db][4 * j + 0] * inv, x1 = ws.o[db][4 * j + 1] * inv;
        const float x2 = ws.o[db][4 * j + 2] * inv, x3 = ws.o[db][4 * j + 3] * inv;
        if constexpr (__is_same(Tio, float)) {
          *reinterpret_cast<f32x4*>(orow + d) = f32x4{x0, x1, x2, x3};
        } else {
          *reinterpret_cast<f16x4*>(orow + d) =
              f16x4{(_Float16)x0, (_Float16)x1, (_Float16)x2, (_Float16)x3};
        }
      }
    }
    if (out_g == 0) {
      a.lse[(static_cast<size_t>(b) * a.H + h) * static_cast<size_t>(N) + out_row] =
          (lt > 0.f && ws.m != -__builtin_inff()) ? ws.m * a.scale + log2_hw(lt) * kLn2
                                                   : __builtin_inff();
    }
  }
};

// Kernel entry point of the fp32 rung (profiler-visible name of stage 3).
template <typename T, int D, int WAVES, int BC>
__global__ __launch_bounds__(64 * WAVES) void fa_s3_fused(KArgs a) {
  using A = Attn<T, D, WAVES, BC, true>;
  __shared__ __attribute__((aligned(16))) float lds[A::kLdsElems];
  A::run(a, where(a), lds);
}

// Host-side launch of one instantiated stage-3 variant.
template <typename T, int D, int WAVES, int BC>
int launch_s3(const KArgs& in, hipStream_t stream) {
  using A = Attn<T, D, WAVES, BC, true>;
  KArgs a = in;
  a.n_qtiles = (a.N + A::kBr - 1) / A::kBr;
  const long long grid = static_cast<long long>(a.n_qtiles) * a.B * a.H;
  if (grid <= 0 || grid > 0x7fffffffLL) return static_cast<int>(hipErrorInvalidValue);
  fill_grid(a);
  hipLaunchKernelGGL((fa_s3_fused<T, D, WAVES, BC>), dim3(static_cast<unsigned>(grid)),
                     dim3(A::kThreads), 0, stream, a);
  return static_cast<int>(hipGetLastError());
}

template <typename T, int D, int WAVES, int BC>
constexpr Variant variant_s3() {
  return Variant{D, 32 * WAVES, BC, &launch_s3<T, D, WAVES, BC>, WAVES};
}

// Stage 3: BR fixed at 128, BC in {32, 64}.
template <typename T>
VariantList s3_table() {
  static const Variant t[] = {variant_s3<T, 64, 4, 32>(), variant_s3<T, 64, 4, 64>(),
                              variant_s3<T, 128, 4, 32>(), variant_s3<T, 128, 4, 64>()};
  return VariantList{t, static_cast<int>(sizeof(t) / sizeof(t[0]))};
}

}  // namespace kern
}  // namespace fa
