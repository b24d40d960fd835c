// MFMA GEMM for prefill and batched decode: C[M, N] = A[M, K] x W[N, K]^T with fused epilogues.
// Both operands are K-contiguous and accumulation is float32; bf16 uses v_mfma_f32_32x32x16_bf16, float32 uses
// v_mfma_f32_32x32x2_f32 (true fp32) up to 32 rows.  Four kernels share the epilogues:
//   gemm_kernel      any dtype and shape: global -> registers -> LDS (padded rows, so that the 16-byte fragment
//                    reads of a 32x32 MFMA hit distinct banks), LDS double-buffered;
//   gemm_dma_kernel  large 16-bit problems: 256x256x64 tiles written straight into LDS by the memory pipeline
//                    (buffer_load ... lds), rows xor-swizzled instead of padded, no staging registers;
//   gemm_stream_kernel  16-bit problems of few rows: the same operand path, all rows in one tile, three or four stages;
//   gemm_split_kernel  float32 problems of more than 32 rows: every operand as a sum of three bf16 numbers, float32 totals of
//                    short sums (more exact than v_mfma_f32_32x32x2_f32 over the same K).
#include "mtj_common.h"
#include <type_traits>

namespace {

template <typename T> struct mma;
template <> struct mma<bf16_t> {
  static constexpr int EPC = 8;  // elements per 16-byte chunk
  struct frag { bf16x8 v; };
  __device__ static __forceinline__ frag load(const bf16_t* p) {
    frag f;
    f.v = *reinterpret_cast<const bf16x8*>(p);
    return f;
  }
  __device__ static __forceinline__ void run(floatx16& c, const frag& a, const frag& b) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b.v, c, 0, 0, 0);
  }
  __device__ static __forceinline__ void run16(floatx4& c, const frag& a, const frag& b) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, c, 0, 0, 0);
  }
};
template <> struct mma<f16_t> {
  static constexpr int EPC = 8;
  struct frag { f16x8 v; };
  __device__ static __forceinline__ frag load(const f16_t* p) {
    frag f;
    f.v = *reinterpret_cast<const f16x8*>(p);
    return f;
  }
  __device__ static __forceinline__ void run(floatx16& c, const frag& a, const frag& b) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.v, b.v, c, 0, 0, 0);
  }
  __device__ static __forceinline__ void run16(floatx4& c, const frag& a, const frag& b) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.v, b.v, c, 0, 0, 0);
  }
};
template <> struct mma<float> {
  static constexpr int EPC = 4;
  struct frag { floatx4 lo, hi; };
  __device__ static __forceinline__ frag load(const float* p) {
    frag f;
    f.lo = *reinterpret_cast<const floatx4*>(p);
    f.hi = *reinterpret_cast<const floatx4*>(p + 4);
    return f;
  }
  __device__ static __forceinline__ void run(floatx16& c, const frag& a, const frag& b) {
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.lo.x, b.lo.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.lo.y, b.lo.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.lo.z, b.lo.z, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.lo.w, b.lo.w, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.hi.x, b.hi.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.hi.y, b.hi.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.hi.z, b.hi.z, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.hi.w, b.hi.w, c, 0, 0, 0);
  }
};

struct gemm_args {
  const void* A;
  int64_t lda;
  const void* W;
  const float* bias;
  int M, N, K;
  void* out;
  int64_t ldo;
  int out_dtype;
  float alpha;            // multiplies the accumulator first (undoes a power-of-two scale of the packed weights)
  int m_base;             // INPROJ: what row 0 is the row of (a call may run as two launches)
  int splits;             // > 1: blockIdx.y owns a K range and stores a raw float32 partial at out + y * split_stride
  int64_t split_stride;
  mtj_inproj ip;
  // MTJ_EPI_XENT: the product is never stored; per (row, column tile) the maximum and the sum of exp(logit - maximum)
  const int32_t* target;  // [M]
  float* pmax;            // [tiles_n, M]
  float* psum;            // [tiles_n, M]
  float* tlogit;          // [M]: the logit of the target column (written by the one tile that holds it)
};

constexpr int MTJ_EPI_XENT = 3;   // internal: logits + cross entropy (ProjectionShard.loss, layers.py:569-593)

// 16 consecutive elements, 16-byte vector stores (idx is a multiple of 16 elements, base 16-byte aligned)
__device__ __forceinline__ void store16(void* base, int64_t idx, const float* v, int dtype) {
  if (dtype == MTJ_F32) {
    floatx4* p = reinterpret_cast<floatx4*>(reinterpret_cast<float*>(base) + idx);
#pragma unroll
    for (int q = 0; q < 4; ++q) p[q] = floatx4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
  } else {
    uint32x4* p = reinterpret_cast<uint32x4*>(reinterpret_cast<uint16_t*>(base) + idx);
#pragma unroll
    for (int q = 0; q < 2; ++q)
      p[q] = uint32x4{pack_16x2(v[8 * q], v[8 * q + 1], dtype), pack_16x2(v[8 * q + 2], v[8 * q + 3], dtype),
                      pack_16x2(v[8 * q + 4], v[8 * q + 5], dtype), pack_16x2(v[8 * q + 6], v[8 * q + 7], dtype)};
  }
}

// compile-time loop over the accumulator tiles (i, j) of a wavefront: the indices must be constants for the
// accumulators to stay in registers
template <int I, int J, int WM, int WN, class F>
__device__ __forceinline__ void for_tiles(F&& f) {
  f(std::integral_constant<int, I>{}, std::integral_constant<int, J>{});
  if constexpr (I + 1 < WM) for_tiles<I + 1, J, WM, WN>(f);
  else if constexpr (J + 1 < WN) for_tiles<0, J + 1, WM, WN>(f);
}

template <int S, int NS, class F>
__device__ __forceinline__ void for_stages(F&& f) {
  f(std::integral_constant<int, S>{});
  if constexpr (S + 1 < NS) for_stages<S + 1, NS>(f);
}

// per-tile operands of the fused input-projection epilogue, fetched one tile ahead of their use:
// fc_in columns: 16 bias values; rotary q/k columns: 8 sines then 8 cosines
struct epi_ops { floatx4 o[4]; };

// Epilogue of a workgroup tile whose wavefront (wm, wn) holds WM x WN accumulator tiles of 32x32.  `smem` (the
// operand staging area, no longer needed) must hold 3*BM ints and one 32x36 float patch per wavefront.
// Two accumulator layouts:
//   MI16 false  acc is floatx16[WM][WN] from 32x32 MFMAs: register v of lane l holds C[8*(v/4) + 4*(l/32) + v%4][l%32];
//   MI16 true   acc is floatx4[2*WM][2*WN] from 16x16x32 MFMAs issued with the WEIGHT fragment as the first operand:
//               register v of lane l of block (i, j) holds C[16*i + l%16][16*j + 4*(l/16) + v], four consecutive
//               columns of one row, so stores are 8 or 16 bytes per lane.
template <int EPI, int WAVES_M, int WAVES_N, int WM, int WN, bool MI16 = false, class ACC>
__device__ __forceinline__ void epilogue(const gemm_args& a, void* out, ACC& acc, unsigned char* smem, int m0, int n0) {
  constexpr int NT = WAVES_M * WAVES_N * 64, BM = WAVES_M * WM * 32;
  constexpr int PS = 36;   // patch row stride in floats: 16-byte aligned rows, and 16-byte reads of 8 lanes hit distinct banks
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  const int fr = lane & 31, fg = lane >> 5;
  if (EPI == MTJ_EPI_XENT) {
    // Row statistics of this workgroup's column tile: accumulator register v of lane (fr, fg) is row 8*(v/4) + 4*fg +
    // v%4, column fr of a 32x32 tile, so a row is reduced over the WN tiles in registers, then over the 32 lanes
    // with the same fg by shuffles, then over the WAVES_N wavefronts through LDS.
    constexpr int BN = WAVES_N * WN * 32;
    __syncthreads();                                       // every wavefront is done with the operand tiles
    float* red = reinterpret_cast<float*>(smem);           // [WAVES_N][BM][2]
    if constexpr (MI16) {
      // a lane holds 4 columns of each of the 2*WN column blocks of its row; a row is completed by the four lanes
      // l%16 + 16*q, then by the WAVES_N wavefronts through LDS
      const int r16 = lane & 15, q16 = lane >> 4;
      float bias[2 * WN][4];
      bool ok[2 * WN][4];
#pragma unroll
      for (int j = 0; j < 2 * WN; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int n = n0 + (wn * WN * 2 + j) * 16 + 4 * q16 + v;
          ok[j][v] = n < a.N;
          bias[j][v] = (a.bias && ok[j][v]) ? a.bias[n] : 0.f;
        }
      for_tiles<0, 0, 2 * WM, 1>([&](auto I_, auto) {
        constexpr int i = decltype(I_)::value;
        const int r = (wm * WM * 2 + i) * 16 + r16;
        const int m = m0 + r;
        float val[2 * WN][4];
        float mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < 2 * WN; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            val[j][v] = ok[j][v] ? acc[i][j][v] * a.alpha + bias[j][v] : -INFINITY;
            mx = fmaxf(mx, val[j][v]);
          }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        // exp(-inf) = 0 for columns beyond N; without a maximum the sum is 0, or NaN if a logit is
        const float ref = mx == -INFINITY ? 0.f : mx;
        float sm = 0.f;
#pragma unroll
        for (int j = 0; j < 2 * WN; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v) sm += __expf(val[j][v] - ref);
        sm += __shfl_xor(sm, 16);
        sm += __shfl_xor(sm, 32);
        if (m < a.M) {
          const int t = a.target[m];
#pragma unroll
          for (int j = 0; j < 2 * WN; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              if (n0 + (wn * WN * 2 + j) * 16 + 4 * q16 + v == t) a.tlogit[m] = val[j][v];
        }
        if (q16 == 0) {
          red[(wn * BM + r) * 2] = mx;
          red[(wn * BM + r) * 2 + 1] = sm;
        }
      });
    } else
    for_tiles<0, 0, WM, 1>([&](auto I_, auto) {
      constexpr int i = decltype(I_)::value;
      float val[WN][16];
      int col[WN];
      for_tiles<0, 0, 1, WN>([&](auto, auto J_) {
        constexpr int j = decltype(J_)::value;
        const int n = n0 + (wn * WN + j) * 32 + fr;
        col[j] = n;
        const bool n_ok = n < a.N;
        const float bias = (a.bias && n_ok) ? a.bias[n] : 0.f;
#pragma unroll
        for (int v = 0; v < 16; ++v) val[j][v] = n_ok ? acc[i][j][v] * a.alpha + bias : -INFINITY;
      });
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int r = (wm * WM + i) * 32 + 8 * (v / 4) + 4 * fg + (v % 4);
        const int m = m0 + r;
        float mx = val[0][v];
#pragma unroll
        for (int j = 1; j < WN; ++j) mx = fmaxf(mx, val[j][v]);
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        float sm = 0.f;
        if (mx != -INFINITY) {
#pragma unroll
          for (int j = 0; j < WN; ++j) sm += __expf(val[j][v] - mx);      // exp(-inf) = 0 for columns beyond N
        }
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) sm += __shfl_xor(sm, o);
        if (m < a.M) {
          const int t = a.target[m];
#pragma unroll
          for (int j = 0; j < WN; ++j)
            if (col[j] == t) a.tlogit[m] = val[j][v];
        }
        if (fr == 0) {
          red[(wn * BM + r) * 2] = mx;
          red[(wn * BM + r) * 2 + 1] = sm;
        }
      }
    });
    __syncthreads();
    const int tn = n0 / BN;
    for (int r = tid; r < BM; r += NT) {
      const int m = m0 + r;
      if (m >= a.M) continue;
      float mx = -INFINITY;
#pragma unroll
      for (int w = 0; w < WAVES_N; ++w) mx = fmaxf(mx, red[(w * BM + r) * 2]);
      float sm = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES_N; ++w) {
        const float pm = red[(w * BM + r) * 2], ps = red[(w * BM + r) * 2 + 1];
        sm += pm == -INFINITY ? ps : __expf(pm - mx) * ps;     // (0 or NaN where there is no maximum)
      }
      a.pmax[(int64_t)tn * a.M + m] = mx;
      a.psum[(int64_t)tn * a.M + m] = sm;
    }
  } else if (EPI == MTJ_EPI_INPROJ) {
    // Each 32x32 accumulator tile goes through a private LDS patch of its wavefront and comes back with one
    // lane owning 16 consecutive columns of one row: rotary pairs are then lane-local and every destination
    // (q, K/V window, gelu(fc_in)) gets 32- or 64-byte stores.
    __syncthreads();                                       // every wavefront is done with the operand tiles
    int* row_b = reinterpret_cast<int*>(smem);
    int* row_pos = row_b + BM;
    int* row_t = row_pos + BM;
    float* patch = reinterpret_cast<float*>(smem) + 3 * BM + wave * (32 * PS);
    for (int r = tid; r < BM; r += NT) {
      const int m = m0 + r;
      int b = 0, pos = -1, t = 0;
      if (m < a.M) {
        const int rect = a.ip.rows ? a.ip.rows[m + a.m_base] : m + a.m_base;     // row of the [B, Tp] rectangle
        b = rect / a.ip.Tp;
        t = rect - b * a.ip.Tp;
        pos = a.ip.pos0[b] + t;
      }
      row_b[r] = b;
      row_pos[r] = pos;
      row_t[r] = t;
    }
    __syncthreads();
    const int d = a.ip.n_heads * a.ip.d_head, dh = a.ip.d_head, rd = a.ip.rotary_dims, Tp = a.ip.Tp;
    const int prow = lane >> 1, pcol = (lane & 1) * 16;     // my row / first column inside a tile

    // tile-uniform facts of accumulator tile column j, and my first column inside its segment
    struct col_info { bool is_fc, n_ok; int seg, c0, h, e0; };
    auto column = [&](int j) {
      col_info c;
      const int nb = n0 + (wn * WN + j) * 32;               // first column of the tile
      c.is_fc = nb >= 3 * d;
      c.seg = c.is_fc ? 3 : nb / d;                         // 0 q, 1 v, 2 k
      c.c0 = nb - c.seg * d + pcol;
      c.h = c.c0 / dh;
      c.e0 = c.c0 - c.h * dh;
      c.n_ok = nb + pcol < a.N;                             // N is a multiple of 16 columns here
      return c;
    };
    auto load_ops = [&](int i, int j) {
      epi_ops p;
#pragma unroll
      for (int q = 0; q < 4; ++q) p.o[q] = floatx4{0.f, 0.f, 0.f, 0.f};
      const col_info c = column(j);
      if (!c.n_ok) return p;
      if (c.is_fc) {
        const floatx4* bp = reinterpret_cast<const floatx4*>(a.bias + c.c0);   // c0 is a multiple of 16
#pragma unroll
        for (int q = 0; q < 4; ++q) p.o[q] = bp[q];
      } else if (c.seg != 1 && c.e0 < rd) {                 // rd is a multiple of 16 (checked on the host)
        const int pos = row_pos[(wm * WM + i) * 32 + prow];
        if (pos >= 0) {
          const int pp = pos < a.ip.max_pos ? pos : a.ip.max_pos - 1;
          const floatx4* sp = reinterpret_cast<const floatx4*>(a.ip.sin_tab + (int64_t)pp * (rd / 2) + (c.e0 >> 1));
          const floatx4* cp = reinterpret_cast<const floatx4*>(a.ip.cos_tab + (int64_t)pp * (rd / 2) + (c.e0 >> 1));
          p.o[0] = sp[0]; p.o[1] = sp[1]; p.o[2] = cp[0]; p.o[3] = cp[1];
        }
      }
      return p;
    };
    epi_ops cur = load_ops(0, 0);
    for_tiles<0, 0, WM, WN>([&](auto I_, auto J_) {
      constexpr int i = decltype(I_)::value, j = decltype(J_)::value;
      constexpr int ni = i + 1 < WM ? i + 1 : 0, nj = i + 1 < WM ? j : j + 1;
      epi_ops nxt = cur;
      if constexpr (nj < WN) nxt = load_ops(ni, nj);
      const col_info c = column(j);
      if constexpr (MI16) {
#pragma unroll
        for (int ii = 0; ii < 2; ++ii)
#pragma unroll
          for (int jj = 0; jj < 2; ++jj)
            *reinterpret_cast<floatx4*>(patch + (ii * 16 + (lane & 15)) * PS + jj * 16 + 4 * (lane >> 4)) =
                acc[2 * i + ii][2 * j + jj] * a.alpha;
      } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) patch[(8 * (v / 4) + 4 * fg + (v % 4)) * PS + fr] = acc[i][j][v] * a.alpha;
      }
      __builtin_amdgcn_wave_barrier();
      float val[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const floatx4 t = *reinterpret_cast<const floatx4*>(patch + prow * PS + pcol + 4 * q);
        val[4 * q] = t.x; val[4 * q + 1] = t.y; val[4 * q + 2] = t.z; val[4 * q + 3] = t.w;
      }
      __builtin_amdgcn_wave_barrier();
      const int r = (wm * WM + i) * 32 + prow;
      const int m = m0 + r;
      if (m < a.M && c.n_ok) {
        if (c.is_fc) {
#pragma unroll
          for (int k = 0; k < 16; ++k) val[k] = gelu_tanh(val[k] + cur.o[k >> 2][k & 3]);
          store16(a.ip.act, (int64_t)(m + a.m_base) * a.ip.ld_act + d + c.c0, val, a.ip.act_dtype);
        } else {
          const int pos = row_pos[r];
          if (pos >= 0) {
            const int b = row_b[r];
            if (c.seg != 1 && c.e0 < rd) {
#pragma unroll
              for (int k = 0; k < 16; k += 2) {
                const float sn = cur.o[k >> 3][(k >> 1) & 3], cs = cur.o[2 + (k >> 3)][(k >> 1) & 3];
                const float x0 = val[k], x1 = val[k + 1];
                val[k] = x0 * cs - x1 * sn;
                val[k + 1] = x1 * cs + x0 * sn;
              }
            }
            const int64_t bh = (int64_t)b * a.ip.n_heads + c.h;
            if (c.seg == 0) {
              store16(a.ip.q, (bh * Tp + row_t[r]) * dh + c.e0, val, a.ip.q_dtype);
            } else {
              const int slot = pos % a.ip.Tcap;
              store16(c.seg == 1 ? a.ip.v_cache : a.ip.k_cache, (bh * a.ip.Tcap + slot) * dh + c.e0, val, a.ip.kv_dtype);
              if (c.seg == 1 && a.ip.v_t && pos < a.ip.ldvt) {
#pragma unroll
                for (int k = 0; k < 16; ++k) store_as(a.ip.v_t, (bh * dh + c.e0 + k) * a.ip.ldvt + pos, val[k], a.ip.kv_dtype);
              }
            }
          }
        }
      }
      cur = nxt;
    });
  } else if constexpr (MI16) {
    // four consecutive columns per lane: 16-byte (float32) or 8-byte (16-bit) accesses when the rows of `out` allow it
    const int r16 = lane & 15, q16 = lane >> 4;
    const int esz = (EPI == MTJ_EPI_RESID || a.out_dtype == MTJ_F32) ? 4 : 2;
    const bool vec = a.ldo % 4 == 0 && (reinterpret_cast<uintptr_t>(out) % (4 * esz)) == 0;
    for_tiles<0, 0, 1, 2 * WN>([&](auto, auto J_) {
      constexpr int j = decltype(J_)::value;
      const int nb = n0 + (wn * WN * 2 + j) * 16 + 4 * q16;
      float bias[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) bias[v] = (a.bias && nb + v < a.N) ? a.bias[nb + v] : 0.f;
      const bool full = vec && nb + 3 < a.N;
      for_tiles<0, 0, 2 * WM, 1>([&](auto I_, auto) {
        constexpr int i = decltype(I_)::value;
        const int m = m0 + (wm * WM * 2 + i) * 16 + r16;
        if (m >= a.M) return;
        const int64_t idx = (int64_t)m * a.ldo + nb;
        float val[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) val[v] = acc[i][j][v] * a.alpha + bias[v];
        if (full) {
          if (EPI == MTJ_EPI_RESID) {
            floatx4* o = reinterpret_cast<floatx4*>(reinterpret_cast<float*>(out) + idx);
            const floatx4 old = *o;
            *o = floatx4{old.x + val[0], old.y + val[1], old.z + val[2], old.w + val[3]};
          } else if (a.out_dtype == MTJ_F32) {
            *reinterpret_cast<floatx4*>(reinterpret_cast<float*>(out) + idx) = floatx4{val[0], val[1], val[2], val[3]};
          } else {
            *reinterpret_cast<uint32x2*>(reinterpret_cast<uint16_t*>(out) + idx) =
                uint32x2{pack_16x2(val[0], val[1], a.out_dtype), pack_16x2(val[2], val[3], a.out_dtype)};
          }
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (nb + v < a.N) {
              if (EPI == MTJ_EPI_RESID) reinterpret_cast<float*>(out)[idx + v] += val[v];
              else store_as(out, idx + v, val[v], a.out_dtype);
            }
        }
      });
    });
  } else {
    for_tiles<0, 0, WM, WN>([&](auto I_, auto J_) {
      constexpr int i = decltype(I_)::value, j = decltype(J_)::value;
      const int n = n0 + (wn * WN + j) * 32 + fr;
      const bool n_ok = n < a.N;
      const float bias = (a.bias && n_ok) ? a.bias[n] : 0.f;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = m0 + (wm * WM + i) * 32 + 8 * (v / 4) + 4 * fg + (v % 4);
        if (m < a.M && n_ok) {
          const int64_t idx = (int64_t)m * a.ldo + n;
          const float val = acc[i][j][v] * a.alpha + bias;
          if (EPI == MTJ_EPI_RESID) reinterpret_cast<float*>(out)[idx] += val;
          else store_as(out, idx, val, a.out_dtype);
        }
      }
    });
  }
}

// Workgroup tile (WAVES_M*WM*32) x (WAVES_N*WN*32), K step BK elements, NS register stages, epilogue EPI.
//
// Pipeline: k-tile kt is multiplied out of LDS (two buffers) while the loads of k-tiles kt+1 .. kt+NS sit in
// registers or are still in flight; one k-tile in flight does not cover the load latency of a loaded GPU.
// Global reads are bounds-checked buffer loads (rows beyond M or N read as zero), whose addressing needs one
// VGPR per operand: the per-chunk and per-k-tile offsets are scalar.
template <typename T, int EPI, int WAVES_M, int WAVES_N, int WM, int WN, int BK, int NS>
__global__ __launch_bounds__(WAVES_M* WAVES_N * 64) void gemm_kernel(const gemm_args a) {
  constexpr int NT = WAVES_M * WAVES_N * 64;
  constexpr int BM = WAVES_M * WM * 32, BN = WAVES_N * WN * 32;
  constexpr int EPC = mma<T>::EPC;
  constexpr int ESZ = (int)sizeof(T);
  constexpr int CPR = BK / EPC;          // 16-byte chunks per tile row
  constexpr int LDS_ROW = BK + EPC;      // padded row, elements (row stride 144 B for both types)
  constexpr int A_CHUNKS = BM * CPR / NT, B_CHUNKS = BN * CPR / NT;
  constexpr int ROWS_PER_PASS = NT / CPR;   // tile rows covered by one chunk index
  static_assert(BM * CPR % NT == 0 && BN * CPR % NT == 0 && NT % CPR == 0, "tile does not divide over threads");
  static_assert(BK % 16 == 0, "BK must hold whole MFMA k-steps");

  extern __shared__ __align__(16) unsigned char smem[];
  T* As = reinterpret_cast<T*>(smem);                    // [2][BM][LDS_ROW]
  T* Bs = As + 2 * BM * LDS_ROW;                         // [2][BN][LDS_ROW]

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  const int fr = lane & 31, fg = lane >> 5;

  // ---- tile id: give each XCD (workgroups are dealt round-robin over 8 XCDs) a contiguous range of
  // tiles, then walk that range in groups of 8 row-tiles so one XCD's L2 sees few distinct W panels.
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
  const int nblk = tiles_m * tiles_n;
  int pid = blockIdx.x;
  {
    const int per = nblk / 8;
    if (pid < per * 8) pid = (pid % 8) * per + pid / 8;
  }
  constexpr int GM = 8;
  const int group = pid / (GM * tiles_n);
  const int first_m = group * GM;
  const int gsz = (tiles_m - first_m < GM) ? tiles_m - first_m : GM;
  const int tm = first_m + (pid % (GM * tiles_n)) % gsz;
  const int tn = (pid % (GM * tiles_n)) / gsz;
  const int m0 = tm * BM, n0 = tn * BN;

  // buffer resources over the rows of this tile: [m0, min(M, m0+BM)) of A and [n0, min(N, n0+BN)) of W
  const int rows_a = (a.M - m0 < BM) ? a.M - m0 : BM, rows_b = (a.N - n0 < BN) ? a.N - n0 : BN;
  const T* tile_a = reinterpret_cast<const T*>(a.A) + (int64_t)m0 * a.lda;
  const T* tile_b = reinterpret_cast<const T*>(a.W) + (int64_t)n0 * a.K;
  const __amdgpu_buffer_rsrc_t ra_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(tile_a), 0, (int)((((int64_t)rows_a - 1) * a.lda + a.K) * ESZ), 0x00020000);
  const __amdgpu_buffer_rsrc_t rb_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(tile_b), 0, (int)((((int64_t)rows_b - 1) * a.K + a.K) * ESZ), 0x00020000);
  const int row0 = tid / CPR, cc0 = tid % CPR;
  const int voff_a = (int)(((int64_t)row0 * a.lda + cc0 * EPC) * ESZ);
  const int voff_b = (int)(((int64_t)row0 * a.K + cc0 * EPC) * ESZ);
  const int pass_a = (int)((int64_t)ROWS_PER_PASS * a.lda * ESZ), pass_b = (int)((int64_t)ROWS_PER_PASS * a.K * ESZ);

  const int kt0 = (int)((int64_t)blockIdx.y * (a.K / BK) / a.splits);   // first k-tile of my K range
  const int KT = (int)((int64_t)(blockIdx.y + 1) * (a.K / BK) / a.splits) - kt0;
  // With few rows the weights are streamed once and every workgroup would ask for the same k offset of its rows at
  // the same time - addresses that differ by multiples of the row pitch, a power of two, which crowd into few memory
  // channels.  Each workgroup therefore starts its walk over k at a different k-tile and wraps around (M = 32,
  // N = 28672, K = 4096: 48.8 -> 41.5 us; which multiplier spreads the starts does not matter).  The start is a function
  // of the column tile alone: an output row is summed in the same order whatever else is in the batch.
  const int krot = BM <= 64 ? (int)(((unsigned)tn * 5u) % (unsigned)KT) : 0;
  uint32x4 ra[NS][A_CHUNKS], rb[NS][B_CHUNKS];
  auto load_global = [&](auto ST_, int kt) {
    constexpr int st = decltype(ST_)::value;
    const int kr = kt + krot;
    const int koff = (kt0 + (kr >= KT ? kr - KT : kr)) * BK * ESZ;
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i)
      ra[st][i] = __builtin_amdgcn_raw_buffer_load_b128(ra_rsrc, voff_a, koff + i * pass_a, 0);
#pragma unroll
    for (int i = 0; i < B_CHUNKS; ++i)
      rb[st][i] = __builtin_amdgcn_raw_buffer_load_b128(rb_rsrc, voff_b, koff + i * pass_b, BM <= 64 ? 2 : 0);  // nt: streamed once
  };
  auto store_lds = [&](auto ST_, int buf) {
    constexpr int st = decltype(ST_)::value;
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i)
      *reinterpret_cast<uint32x4*>(As + (buf * BM + row0 + i * ROWS_PER_PASS) * LDS_ROW + cc0 * EPC) = ra[st][i];
#pragma unroll
    for (int i = 0; i < B_CHUNKS; ++i)
      *reinterpret_cast<uint32x4*>(Bs + (buf * BN + row0 + i * ROWS_PER_PASS) * LDS_ROW + cc0 * EPC) = rb[st][i];
  };

  floatx16 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // k-tile t lives in register stage t % NS.  Prologue: request k-tiles 0 .. NS-1, park k-tile 0 in LDS,
  // reuse its stage for k-tile NS.
  for_stages<0, NS>([&](auto ST_) {
    if (decltype(ST_)::value < KT) load_global(ST_, decltype(ST_)::value);
  });
  store_lds(std::integral_constant<int, 0>{}, 0);
  if (NS < KT) load_global(std::integral_constant<int, 0>{}, NS);
  __syncthreads();

  // one k-tile; PARK = stage of k-tile kt+1 (a compile-time index: the k loop is unrolled by NS).  STEADY: k-tiles
  // kt+1 and kt+1+NS both exist, so the park and the request are unconditional.  That matters: the wait the
  // compiler puts before the park is the strictest over all paths that reach it, and with the request under a
  // condition that is "everything outstanding", the request of one iteration ago included.
  auto k_tile = [&](int kt, auto PARK_, auto STEADY_) {
    constexpr bool steady = decltype(STEADY_)::value;
    const int buf = kt & 1;
    const T* as = As + (buf * BM + wm * WM * 32 + fr) * LDS_ROW + fg * 8;
    const T* bs = Bs + (buf * BN + wn * WN * 32 + fr) * LDS_ROW + fg * 8;
    // fragments of k-step ks+1 are read from LDS while the MFMAs of k-step ks run
    typename mma<T>::frag fa[2][WM], fb[2][WN];
#pragma unroll
    for (int i = 0; i < WM; ++i) fa[0][i] = mma<T>::load(as + i * 32 * LDS_ROW);
#pragma unroll
    for (int j = 0; j < WN; ++j) fb[0][j] = mma<T>::load(bs + j * 32 * LDS_ROW);
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      const int cur = ks & 1, nxt = cur ^ 1;
      if (ks + 1 < BK / 16) {
#pragma unroll
        for (int i = 0; i < WM; ++i) fa[nxt][i] = mma<T>::load(as + i * 32 * LDS_ROW + (ks + 1) * 16);
#pragma unroll
        for (int j = 0; j < WN; ++j) fb[nxt][j] = mma<T>::load(bs + j * 32 * LDS_ROW + (ks + 1) * 16);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) mma<T>::run(acc[i][j], fa[cur][i], fb[cur][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (steady || kt + 1 < KT) store_lds(PARK_, buf ^ 1);
    if (steady || kt + 1 + NS < KT) load_global(PARK_, kt + 1 + NS);
    __syncthreads();
  };
  int kt = 0;
  for (; kt + 2 * NS < KT; kt += NS)          // the last k-tile of the round, kt+NS-1, still requests kt+2*NS
    for_stages<0, NS>([&](auto S_) {
      constexpr int s = decltype(S_)::value;
      k_tile(kt + s, std::integral_constant<int, (s + 1) % NS>{}, std::true_type{});
    });
  for (; kt < KT; kt += NS)
    for_stages<0, NS>([&](auto S_) {
      constexpr int s = decltype(S_)::value;
      if (kt + s < KT) k_tile(kt + s, std::integral_constant<int, (s + 1) % NS>{}, std::false_type{});
    });

  void* out = a.splits > 1 ? (void*)(reinterpret_cast<float*>(a.out) + blockIdx.y * a.split_stride) : a.out;
  epilogue<EPI, WAVES_M, WAVES_N, WM, WN>(a, out, acc, smem, m0, n0);
}

// float32 operands on the bf16 matrix cores.  A float32 number is the sum of three bf16 numbers without an error (rounded to
// nearest, each takes 8 of the 24 significant bits of what the ones before it leave), so a product is nine products of
// parts; the six with the largest weights are taken - the other three together are below 2^-24 of the product -.  So that the
// lowest part of the smallest number is a normal bf16 number too, both operands are multiplied by 2^24 first (every float32 number
// is then a multiple of 2^-125); the sums are taken back by 2^-48.
// The bf16 matrix instruction drops low bits of what it adds to a large accumulator, and not symmetrically: with one accumulator
// for all of K the results lay 1e-7 (K = 2560) to 1e-6 (K = 20480) of their root mean square too low, whatever their sign.
// So a sum is only CH k-tiles long and then added to a float32 total by the vector unit, and every second sum (and K range) is
// of products with the sign of A turned, so that what is left of the bias cancels.
// Error against float64, 2-norm / mean, both over the root mean square of the result, with v_mfma_f32_32x32x2_f32 and here:
//   normal operands    K = 512   4.1e-7 / -1e-9  and 1.4e-7 / -2e-9      4096   1.2e-6 / -4e-9 and 1.9e-7 / -1e-9
//                      K = 20480 2.6e-6 /  5e-9  and 3.0e-7 / -1e-9      in four ranges 1.3e-6 / -1e-9 and 2.1e-7 / -2e-10
//   gelu(2 x normal)   K = 4096  1.1e-6 / -3e-10 and 1.9e-7 / -1e-9      20480  2.6e-6 / -8e-10 and 3.0e-7 / -8e-10
//   positive operands  K = 4096  9.3e-7 / -7e-9  and 9.9e-8 / -2e-10     20480  1.9e-6 / -2e-7 and 2.0e-7 / -2e-10
// What is not finite (an operand from 2^103 on or NaN, products or sums from 2^79 on, which the scale takes beyond the largest
// number) is computed again with v_mfma_f32_32x32x2_f32, straight from memory,
// in the tiles of 32 x 32 that hold it (one infinite operand in 200 rows of N = 28672, K = 4096: 734 us instead of 377, 1386 with a
// serial walk per element).
//
// Bound by the vector unit, the barriers and the matrix cores in about equal parts: six v_mfma_f32_32x32x16_bf16 instead of
// eight v_mfma_f32_32x32x2_f32 of twice the length, 13 vector instructions to split two elements, one per accumulator and sum.
// us before and now: N = 28672, K = 4096, 65 / 199 / 600 / 2048 rows 290 / 544 / 1319 / 3516 -> 209 / 346 / 848 / 2420 (1.2 PFLOP/s of bf16
// products); N = 4096, K = 20480, 65 / 128 / 400 / 1024 rows (4 ranges before, up to 16 now) 362 / 380 / 688 / 1379 -> 132 / 150 / 449 /
// 900; N = 3584, K = 512, 127 / 1500 rows 48 / 77 -> 22 / 54.  The sums cost 4 - 6 % of these (a single accumulator: 600 rows 804).
// A k-tile of 16 goes global -> registers (NS k-tiles in flight) -> three bf16 planes per row in LDS, double-buffered: rows
// of 3 x 32 bytes, padded to 112 so that the 16-byte fragment reads of 16 consecutive rows hit distinct banks.
__device__ __forceinline__ bool not_finite(float x) { return !(fabsf(x) < INFINITY); }
constexpr float SPLIT_UP = 0x1p24f, SPLIT_DOWN = 0x1p-48f;

template <int EPI, int WAVES_M, int WAVES_N, int WM, int WN, int NS>
__global__ __launch_bounds__(WAVES_M* WAVES_N * 64, WM * WN > 2 ? 2 : 3) void gemm_split_kernel(const gemm_args a) {
  constexpr int NT = WAVES_M * WAVES_N * 64, BK = 16, CH = 2 * NS;
  constexpr int BM = WAVES_M * WM * 32, BN = WAVES_N * WN * 32;
  constexpr int ROWB = 112, PLANE = 32, STAGEB = (BM + BN) * ROWB;
  constexpr int ROWS_PER_PASS = NT / 2;                    // a thread takes 8 elements of a row at a time
  constexpr int A_U = (BM + ROWS_PER_PASS - 1) / ROWS_PER_PASS, B_U = (BN + ROWS_PER_PASS - 1) / ROWS_PER_PASS;
  static_assert((A_U == 1 || BM % ROWS_PER_PASS == 0) && (B_U == 1 || BN % ROWS_PER_PASS == 0), "tile does not divide over threads");
  extern __shared__ __align__(16) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  const int fr = lane & 31, fg = lane >> 5;

  // tile id as in gemm_kernel
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
  const int nblk = tiles_m * tiles_n;
  int pid = blockIdx.x;
  {
    const int per = nblk / 8;
    if (pid < per * 8) pid = (pid % 8) * per + pid / 8;
  }
  constexpr int GM = 8;
  const int group = pid / (GM * tiles_n);
  const int first_m = group * GM;
  const int gsz = (tiles_m - first_m < GM) ? tiles_m - first_m : GM;
  // (kept in scalar registers: the buffer descriptors are made of them)
  const int tm = __builtin_amdgcn_readfirstlane(first_m + (pid % (GM * tiles_n)) % gsz);
  const int tn = __builtin_amdgcn_readfirstlane((pid % (GM * tiles_n)) / gsz);
  const int m0 = tm * BM, n0 = tn * BN;

  const int rows_a = (a.M - m0 < BM) ? a.M - m0 : BM, rows_b = (a.N - n0 < BN) ? a.N - n0 : BN;
  const float* tile_a = reinterpret_cast<const float*>(a.A) + (int64_t)m0 * a.lda;
  const float* tile_b = reinterpret_cast<const float*>(a.W) + (int64_t)n0 * a.K;
  const __amdgpu_buffer_rsrc_t ra_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(tile_a), 0, (int)((((int64_t)rows_a - 1) * a.lda + a.K) * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t rb_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(tile_b), 0, (int)((((int64_t)rows_b - 1) * a.K + a.K) * 4), 0x00020000);
  const int row0 = tid / 2, half = tid % 2;
  const int voff_a = (int)(((int64_t)row0 * a.lda + half * 8) * 4), voff_b = (int)(((int64_t)row0 * a.K + half * 8) * 4);
  const int pass_a = (int)((int64_t)ROWS_PER_PASS * a.lda * 4), pass_b = (int)((int64_t)ROWS_PER_PASS * a.K * 4);

  const int kt0 = __builtin_amdgcn_readfirstlane((int)((int64_t)blockIdx.y * (a.K / BK) / a.splits));
  const int KT = __builtin_amdgcn_readfirstlane((int)((int64_t)(blockIdx.y + 1) * (a.K / BK) / a.splits)) - kt0;
  uint32x4 ra[NS][A_U][2], rb[NS][B_U][2];
  auto load_global = [&](auto ST_, int kt) {
    constexpr int st = decltype(ST_)::value;
    const int koff = (kt0 + kt) * BK * 4;
#pragma unroll
    for (int i = 0; i < A_U; ++i)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        ra[st][i][c] = __builtin_amdgcn_raw_buffer_load_b128(ra_rsrc, voff_a + 16 * c, koff + i * pass_a, 0);
#pragma unroll
    for (int i = 0; i < B_U; ++i)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        rb[st][i][c] = __builtin_amdgcn_raw_buffer_load_b128(rb_rsrc, voff_b + 16 * c, koff + i * pass_b, 0);
  };
  // eight float32 numbers times `scale` -> three times eight bf16
  auto split_store = [&](unsigned char* dst, const uint32x4 (&r)[2], float scale) {
    float x[8];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) x[4 * c + e] = __uint_as_float(r[c][e]) * scale;
#pragma unroll
    for (int part = 0; part < 3; ++part) {
      uint32x4 p;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p[e] = pack_bf16x2(x[2 * e], x[2 * e + 1]);
        if (part < 2) { x[2 * e] -= bf16_lo(p[e]); x[2 * e + 1] -= bf16_hi(p[e]); }
      }
      *reinterpret_cast<uint32x4*>(dst + part * PLANE) = p;
    }
  };
  const uint32_t range = blockIdx.y;
  auto turned = [&](int kt) { return ((uint32_t)kt / CH + range) & 1u; };      // is k-tile kt of a sum with turned signs?
  auto store_lds = [&](auto ST_, int buf, int kt) {
    const float scale = turned(kt) ? -SPLIT_UP : SPLIT_UP;
    constexpr int st = decltype(ST_)::value;
    unsigned char* d = smem + buf * STAGEB + row0 * ROWB + half * 16;
#pragma unroll
    for (int i = 0; i < A_U; ++i)
      if (BM >= ROWS_PER_PASS || row0 < BM) split_store(d + i * ROWS_PER_PASS * ROWB, ra[st][i], scale);
#pragma unroll
    for (int i = 0; i < B_U; ++i)
      if (BN >= ROWS_PER_PASS || row0 < BN) split_store(d + (BM + i * ROWS_PER_PASS) * ROWB, rb[st][i], SPLIT_UP);
  };

  floatx16 acc[WM][WN], sum[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  for_stages<0, NS>([&](auto ST_) {
    if (decltype(ST_)::value < KT) load_global(ST_, decltype(ST_)::value);
  });
  store_lds(std::integral_constant<int, 0>{}, 0, 0);
  if (NS < KT) load_global(std::integral_constant<int, 0>{}, NS);
  __syncthreads();

  // k-tile kt, the S-th of its sum; as in gemm_kernel: PARK = stage of k-tile kt+1, STEADY: k-tiles kt+1 and kt+1+NS both exist
  auto k_tile = [&](int kt, auto S_, auto STEADY_) {
    constexpr int s = decltype(S_)::value;
    constexpr std::integral_constant<int, (s + 1) % NS> PARK_{};
    constexpr bool steady = decltype(STEADY_)::value;
    const int buf = kt & 1;
    const unsigned char* as = smem + buf * STAGEB + (wm * WM * 32 + fr) * ROWB + fg * 16;
    const unsigned char* bs = smem + buf * STAGEB + (BM + wn * WN * 32 + fr) * ROWB + fg * 16;
    bf16x8 fa[WM][3], fb[WN][3];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int i = 0; i < WM; ++i) fa[i][p] = *reinterpret_cast<const bf16x8*>(as + i * 32 * ROWB + p * PLANE);
#pragma unroll
      for (int j = 0; j < WN; ++j) fb[j][p] = *reinterpret_cast<const bf16x8*>(bs + j * 32 * ROWB + p * PLANE);
    }
    if (steady || kt + 1 < KT) store_lds(PARK_, buf ^ 1, kt + 1);
    if (steady || kt + 1 + NS < KT) load_global(PARK_, kt + 1 + NS);
    // the small products first
    constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
          sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][pa[t]], fb[j][pb[t]], s == 0 && t == 0 ? floatx16{} : sum[i][j], 0, 0, 0);
    __syncthreads();
  };
  auto add_sum = [&](int kt) {
    const float scale = turned(kt) ? -SPLIT_DOWN : SPLIT_DOWN;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = fmaf(scale, sum[i][j][v], acc[i][j][v]);
  };
  int kt = 0;
  for (; kt + CH + NS < KT; kt += CH) {
    for_stages<0, CH>([&](auto S_) { k_tile(kt + decltype(S_)::value, S_, std::true_type{}); });
    add_sum(kt);
  }
  for (; kt < KT; kt += CH) {
    for_stages<0, CH>([&](auto S_) {
      if (kt + decltype(S_)::value < KT) k_tile(kt + decltype(S_)::value, S_, std::false_type{});
    });
    add_sum(kt);
  }

  for_tiles<0, 0, WM, WN>([&](auto I_, auto J_) {
    constexpr int i = decltype(I_)::value, j = decltype(J_)::value;
    bool again = false;
#pragma unroll
    for (int v = 0; v < 16; ++v) again |= not_finite(acc[i][j][v]);
    if (!__any(again)) return;
    floatx16 plain = {};
    const int off_a = (int)((((int64_t)(wm * WM + i) * 32 + fr) * a.lda + fg * 8) * 4);
    const int off_b = (int)((((int64_t)(wn * WN + j) * 32 + fr) * a.K + fg * 8) * 4);
    for (int k = kt0; k < kt0 + KT; ++k) {
      mma<float>::frag fa, fb;
      fa.lo = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(ra_rsrc, off_a, k * BK * 4, 0));
      fa.hi = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(ra_rsrc, off_a + 16, k * BK * 4, 0));
      fb.lo = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rb_rsrc, off_b, k * BK * 4, 0));
      fb.hi = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rb_rsrc, off_b + 16, k * BK * 4, 0));
      mma<float>::run(plain, fa, fb);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v)
      if (not_finite(acc[i][j][v])) acc[i][j][v] = plain[v];
  });
  void* out = a.splits > 1 ? (void*)(reinterpret_cast<float*>(a.out) + blockIdx.y * a.split_stride) : a.out;
  epilogue<EPI, WAVES_M, WAVES_N, WM, WN>(a, out, acc, smem, m0, n0);
}

// 16-bit operands, 256x256 workgroup tile, 8 wavefronts of 128x64, K step 64, two LDS stages of 64 KiB,
// v_mfma_f32_16x16x32 (under the board's power limit it sustains a higher clock than the 32x32x16 form: 1820 against
// 1570 TFLOP/s in a register-only loop on random float16 data).
//
// The memory pipeline writes the operand tiles straight into LDS (buffer_load_dwordx4 ... lds: 64 lanes x
// 16 bytes land at consecutive LDS addresses), so there are no staging registers and no ds_write.  A tile row is
// 128 bytes = 8 chunks; LDS position (row, c) holds chunk c ^ ((row >> 1) & 7) of the row, which each lane arranges
// by choosing its global address, and which makes the 16-byte fragment reads of 16 consecutive rows hit 16 distinct
// bank groups without padding.  Rows beyond M or N are outside the buffer resource and read as zero.
//
// The two wavefronts of a SIMD (wave w and w + 4) never compete for the matrix pipe: a k-tile is eight clusters,
// memory clusters (fragment reads from LDS, two global->LDS loads, the wait for an older load) alternating with
// MFMA clusters (one quarter of the wavefront's tile: 64 rows x 32 columns x 64 k = 16 MFMAs), every cluster ends
// in a workgroup barrier, and wavefronts 4..7 run one cluster behind wavefronts 0..3, so that at any time four
// wavefronts multiply while the other four read.  Operands are loaded in four sets per k-tile (A rows / W rows
// of the first and second half of every wavefront's tile) in the order the clusters consume them, each set into
// the place of the same set two k-tiles earlier as soon as both groups have read that one; every load is issued
// nine to ten clusters before its first reader.
template <typename T, int EPI>
__global__ __launch_bounds__(512) void gemm_dma_kernel(const gemm_args a) {
  static_assert(sizeof(T) == 2, "16-bit operands");
  constexpr int WAVES_M = 2, WAVES_N = 4, WM = 4, WN = 2, BM = 256, BN = 256, BK = 64;
  constexpr int ROWB = BK * 2, OPB = BM * ROWB, STAGEB = 2 * OPB;
  extern __shared__ __align__(16) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int fr = lane & 15, fq = lane >> 4;

  // tile id: contiguous tile ranges per XCD; the 32 workgroups that an XCD runs at a time form 8 x 4 tiles (row-tiles x
  // column-tiles), or 4 x 8 when the problem has few column-tiles (the out projection: each row panel is then fetched
  // from memory twice instead of four times, the small weight matrix more often; 1.4 % faster there, 0.9 % slower on
  // the input projection)
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
  const int nblk = tiles_m * tiles_n;
  int pid = blockIdx.x;
  {
    const int per = nblk / 8;
    if (pid < per * 8) pid = (pid % 8) * per + pid / 8;
  }
  const int GM = tiles_n <= 16 ? 4 : 8;
  const int group = pid / (GM * tiles_n);
  const int first_m = group * GM;
  const int gsz = (tiles_m - first_m < GM) ? tiles_m - first_m : GM;
  const int tm = first_m + (pid % (GM * tiles_n)) % gsz;
  const int tn = (pid % (GM * tiles_n)) / gsz;
  const int m0 = tm * BM, n0 = tn * BN;

  const int rows_a = (a.M - m0 < BM) ? a.M - m0 : BM, rows_b = (a.N - n0 < BN) ? a.N - n0 : BN;
  const T* tile_a = reinterpret_cast<const T*>(a.A) + (int64_t)m0 * a.lda;
  const T* tile_b = reinterpret_cast<const T*>(a.W) + (int64_t)n0 * a.K;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(tile_a), 0, (int)((((int64_t)rows_a - 1) * a.lda + a.K) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(tile_b), 0, (int)((((int64_t)rows_b - 1) * a.K + a.K) * 2), 0x00020000);

  // a wavefront load = 8 rows x 128 bytes at 1 KiB of consecutive LDS; lane l fetches, for LDS position l % 8 of
  // row l / 8, chunk (l % 8) ^ swizzle(row): every row base used below is a multiple of 8 whose bit 3 is wave & 1
  const int chunk = (lane & 7) ^ ((lane >> 4) & 3) ^ ((wave & 1) << 2);
  const int voff_a = (int)((int64_t)(lane >> 3) * a.lda * 2) + chunk * 16;
  const int voff_b = (int)((int64_t)(lane >> 3) * a.K * 2) + chunk * 16;
  // my two loads of a set: A rows wave*8 and 128 + wave*8 (+64 for the second-half set), W rows
  // (wave/4)*64 + (wave%4)*8 and 128 more (+32 for the second-half set)
  const int ra0 = wave * 8, rb0 = (wave >> 2) * 64 + (wave & 3) * 8;

  // my K range (split-K: blockIdx.y; the whole of K otherwise), in k-tiles
  const int kt0 = (int)((int64_t)blockIdx.y * (a.K / BK) / a.splits);
  const int KT = (int)((int64_t)(blockIdx.y + 1) * (a.K / BK) / a.splits) - kt0;
  // Every operand row of a k-tile lies at the same offset inside its row, and the rows are a power of two apart: when
  // the whole chip walks k in step it asks at any moment for addresses that fall into few memory channels.  With one
  // group of row tiles (a short prompt: every XCD then has its own range of column tiles, and all workgroups run at
  // once) the walk starts an eighth of the k range further on in every eighth of the column tiles and wraps around:
  // the workgroups of an XCD still walk together and share their activation panels through its L2, the XCDs do not.
  // The start depends on the column tile alone.
  const int krot = tiles_m <= 8 ? (int)((((int64_t)tn * 8) / tiles_n) * KT / 8) : 0;

  // set 0: A first half, 1: W first half, 2: W second half, 3: A second half
  auto issue = [&](int st, int kt, auto SET_) {
    constexpr int set = decltype(SET_)::value;
    const int kr = kt + krot;
    const int koff = (kt0 + (kr >= KT ? kr - KT : kr)) * ROWB;
    // a k-tile beyond the range is requested all the same (the wait counts stay the same in every k-tile) but with an
    // offset far outside the buffer: such a load fetches nothing and writes zeros into a stage that is not read again
    const int beyond = kt < KT ? 0 : 0x40000000;
    if constexpr (set == 0 || set == 3) {
      const int r = ra0 + (set == 3 ? 64 : 0);
      unsigned char* d = smem + st * STAGEB + r * ROWB;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr)d, 16, voff_a + beyond, koff + (int)((int64_t)r * a.lda * 2), 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr)(d + 128 * ROWB), 16, voff_a + beyond,
                                               koff + (int)((int64_t)(r + 128) * a.lda * 2), 0, 0);
    } else {
      const int r = rb0 + (set == 2 ? 32 : 0);
      unsigned char* d = smem + st * STAGEB + OPB + r * ROWB;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr)d, 16, voff_b + beyond, koff + (int)((int64_t)r * a.K * 2), 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr)(d + 128 * ROWB), 16, voff_b + beyond,
                                               koff + (int)((int64_t)(r + 128) * a.K * 2), 0, 0);
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;

  floatx4 acc[2 * WM][2 * WN];
#pragma unroll
  for (int i = 0; i < 2 * WM; ++i)
#pragma unroll
    for (int j = 0; j < 2 * WN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  issue(0, 0, I0{}); issue(0, 0, I1{}); issue(0, 0, I2{}); issue(0, 0, I3{});
  issue(1, 1, I0{}); issue(1, 1, I1{});

  // fragments of a 16x16x32 MFMA: lane (fr, fq) supplies elements [8*fq, 8*fq + 8) of the 32-wide k-step of row fr
  int xo[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) xo[ks] = ((4 * ks + fq) ^ ((fr >> 1) & 7)) * 16;
  const int a_row = (wm * 128 + fr) * ROWB, b_row = OPB + (wn * 64 + fr) * ROWB;
  typename mma<T>::frag fa[2 * WM][2], fb[2 * WN][2];
  // read number n = 4*ks + i of A half h (row blocks 4h .. 4h+3), reads [n_lo, n_hi)
  auto read_a = [&](int st, int h, int n_lo, int n_hi) {
#pragma unroll
    for (int n = 0; n < 8; ++n)
      if (n >= n_lo && n < n_hi)
        fa[4 * h + (n & 3)][n >> 2] =
            mma<T>::load(reinterpret_cast<const T*>(smem + st * STAGEB + a_row + (4 * h + (n & 3)) * 16 * ROWB + xo[n >> 2]));
  };
  auto read_b = [&](int st, int h) {
#pragma unroll
    for (int n = 0; n < 4; ++n)
      fb[2 * h + (n & 1)][n >> 1] =
          mma<T>::load(reinterpret_cast<const T*>(smem + st * STAGEB + b_row + (2 * h + (n & 1)) * 16 * ROWB + xo[n >> 1]));
  };
  // 64 rows (A half ha) x 32 columns (W half hb) x 64: the two MFMAs of an accumulator are 8 instructions apart
  auto multiply = [&](auto HA_, auto HB_) {
    constexpr int ha = decltype(HA_)::value, hb = decltype(HB_)::value;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) mma<T>::run16(acc[4 * ha + i][2 * hb + j], fb[2 * hb + j][ks], fa[4 * ha + i][ks]);
    __builtin_amdgcn_s_setprio(0);
  };
  // end of a memory cluster: the set that the next memory cluster reads was issued four sets ago
  auto landed = [&]() { __builtin_amdgcn_s_waitcnt(wait_vmcnt(8)); };
  auto cluster_end = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  landed();
  __builtin_amdgcn_s_barrier();
  if (wm) __builtin_amdgcn_s_barrier();        // wavefronts 4..7 start one cluster late
  __builtin_amdgcn_sched_barrier(0);
  read_a(0, 0, 0, 6);

  // k-tile kt in stage st; fragment reads per memory cluster: 6 + 6 + 4 + 8
  auto k_tile = [&](int kt, auto ST_) {
    constexpr int st = decltype(ST_)::value;
    read_a(st, 0, 6, 8);
    read_b(st, 0);
    issue(st ^ 1, kt + 1, I2{});
    landed();
    cluster_end();
    multiply(I0{}, I0{});
    cluster_end();
    read_b(st, 1);
    issue(st ^ 1, kt + 1, I3{});
    landed();
    cluster_end();
    multiply(I0{}, I1{});
    cluster_end();
    read_a(st, 1, 0, 8);
    issue(st, kt + 2, I0{});
    landed();
    cluster_end();
    multiply(I1{}, I0{});
    cluster_end();
    read_a(st ^ 1, 0, 0, 6);                   // of k-tile kt+1
    issue(st, kt + 2, I1{});
    landed();
    cluster_end();
    multiply(I1{}, I1{});
    cluster_end();
  };
  int kt = 0;
  for (; kt + 1 < KT; kt += 2) {
    k_tile(kt, I0{});
    k_tile(kt + 1, I1{});
  }
  if (kt < KT) k_tile(kt, I0{});
  __builtin_amdgcn_s_waitcnt(wait_vmcnt(0));   // the surplus loads land before this workgroup's LDS is given away
  if (!wm) __builtin_amdgcn_s_barrier();
  __syncthreads();                             // every wavefront's loads have landed: the epilogue may reuse the stages

  void* out = a.splits > 1 ? (void*)(reinterpret_cast<float*>(a.out) + blockIdx.y * a.split_stride) : a.out;
  epilogue<EPI, WAVES_M, WAVES_N, WM, WN, true>(a, out, acc, smem, m0, n0);
}

// 16-bit operands, up to 256 rows (a short prompt, a few scored continuations) or K ranges of a few rows: bound by the
// weights, which come from memory once, and by the operand path into LDS.  Row tiles of BM rows - normally ONE, so that no
// weight is read twice -, BN = 128 columns per workgroup, 8 wavefronts, K step 64, S LDS stages written by the memory
// pipeline as in gemm_dma_kernel (same row layout and swizzle): S - 1 k-tiles in flight without a register for them.
//
// Per k-tile there is one workgroup barrier.  Before it a wavefront waits for its own loads of the next k-tile and its own
// fragment reads of this one, so behind it every operand of the next k-tile is in LDS and this k-tile's stage is free.
// The fragments of a k-step are read while the MFMAs of the k-step before run, and the loads of k-tile kt+S are spread
// over the MFMAs of two k-steps: issued in one burst (6 loads of 1 KiB per wavefront, which a CU accepts in ~800 cycles)
// they held the MFMAs behind them up and cost 5 %.
//
// Measured at the 6B shapes (input projection N = 28672, K = 4096 / out projection N = 4096, K = 20480 in 8 ranges with
// its reduce; weights of six layers in rotation) against the register-staged tiles this replaced: M = 64 40.3 / 37.1 us
// (43.2 / 42.2 with 64 x 128 tiles), M = 128 51 / 45 (62 / 58), M = 256 70 / 57 (93 / 82, 128 x 128 tiles); M = 32 with K
// ranges 34.1 (37.2).  The loads alone take 48 (M = 128) and 60 us (M = 256) for the input projection, the MFMAs and
// fragment reads alone 23 and 43.  Counters at 61 / 128 / 244 rows (40 / 49 / 64 us with a plain store): every weight comes from
// memory once (5.9 / 5.0 / 3.9 TB/s), 347 / 470 / 683 MB go through L2 into LDS (8.6 / 9.6 / 10.6 TB/s), the matrix units of the
// CUs in use are busy 16 / 28 / 45 % of the time, no bank conflicts: few rows are bound by the weight stream, many by the
// path into LDS, and neither more stages nor another walk over k changes it.
template <typename T, int EPI, int BM, int S>
__global__ __launch_bounds__(512) void gemm_stream_kernel(const gemm_args a) {
  static_assert(sizeof(T) == 2, "16-bit operands");
  constexpr int BN = 128, BK = 64, ROWB = BK * 2;
  constexpr int WAVES_M = BM == 64 ? 2 : 4, WAVES_N = 8 / WAVES_M, WM = BM / 32 / WAVES_M, WN = BN / 32 / WAVES_N;
  constexpr int OPB = BM * ROWB, STAGEB = OPB + BN * ROWB;
  constexpr int NW = BN / 64, NL = NW + BM / 64;                     // loads per wavefront and k-tile: of W, in all
  extern __shared__ __align__(16) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  const int fr = lane & 15, fq = lane >> 4;

  // workgroups are dealt round-robin over the XCDs: with a multiple of 8 K ranges an XCD sees one or two of them and
  // keeps that part of the activations in its L2 for all column tiles; without a split the row tiles of a column tile
  // follow each other at a distance of 8, on one XCD, whose L2 then reads each weight once
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
  const int y = blockIdx.x % a.splits, t = blockIdx.x / a.splits;
  const int first_n = t / (8 * tiles_m) * 8, tl = t - first_n * tiles_m;
  const int gs = tiles_n - first_n < 8 ? tiles_n - first_n : 8;
  const int tm = tl / gs, tn = first_n + tl - tm * gs;
  const int m0 = tm * BM, n0 = tn * BN;
  const int rows_a = (a.M - m0 < BM) ? a.M - m0 : BM, rows_b = (a.N - n0 < BN) ? a.N - n0 : BN;
  const T* tile_a = reinterpret_cast<const T*>(a.A) + (int64_t)m0 * a.lda;
  const T* tile_b = reinterpret_cast<const T*>(a.W) + (int64_t)n0 * a.K;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(tile_a), 0, (int)((((int64_t)rows_a - 1) * a.lda + a.K) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(tile_b), 0, (int)((((int64_t)rows_b - 1) * a.K + a.K) * 2), 0x00020000);

  const int chunk = (lane & 7) ^ ((lane >> 4) & 3) ^ ((wave & 1) << 2);
  const int row = wave * 8 + (lane >> 3);
  const int voff_a = (int)((int64_t)row * a.lda * 2) + chunk * 16;
  const int voff_b = (int)((int64_t)row * a.K * 2) + chunk * 16;

  const int kt0 = (int)((int64_t)y * (a.K / BK) / a.splits);
  const int KT = (int)((int64_t)(y + 1) * (a.K / BK) / a.splits) - kt0;
  const int krot = (int)(((unsigned)tn * 5u) % (unsigned)KT);        // see gemm_kernel
  // load n of k-tile kt into stage st: W rows first, then A rows, 64 rows each
  auto issue_one = [&](int st, int kt, auto N_) {
    constexpr int n = decltype(N_)::value;
    const int kr = kt + krot;
    const int koff = (kt0 + (kr >= KT ? kr - KT : kr)) * ROWB;
    const int beyond = kt < KT ? 0 : 0x40000000;                     // see gemm_dma_kernel
    unsigned char* d = smem + st * STAGEB + wave * 8 * ROWB;
    if constexpr (n < NW)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr)(d + OPB + n * 64 * ROWB), 16, voff_b + beyond,
                                               koff + (int)((int64_t)n * 64 * a.K * 2), 0, 2);   // nt: streamed once
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr)(d + (n - NW) * 64 * ROWB), 16, voff_a + beyond,
                                               koff + (int)((int64_t)(n - NW) * 64 * a.lda * 2), 0, 0);
  };

  floatx4 acc[2 * WM][2 * WN];
#pragma unroll
  for (int i = 0; i < 2 * WM; ++i)
#pragma unroll
    for (int j = 0; j < 2 * WN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int st = 0; st < S - 1; ++st) for_stages<0, NL>([&](auto N_) { issue_one(st, st, N_); });

  int xo[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) xo[ks] = ((4 * ks + fq) ^ ((fr >> 1) & 7)) * 16;
  const int a_row = (wm * WM * 32 + fr) * ROWB, b_row = OPB + (wn * WN * 32 + fr) * ROWB;

  typename mma<T>::frag fa[2][2 * WM], fb[2][2 * WN];
  auto read = [&](int st, auto KS_) {
    constexpr int ks = decltype(KS_)::value;
    const unsigned char* sb = smem + st * STAGEB;
#pragma unroll
    for (int j = 0; j < 2 * WN; ++j) fb[ks][j] = mma<T>::load(reinterpret_cast<const T*>(sb + b_row + j * 16 * ROWB + xo[ks]));
#pragma unroll
    for (int i = 0; i < 2 * WM; ++i) fa[ks][i] = mma<T>::load(reinterpret_cast<const T*>(sb + a_row + i * 16 * ROWB + xo[ks]));
  };
  // the MFMAs of one k-step with the loads [N0, N1) of k-tile kt between them
  auto multiply = [&](auto KS_, auto N0_, auto N1_, int st, int kt) {
    constexpr int ks = decltype(KS_)::value, n0_ = decltype(N0_)::value, n1_ = decltype(N1_)::value;
    for_stages<0, 2 * WM>([&](auto I_) {
      constexpr int i = decltype(I_)::value;
      if constexpr (n0_ + i < n1_) {
        issue_one(st, kt, std::integral_constant<int, n0_ + i>{});
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < 2 * WN; ++j) mma<T>::run16(acc[i][j], fb[ks][j], fa[ks][i]);
      __builtin_amdgcn_sched_barrier(0);
    });
    for_stages<0, NL>([&](auto N_) {             // more loads than rows of blocks
      constexpr int n = decltype(N_)::value;
      if constexpr (n >= n0_ + 2 * WM && n < n1_) issue_one(st, kt, N_);
    });
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using IH = std::integral_constant<int, NL / 2>;
  using IL = std::integral_constant<int, NL>;
  // my loads of the next k-tile have landed, and so have my fragment reads of this one; behind the barrier both hold
  // for the whole workgroup
  auto next_tile = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(wait_vmcnt((S - 2) * NL) & wait_lgkmcnt(0));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  next_tile();
  for_stages<0, NL / 2>([&](auto N_) { issue_one(S - 1, S - 1, N_); });
  read(0, I0{});
  int st = 0;
  for (int kt = 0; kt < KT; ++kt) {
    const int nx = st + 1 == S ? 0 : st + 1;
    read(st, I1{});
    __builtin_amdgcn_sched_barrier(0);
    multiply(I0{}, IH{}, IL{}, st == 0 ? S - 1 : st - 1, kt + S - 1);   // second half of the loads of k-tile kt+S-1
    next_tile();
    read(nx, I0{});                            // beyond the last k-tile: zeros that nothing multiplies
    __builtin_amdgcn_sched_barrier(0);
    multiply(I1{}, I0{}, IH{}, st, kt + S);    // first half of those of k-tile kt+S
    st = nx;
  }
  __builtin_amdgcn_s_waitcnt(wait_vmcnt(0));   // the surplus loads land before the stages are reused
  __syncthreads();

  void* out = a.splits > 1 ? (void*)(reinterpret_cast<float*>(a.out) + y * a.split_stride) : a.out;
  epilogue<EPI, WAVES_M, WAVES_N, WM, WN, true>(a, out, acc, smem, m0, n0);
}

template <typename T, int EPI, int BM, int S>
int launch_stream(const gemm_args& a, hipStream_t s) {
  constexpr size_t lds = (size_t)S * (BM + 128) * 128;
  static_assert(lds >= 3 * BM * sizeof(int) + 8 * 32 * 36 * sizeof(float), "epilogue scratch does not fit");
  static mtj_device_once once;
  if (int rc = mtj_allow_lds(once, "mtj_gemm", &gemm_stream_kernel<T, EPI, BM, S>, lds)) return rc;
  gemm_stream_kernel<T, EPI, BM, S><<<(unsigned)((a.M + BM - 1) / BM * ((a.N + 127) / 128) * a.splits), 512, lds, s>>>(a);
  return mtj_check_launch("mtj_gemm");
}

template <typename T, int EPI>
int launch_dma(const gemm_args& a, hipStream_t s) {
  constexpr size_t lds = 2 * 2 * 256 * 64 * 2;
  static mtj_device_once once;
  if (int rc = mtj_allow_lds(once, "mtj_gemm", &gemm_dma_kernel<T, EPI>, lds)) return rc;
  const int tiles = ((a.M + 255) / 256) * ((a.N + 255) / 256);
  gemm_dma_kernel<T, EPI><<<dim3(tiles, a.splits), 512, lds, s>>>(a);
  return mtj_check_launch("mtj_gemm");
}

template <typename T, int EPI, int WAVES_M, int WAVES_N, int WM, int WN, int BK, int NS>
int launch(const gemm_args& a, hipStream_t s) {
  constexpr int BM = WAVES_M * WM * 32, BN = WAVES_N * WN * 32;
  constexpr size_t lds = 2 * (size_t)(BM + BN) * (BK + mma<T>::EPC) * sizeof(T);
  static_assert(lds <= 160 * 1024, "tile does not fit LDS");
  static_assert(lds >= 3 * BM * sizeof(int) + WAVES_M * WAVES_N * 32 * 36 * sizeof(float), "epilogue scratch does not fit");
  static mtj_device_once once;
  if (int rc = mtj_allow_lds(once, "mtj_gemm", &gemm_kernel<T, EPI, WAVES_M, WAVES_N, WM, WN, BK, NS>, lds)) return rc;
  const int tiles = ((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  gemm_kernel<T, EPI, WAVES_M, WAVES_N, WM, WN, BK, NS><<<dim3(tiles, a.splits), WAVES_M * WAVES_N * 64, lds, s>>>(a);
  return mtj_check_launch("mtj_gemm");
}

template <int EPI, int WAVES_M, int WAVES_N, int WM, int WN, int NS>
int launch_split(const gemm_args& a, hipStream_t s) {
  constexpr int BM = WAVES_M * WM * 32, BN = WAVES_N * WN * 32;
  constexpr size_t stages = 2 * (size_t)(BM + BN) * 112, patches = 3 * BM * sizeof(int) + WAVES_M * WAVES_N * 32 * 36 * sizeof(float);
  constexpr size_t lds = stages > patches ? stages : patches;
  static_assert(lds <= 160 * 1024, "tile does not fit LDS");
  static mtj_device_once once;
  if (int rc = mtj_allow_lds(once, "mtj_gemm", &gemm_split_kernel<EPI, WAVES_M, WAVES_N, WM, WN, NS>, lds)) return rc;
  const int tiles = ((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  gemm_split_kernel<EPI, WAVES_M, WAVES_N, WM, WN, NS><<<dim3(tiles, a.splits), WAVES_M * WAVES_N * 64, lds, s>>>(a);
  return mtj_check_launch("mtj_gemm");
}

// 256 x 256 tiles of gemm_dma_kernel, one workgroup per CU, from this many of them on: N = 4096, K = 20480 in one K range,
// 144 tiles 486 us (602 with 128 x 128 tiles), 192 tiles 458 (650); 96 tiles 455 against 384 for two ranges of 128 x 128.
// So are 144 .. 196 tiles with the other epilogues, us against 128 x 128 tiles, at every K from 256 on: STORE 144 tiles 19 (33) at
// K = 256, 31 (53) at 1024, 49 (80) at 2048; XENT the same; the fused input projection 61 (70) for 513 rows of d_model 2048, 43
// (49) for 1536 of 1024, 36.4 (37.5) for 1742 of 768.  Its epilogue is long, so with fewer than 12 k-tiles in front of it several
// small workgroups per CU hide it better: d_model 512, 2766 / 3022 / 3278 rows (154 / 168 / 182 tiles) 32 - 33 us (28 - 30),
// 3534 rows (196) 33 (34); that epilogue keeps a line of 200 tiles there.
constexpr int64_t DMA_MIN_TILES = 144;
constexpr int64_t DMA_MIN_TILES_SHORT_INPROJ = 200;
int64_t dma_tiles(int64_t M, int64_t N) { return ((M + 255) / 256) * ((N + 255) / 256); }

template <typename T, int EPI, int BK>
int dispatch_tile(const gemm_args& a, hipStream_t s) {
  if constexpr (sizeof(T) == 2) {
    // 32 x 128 tiles, up to three workgroups per CU: batched decode without a split.  Against the stream kernel at M = 8:
    // 38.4 / 39.2 us for the input projection, 66.7 / 67.9 for 50400 logits (two rounds of one workgroup per CU); with K
    // ranges (the out projection) the stream kernel's deeper queue wins, 32.8 against 34.5 us.
    if (a.M <= 32 && a.splits == 1) return launch<T, EPI, 1, 4, 1, 1, BK, 2>(a, s);
    // 33 .. 64 rows of more than one round of column tiles with a short K: 64 x 128 tiles of the same kernel, two or three
    // workgroups per CU against one.  50400 columns, 33 / 48 / 64 rows: K = 512 16.8 / 18.6 / 19.4 us (stream kernel 18.2 / 18.8 /
    // 19.3), K = 1024 26.7 / 28.8 / 31.1 (28.6 / 29.1 / 29.8), K = 2048 46.5 / 48.0 / 52.0 (48.6 / 51.9 / 52.6); at K = 4096, 81.1 /
    // 86.4 / 89.8 (83.8 / 85.6 / 88.9), and with one round, 16384 columns at K = 1024, 16.5 / 17.8 / 17.7 (13.7 / 15.0 / 13.4)
    // the stream kernel's queue is the better one.  So it is for XENT (K = 512, with the merge 24 us against 32).
    if constexpr (EPI != MTJ_EPI_XENT)
      if (a.M <= 64 && a.splits == 1 && a.K < 4096 && (a.N + 127) / 128 > 256) return launch<T, EPI, 1, 4, 2, 1, BK, 2>(a, s);
    if (a.M <= 64) return launch_stream<T, EPI, 64, 4>(a, s);
    // 129 .. 256 rows: one row tile while that fills more than half of the chip, else two (at d_model 2048, 112 column
    // tiles, M = 256: 28 us in two row tiles, 38 in one; at d_model 4096 the second one would only read the weights again)
    if (a.M > 128 && a.M <= 256 && (a.N + 127) / 128 * a.splits > 128) return launch_stream<T, EPI, 256, 3>(a, s);
    if (a.M <= 256) return launch_stream<T, EPI, 128, 4>(a, s);
  } else {
    if (a.M <= 32) return launch<T, EPI, 1, 4, 1, 1, BK, 2>(a, s);  // 32 x 128: the weights stream once
    // The largest tile that fills most of the chip, two workgroups per CU.  us with 128 x 128 / 64 x 128 / 64 x 64 tiles:
    // N = 28672, K = 4096 64 rows 215 / 149 / 174, 100 rows 221 / 215 / 309; N = 3584, K = 512 60 rows 38 / 25 / 22, 127 rows
    // 38 / 25 / 22, 300 38 / 25 / 26, 500 38 / 26 / 27, 1000 40 / 36 / 45; N = 512, K = 2560 127 rows 45 / 31 / 27, 500
    // 47 / 32 / 29, 2000 53 / 49 / 60; N = 4096, K = 20480 64 rows in eight ranges 155 / 100 / 122, 100 145 / 162 / 215.
    // (33 .. 64 rows took 157, 25 and 111 of these on v_mfma_f32_32x32x2_f32.)  The statistics of XENT are per 128 columns.
    // Tiles of 64 rows take a sixth longer for a row (199 rows 409 against 349) and win where they leave out more than that:
    // 64 rows above, 129 (321 against 288).
    const int64_t rows64 = (a.M + 63) / 64, rows128 = (a.M + 127) / 128, cols128 = (a.N + 127) / 128;
    if (rows128 * cols128 * a.splits >= 200 && 6 * 2 * rows128 <= 7 * rows64) return launch_split<EPI, 2, 2, 2, 2, 3>(a, s);
    if constexpr (EPI == MTJ_EPI_XENT) return launch_split<EPI, 2, 2, 1, 2, 2>(a, s);
    else return rows64 * cols128 * a.splits >= 200 ? launch_split<EPI, 2, 2, 1, 2, 2>(a, s) : launch_split<EPI, 2, 2, 1, 1, 3>(a, s);
  }
  if constexpr (sizeof(T) == 2) {
    // e.g. M = 16384, N = 28672 or N = 4096 (a whole 6B layer at 8 x 2048 tokens): 7168 / 1024 tiles
    const int64_t line = EPI == MTJ_EPI_INPROJ && a.K < 768 ? DMA_MIN_TILES_SHORT_INPROJ : DMA_MIN_TILES;
    if (dma_tiles(a.M, a.N) * a.splits >= line) return launch_dma<T, EPI>(a, s);        // 256 x 256, 8 wavefronts of 128 x 64
    return launch<T, EPI, 2, 2, 2, 2, BK, 2>(a, s);                 // 128 x 128
  }
}

template <typename T, int BK>
int dispatch(const gemm_args& a, int epi, hipStream_t s) {
  if (epi == MTJ_EPI_STORE) return dispatch_tile<T, MTJ_EPI_STORE, BK>(a, s);
  if (epi == MTJ_EPI_RESID) return dispatch_tile<T, MTJ_EPI_RESID, BK>(a, s);
  if (epi == MTJ_EPI_XENT) return dispatch_tile<T, MTJ_EPI_XENT, BK>(a, s);
  return dispatch_tile<T, MTJ_EPI_INPROJ, BK>(a, s);
}

// p[0] + p[stride] + .. + p[(splits - 1) * stride] in this order, four columns.  The loads of up to eight partials are all
// issued before the first is added: a loop that asks for one partial per turn pays the latency of memory `splits` times,
// which for a few rows is most of the launch (product, eight ranges and reduce with LayerNorm, N = 4096, K = 20480: 3 rows
// 36.7 -> 34.7 us, 244 rows 63.5 -> 61.7; 40 rows of N = 1024, K = 5120 15.0 -> 11.7).
template <int C> __device__ __forceinline__ void add_partials(floatx4& acc, const float* __restrict__ p, int64_t stride) {
  floatx4 t[C];
#pragma unroll
  for (int i = 0; i < C; ++i) t[i] = *reinterpret_cast<const floatx4*>(p + i * stride);
#pragma unroll
  for (int i = 0; i < C; ++i) { acc.x += t[i].x; acc.y += t[i].y; acc.z += t[i].z; acc.w += t[i].w; }
}
// C: loads in flight.
template <int C = 8> __device__ __forceinline__ floatx4 sum_partials(const float* __restrict__ p, int splits, int64_t stride) {
  floatx4 acc = *reinterpret_cast<const floatx4*>(p);
  p += stride;
  int left = splits - 1;
  for (; left >= C; left -= C, p += C * stride) add_partials<C>(acc, p, stride);
  for_stages<1, C>([&](auto N_) {
    if (left == decltype(N_)::value) add_partials<decltype(N_)::value>(acc, p, stride);
  });
  return acc;
}

// sums the per-split partial tiles in a fixed order and applies the epilogue (four columns per thread)
template <int EPI>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ work, int splits, int64_t split_stride,
                                                            int M, int N, const float* __restrict__ bias, void* out,
                                                            int64_t ldo, int out_dtype) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;     // quad index over [M, N / 4]
  const int nq = N / 4;
  if (q >= (int64_t)M * nq) return;
  const int m = (int)(q / nq), n = (int)(q - (int64_t)m * nq) * 4;
  floatx4 acc = sum_partials(work + (int64_t)m * N + n, splits, split_stride);
  if (bias) {
    const floatx4 b = *reinterpret_cast<const floatx4*>(bias + n);
    acc.x += b.x; acc.y += b.y; acc.z += b.z; acc.w += b.w;
  }
  const int64_t idx = (int64_t)m * ldo + n;
  if (EPI == MTJ_EPI_RESID) {
    float* o = reinterpret_cast<float*>(out) + idx;
    o[0] += acc.x; o[1] += acc.y; o[2] += acc.z; o[3] += acc.w;
  } else if (out_dtype == MTJ_F32) {
    float* o = reinterpret_cast<float*>(out) + idx;
    o[0] = acc.x; o[1] = acc.y; o[2] = acc.z; o[3] = acc.w;
  } else {
    uint32x2 pk;
    pk.x = pack_16x2(acc.x, acc.y, out_dtype);
    pk.y = pack_16x2(acc.z, acc.w, out_dtype);
    *reinterpret_cast<uint32x2*>(reinterpret_cast<uint16_t*>(out) + idx) = pk;
  }
}

// The RESID reduce of one whole row per workgroup, followed by the LayerNorm of the row it has just completed
// (ReplicatedLayerNorm, layers.py:17-36, of the NEXT layer or of the projection): x += sum of partials + bias, then
// h = scale * (x - mean) * rsqrt(var + 1e-5) + offset in h_dtype.  Saves the LayerNorm launch and its round trip
// through memory between two decode layers.  N <= 4 * RLN_Q * 1024.
// One thread per four columns up to 4096 columns: rows of a narrow model do not wait for idle wavefronts (N = 512, two
// ranges, with the product: 8000 rows 85 us with 1024 threads per row, 53 with 128, 60 with a separate LayerNorm; N = 4096
// as before).  The sums of idle wavefronts were zeros, so the results are the same bits.
// Q quads per thread, one up to 4096 columns.  Two workgroups of 1024 threads per CU need 64 registers or less, and while one
// waits at a barrier the other loads: with 80, N = 4096 in eight ranges, 511 / 700 / 1500 rows took 19.7 / 19.5 / 29.2 us, now
// 15.3 / 14.7 / 20.9 (17.2 / 17.8 / 23.2 with one partial load at a time and 44 registers).
constexpr int RLN_Q = 4;
template <int Q>
__global__ __launch_bounds__(1024, 8) void splitk_reduce_ln_kernel(const float* __restrict__ work, int splits,
                                                                int64_t split_stride, int N, const float* __restrict__ bias,
                                                                float* __restrict__ x, int64_t ldx,
                                                                const float* __restrict__ ln_scale,
                                                                const float* __restrict__ ln_offset, void* __restrict__ h,
                                                                int64_t ldh, int h_dtype) {
  __shared__ float red[2][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = blockIdx.x, nq = N / 4, NT = blockDim.x, NW = NT / 64;
  floatx4 v[Q], sc, of;
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const int q = i * NT + tid;
    if (q < nq) {
      const int n = q * 4;
      float* o = x + (int64_t)m * ldx + n;
      const floatx4 old = *reinterpret_cast<const floatx4*>(o);
      const floatx4 b = bias ? *reinterpret_cast<const floatx4*>(bias + n) : floatx4{0.f, 0.f, 0.f, 0.f};
      if (Q == 1) {                            // needed last, asked for with everything else
        sc = *reinterpret_cast<const floatx4*>(ln_scale + n);
        of = *reinterpret_cast<const floatx4*>(ln_offset + n);
      }
      floatx4 acc = sum_partials<Q == 1 ? 8 : 4>(work + (int64_t)m * N + n, splits, split_stride);
      if (bias) { acc.x += b.x; acc.y += b.y; acc.z += b.z; acc.w += b.w; }
      // the same two roundings per element as "o[j] += acc.j" of the plain reduce
      acc.x = old.x + acc.x; acc.y = old.y + acc.y; acc.z = old.z + acc.z; acc.w = old.w + acc.w;
      *reinterpret_cast<floatx4*>(o) = acc;
      v[i] = acc;
      sum += (acc.x + acc.y) + (acc.z + acc.w);
    }
  }
  sum = wave_sum(sum);
  if (lane == 0) red[0][wave] = sum;
  __syncthreads();
  float tot = 0.f;
  for (int i = 0; i < NW; ++i) tot += red[0][i];
  const float mean = tot / (float)N;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    if (i * NT + tid < nq) {
      const floatx4 t = v[i] - mean;
      sq += (t.x * t.x + t.y * t.y) + (t.z * t.z + t.w * t.w);
    }
  }
  sq = wave_sum(sq);
  if (lane == 0) red[1][wave] = sq;
  __syncthreads();
  float var = 0.f;
  for (int i = 0; i < NW; ++i) var += red[1][i];
  const float inv = rsqrtf(var / (float)N + 1e-5f);
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const int q = i * NT + tid;
    if (q < nq) {
      const int n = q * 4;
      if (Q > 1) {
        sc = *reinterpret_cast<const floatx4*>(ln_scale + n);
        of = *reinterpret_cast<const floatx4*>(ln_offset + n);
      }
      const floatx4 y = (sc * inv) * (v[i] - mean) + of;
      if (h_dtype == MTJ_F32) {
        *reinterpret_cast<floatx4*>(reinterpret_cast<float*>(h) + (int64_t)m * ldh + n) = y;
      } else {
        uint32x2 pk;
        pk.x = pack_16x2(y.x, y.y, h_dtype);
        pk.y = pack_16x2(y.z, y.w, h_dtype);
        *reinterpret_cast<uint32x2*>(reinterpret_cast<uint16_t*>(h) + (int64_t)m * ldh + n) = pk;
      }
    }
  }
}

unsigned rln_threads(int64_t N) { return N >= 4096 ? 1024u : (unsigned)((N + 255) / 256 * 64); }

// Second half of the fused logits + cross entropy: merges the per-column-tile statistics of a row.
// loss = log(sum exp(l - max)) - (l[target] - max), correct = (l[target] == max); a target outside [0, N) selects
// nothing (pred = 0), as in xent_kernel.
// Eight rows per workgroup, 32 threads per row that share its column tiles (394 of 128 columns, 197 of 256 at the 6B
// vocabulary): the maximum over all tiles first, then the sum relative to it, each met in LDS.  With one thread per row the
// chain of dependent loads over all tiles took 180 us for 244 rows and kept one workgroup busy; now 6.5 us.
// A row without a maximum (all logits -inf or NaN) sums exp(-inf - -inf) and gives NaN.
constexpr int XM_ROWS = 8, XM_LANES = 32;
__global__ __launch_bounds__(XM_ROWS * XM_LANES) void xent_merge_kernel(const float* __restrict__ pmax, const float* __restrict__ psum,
                                                         const float* __restrict__ tlogit, const int32_t* __restrict__ target,
                                                         int M, int N, int tiles_n, float* __restrict__ loss,
                                                         uint8_t* __restrict__ correct) {
  __shared__ float part[XM_LANES][XM_ROWS];
  const int r = threadIdx.x % XM_ROWS, l = threadIdx.x / XM_ROWS;
  const int m = blockIdx.x * XM_ROWS + r;
  // all 32 partial results of a row, combined in the same order by every thread
  auto meet = [&](float v, auto combine) {
    __syncthreads();
    part[l][r] = v;
    __syncthreads();
    v = part[0][r];
#pragma unroll
    for (int i = 1; i < XM_LANES; ++i) v = combine(v, part[i][r]);
    return v;
  };
  float mx = -INFINITY, sm = 0.f;
  if (m < M)
#pragma unroll 8
    for (int t = l; t < tiles_n; t += XM_LANES) mx = fmaxf(mx, pmax[(int64_t)t * M + m]);
  mx = meet(mx, [](float a, float b) { return fmaxf(a, b); });
  if (m < M)
#pragma unroll 8
    for (int t = l; t < tiles_n; t += XM_LANES) sm += __expf(pmax[(int64_t)t * M + m] - mx) * psum[(int64_t)t * M + m];
  sm = meet(sm, [](float a, float b) { return a + b; });
  if (l > 0 || m >= M) return;
  const int tg = target[m];
  const float pred = ((uint32_t)tg < (uint32_t)N) ? tlogit[m] - mx : 0.f;
  loss[m] = logf(sm) - pred;
  if (correct) correct[m] = (pred == 0.f) ? 1 : 0;
}

// column-tile width that dispatch_tile will use for this problem
int xent_tile_n(int64_t M, int64_t N, int dtype) {
  if (M > 256 && dtype != MTJ_F32 && dma_tiles(M, N) >= DMA_MIN_TILES) return 256;
  return 128;
}

// Time of `tiles` 256 x 256 tiles in s K ranges each, in tenths of the time of one k-tile: rounds of 256 workgroups, each
// walking kt / s k-tiles, and 1.2 tenths for every partial tile that is written and read back.  Measured: a k-tile takes
// 1.3 .. 1.7 us once 100 .. 256 workgroups run, and 256 tiles of N = 4096, K = 20480 in 1 / 2 / 4 / 8 ranges take 545 / 575 /
// 646 / 815 us, 0.06 / 0.10 / 0.13 us per partial tile.  The weight lies above that (0.16 .. 0.2 us) because a range more also
// costs workspace: with 0.9 tenths 192 tiles get 4 ranges and 180 MiB instead of one range, 452 us against 461, and over 178
// products of N = 512 .. 4096 the choices are 0.6 % faster on average, single ones up to 10 % slower (7552 rows of N = 512,
// K = 4096 55 -> 60 us) or faster (1000 rows of N = 2048, K = 10240, 8 ranges instead of 7: 64.7 -> 61.0).
int64_t dma_cost(int64_t tiles, int64_t kt, int64_t s) {
  return (tiles * s + 255) / 256 * ((kt + s - 1) / s) * 10 + (s > 1 ? tiles * s * 6 / 5 : 0);
}

// Rows of a fused input projection that run on 256 x 256 tiles when the rest, the rows of its last row of tiles, is better
// off as a launch of its own: where that row of tiles starts a round of workgroups of which most CUs have nothing (1.6 us a
// k-tile), and the rest streams the weights once more in less (gemm_stream_kernel: 5.9, 4.8 and 3.6 TB/s for up to 64, 128 and
// 256 rows, 4 us for the launch).  0: one launch.  d_model 4096, 580 / 700 rows 194 / 195 -> 152 / 171 us, 1030 / 1270 279 /
// 297 -> 248 / 276, 2935 606 -> 579, 3400 725 -> 678, 5700 (10 rounds) 1147 -> 1100; d_model 2048, 1085 rows 107 -> 82; 1024, 2420
// rows 73 -> 63; 512, 4730 rows 53 -> 48.
// The rounds of one launch drift apart, the sooner the shorter K is against the epilogue, and a round more then costs little,
// while two launches wait for each other.  So there is a limit of whole rounds in front, by K, from six sizes per round and
// d_model 512, 768, 1024, 1536, 2048, 3072 and 4096: from 4096 on 10 (11: 6590 rows 1236 against 1262), from 1024 on 6 (beyond,
// it wins and loses: 1024 16500 281 against 290, 18750 323 -> 308; 1536 12400 409 -> 403, 15500 519 against 535; 2048 8350 454
// against 462, 11600 624 -> 604; 3072 5510 647 against 657, 7000 830 -> 790), from 768 on 3 (4 .. 11: 15440 176 against 180,
// 34340 358 against 377), below 1 (2: 512 9240 68 against 77, 3: 13930 93 against 103).
int64_t inproj_front(int64_t M, int64_t N, int64_t K) {
  const int64_t front = (M - 1) / 256 * 256, rest = M - front;
  if (dma_tiles(front, N) < (K < 768 ? DMA_MIN_TILES_SHORT_INPROJ : DMA_MIN_TILES)) return 0;
  const int64_t whole = (dma_tiles(front, N) + 255) / 256, rounds = (dma_tiles(M, N) + 255) / 256 - whole;
  if (whole > (K >= 4096 ? 10 : K >= 1024 ? 6 : K >= 768 ? 3 : 1)) return 0;
  const double rate = rest <= 64 ? 5.9e6 : rest <= 128 ? 4.8e6 : 3.6e6;                  // bytes per us
  return (double)rounds * (double)(K / 64) * 1.6 > (double)N * (double)K * 2 / rate + 4.0 ? front : 0;
}

// How a problem is cut so that its output tiles fill the chip evenly: rows [0, front) in one K range with the epilogue of
// the product itself, the rows behind them in `splits` K ranges with a reduce.
struct cut_t { int64_t front; int splits; };

// `most`: ranges of more than 64 rows of float32 (see the end)
cut_t pick_cut(int64_t M, int64_t N, int64_t K, int dtype, int most = 4) {
  if (N % 4) return {0, 1};
  const int bk = dtype == MTJ_F32 ? 32 : 64;
  const int64_t kt = K / bk;
  int splits = 1;
  if (M <= (dtype == MTJ_F32 ? 64 : 256)) {   // one row of tiles, 128 columns each: up to 16 ranges
    const int64_t tiles = (N + 127) / 128;
    while (splits < 16 && tiles * splits * 2 <= 256 && kt % (splits * 2) == 0 && kt / (splits * 2) >= 4) splits *= 2;
    return {0, splits};
  }
  if (dtype != MTJ_F32) {
    // 256 x 256 tiles of the direct-to-LDS kernel, one workgroup per CU.  A short prompt's out projection (N = 4096,
    // 16 column tiles) has fewer tiles than CUs: the number of ranges that costs least.  With powers of two only, what did
    // not come to 200 tiles ran on 128 x 128 ones: 768 rows 207 -> 149 us, 1025 338 -> 198, 1536 384 -> 279, 2304
    // 602 -> 388, 2875 650 -> 461; 257 .. 512, 769 .. 1024 and 1537 .. 2048 rows keep 8, 4 and 2 ranges.
    const int64_t tiles = dma_tiles(M, N);
    if (tiles <= 256) {
      for (int s = 2; s <= 16 && kt / s >= 16; ++s)
        if (dma_cost(tiles, kt, s) < dma_cost(tiles, kt, splits)) splits = s;
      // a short K, whose partials weigh as much as the walk they save: two ranges as long as they fill the chip (K = 2432,
      // N = 4096, 1808 rows 62 us, one range of 128 x 128 tiles 71; N = 512, K = 2560, 14000 rows 75 and 86)
      if (splits == 1 && tiles >= 100 && tiles <= 128 && kt % 2 == 0 && kt >= 32) splits = 2;
      if (tiles * splits >= DMA_MIN_TILES) return {0, splits};
      splits = 1;
    } else {
      // Beyond that the last round would leave most CUs idle for a whole tile's time: whole rounds first, then the rest as
      // a problem of its own, if that costs less (its second launch and the separate LayerNorm of the front rows: 5 us).
      // With the reduce and the following LayerNorm: 4097 rows 1034 -> 590 us, 4900 1024 -> 719, 5632 1029 -> 841, 6500
      // 1024 -> 947 (7000 stays at 1021), 8200 1573 -> 1125, 9000 1552 -> 1255.
      // Only 2, 3, 4, 8 or 16 ranges: 5 would save another 15 us at 48 tiles for more workspace.  (The most that any row count
      // needs at N = 4096, K = 20480 is 120 MiB, three ranges of 160 tiles above; powers of two alone needed 64.)
      const int64_t cols = (N + 255) / 256, rounds = tiles / 256;
      const int64_t front = rounds * 256 / cols * 256;
      if (front > 0 && M - front > 0) {
        const int64_t rest = dma_tiles(M - front, N), front_cost = (front / 256 * cols + 255) / 256 * kt * 10;
        int64_t best = dma_cost(tiles, kt, 1) - front_cost - 36;
        if (M - front <= 256) {              // these rows go to gemm_stream_kernel: its own ranges, a tile of it costs no more
          const int s = pick_cut(M - front, N, K, dtype).splits;
          if (dma_cost(2 * rest, kt, s) < best) splits = s;
        } else {
          for (int s : {2, 3, 4, 8, 16})
            if (kt / s >= 16 && rest * s >= DMA_MIN_TILES && dma_cost(rest, kt, s) < best) {
              best = dma_cost(rest, kt, s);
              splits = s;
            }
        }
        if (splits > 1) return {front, splits};
      }
      return {0, 1};
    }
  }
  // 128 x 128 tiles, two workgroups per CU: up to 4 ranges.  The k-tiles of float32 take longer than the partials they cost, so up to
  // 16 where the workspace holds them (N = 4096, K = 20480, 4 / 8 / 16 at most: 65 rows 184 / 147 / 132 us, 128 rows 197 / 166 /
  // 150, 199 296 / 247 / 252; N = 1024, K = 5120, 100 rows 46 / 29 / 29)
  if (dtype != MTJ_F32) most = 4;
  const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128);
  while (splits < most && tiles * splits * 2 <= 512 && kt % (splits * 2) == 0 && kt / (splits * 2) >= 16) splits *= 2;
  return {0, splits};
}

int64_t cut_bytes(const cut_t& cut, int64_t M, int64_t N) {
  return cut.splits > 1 ? (int64_t)cut.splits * (M - cut.front) * N * (int64_t)sizeof(float) : 0;
}
bool work_holds(const cut_t& cut, int64_t M, int64_t N, const void* work, int64_t work_bytes) {
  return work && mtj_aligned16(work) && work_bytes >= cut_bytes(cut, M, N);
}
// The most ranges that the workspace holds, and four where it holds less: a call with the workspace that
// mtj_gemm_splitk_work_bytes asks for, or with that of another row count, is not refused for the sake of a faster cut.
cut_t cut_for(int64_t M, int64_t N, int64_t K, int dtype, const void* work, int64_t work_bytes) {
  for (int most : {16, 8}) {
    const cut_t cut = pick_cut(M, N, K, dtype, most);
    if (work_holds(cut, M, N, work, work_bytes)) return cut;
  }
  return pick_cut(M, N, K, dtype);
}

// Problems whose tiles of one K range leave more than half of the chip idle: mtj_gemm_splitk asks for an `out` that the
// reduce can take in quads, and for the workspace, for these, whatever pick_cut makes of them.  Every other problem can
// also run in one range, and does where these do not allow a cut.
// (Tiles of 128 columns up to 64 rows, of 128 x 128 beyond, two workgroups per CU; 16-bit operands also count the
// 256 x 256 tiles that two ranges bring to 200 .. 256; a range has at least 4 or 16 k-tiles.)
bool needs_ranges(int64_t M, int64_t N, int64_t K, int dtype) {
  const int64_t kt = K / (dtype == MTJ_F32 ? 32 : 64), cols = (N + 127) / 128;
  if (N % 4 || kt % 2) return false;
  if (M <= 64) return cols <= 128 && kt >= 8;
  const int64_t big = dma_tiles(M, N);
  return kt >= 32 && ((M + 127) / 128 * cols <= 256 || (dtype != MTJ_F32 && big >= 100 && big <= 128));
}

int check_common(const void* A, int64_t lda, const void* W, int64_t M, int64_t N, int64_t K, int dtype, const char* who) {
  MTJ_REQUIRE(A && W, MTJ_EINVAL, "%s: null pointer", who);
  MTJ_REQUIRE(mtj_is_dtype(dtype), MTJ_EDTYPE, "%s: dtype %d", who, dtype);
  const int bk = dtype == MTJ_F32 ? 32 : 64;
  const int esz = mtj_elem_size(dtype);
  MTJ_REQUIRE(M > 0 && N > 0 && K > 0 && K % bk == 0 && lda >= K, MTJ_EINVAL,
              "%s: bad shape M=%lld N=%lld K=%lld lda=%lld (K must be a multiple of %d)", who, (long long)M,
              (long long)N, (long long)K, (long long)lda, bk);
  MTJ_REQUIRE(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), MTJ_ELIMIT, "%s: dimension too large", who);
  MTJ_REQUIRE(mtj_aligned16(A) && mtj_aligned16(W) && (lda * esz) % 16 == 0, MTJ_EALIGN,
              "%s: A, W and the row stride of A must be 16-byte aligned", who);
  MTJ_REQUIRE(256 * lda * esz < (1ll << 30) && 256 * K * esz < (1ll << 30), MTJ_ELIMIT,
              "%s: a 256-row tile of A or W must span less than 1 GiB", who);
  return MTJ_OK;
}

}  // namespace

namespace {
int dispatch_dtype(const gemm_args& a, int dtype, int epi, hipStream_t s) {
  if (dtype == MTJ_BF16) return dispatch<bf16_t, 64>(a, epi, s);
  if (dtype == MTJ_F16) return dispatch<f16_t, 64>(a, epi, s);
  return dispatch<float, 32>(a, epi, s);
}
const void* rows_from(const void* base, int64_t elems, int dtype) {
  return reinterpret_cast<const unsigned char*>(base) + elems * mtj_elem_size(dtype);
}
}  // namespace

extern "C" int mtj_gemm(const void* A, int64_t lda, const void* W, const float* bias, int64_t M, int64_t N, int64_t K,
                        int dtype, int epi, void* out, int64_t ldo, int out_dtype, const mtj_inproj* ip, float alpha,
                        void* stream) {
  if (int rc = check_common(A, lda, W, M, N, K, dtype, "mtj_gemm")) return rc;
  gemm_args a{};
  a.A = A; a.lda = lda; a.W = W; a.bias = bias; a.M = (int)M; a.N = (int)N; a.K = (int)K;
  a.out = out; a.ldo = ldo; a.out_dtype = out_dtype; a.alpha = alpha; a.splits = 1;
  if (epi == MTJ_EPI_INPROJ) {
    MTJ_REQUIRE(ip && bias, MTJ_EINVAL, "mtj_gemm: INPROJ needs ip and the fc_in bias");
    a.ip = *ip;
    const int64_t d = (int64_t)ip->n_heads * ip->d_head;
    MTJ_REQUIRE(ip->Tp > 0 && (ip->rows || M % ip->Tp == 0) && N > 3 * d && N % 32 == 0 && d % 32 == 0 && ip->d_head % 32 == 0 &&
                    ip->rotary_dims % 16 == 0 && ip->ld_act % 16 == 0 &&
                    ip->rotary_dims <= ip->d_head && ip->Tcap > 0 && ip->max_pos > 0 && ip->pos0 && ip->sin_tab &&
                    ip->cos_tab && ip->q && ip->k_cache && ip->v_cache && ip->act && ip->ld_act >= N - 2 * d &&
                    mtj_is_dtype(ip->act_dtype) && mtj_is_dtype(ip->q_dtype) && mtj_is_dtype(ip->kv_dtype) &&
                    (!ip->v_t || ip->ldvt >= ip->Tp),
                MTJ_EINVAL, "mtj_gemm: inconsistent INPROJ geometry");
    MTJ_REQUIRE(mtj_aligned16(bias) && mtj_aligned16(ip->sin_tab) && mtj_aligned16(ip->cos_tab), MTJ_EALIGN,
                "mtj_gemm: the fc_in bias and the rotary tables must be 16-byte aligned");
  } else if (epi == MTJ_EPI_STORE) {
    MTJ_REQUIRE(out && ldo >= N && mtj_is_dtype(out_dtype), MTJ_EINVAL, "mtj_gemm: STORE needs out with ldo >= N");
  } else if (epi == MTJ_EPI_RESID) {
    MTJ_REQUIRE(out && ldo >= N, MTJ_EINVAL, "mtj_gemm: RESID needs out with ldo >= N");
  } else {
    return mtj_fail(MTJ_EINVAL, "mtj_gemm: epilogue %d", epi);
  }
  if (const int64_t front = epi == MTJ_EPI_INPROJ && dtype != MTJ_F32 ? inproj_front(M, N, K) : 0) {
    a.M = (int)front;
    if (int rc = dispatch_dtype(a, dtype, epi, (hipStream_t)stream)) return rc;
    a.A = rows_from(A, front * lda, dtype);
    a.M = (int)(M - front);
    a.m_base = (int)front;
  }
  return dispatch_dtype(a, dtype, epi, (hipStream_t)stream);
}

extern "C" int64_t mtj_gemm_splitk_work_bytes(int64_t M, int64_t N, int64_t K, int dtype) {
  if (M <= 0 || N <= 0 || K <= 0 || !mtj_is_dtype(dtype)) return 0;
  return cut_bytes(pick_cut(M, N, K, dtype), M, N);
}
extern "C" int64_t mtj_gemm_splitk_best_work_bytes(int64_t M, int64_t N, int64_t K, int dtype) {
  if (M <= 0 || N <= 0 || K <= 0 || !mtj_is_dtype(dtype)) return 0;
  return cut_bytes(pick_cut(M, N, K, dtype, 16), M, N);
}

extern "C" int mtj_gemm_splitk(const void* A, int64_t lda, const void* W, const float* bias, int64_t M, int64_t N,
                               int64_t K, int dtype, int epi, void* out, int64_t ldo, int out_dtype, void* work,
                               int64_t work_bytes, float alpha, void* stream) {
  MTJ_REQUIRE(epi == MTJ_EPI_STORE || epi == MTJ_EPI_RESID, MTJ_EINVAL, "mtj_gemm_splitk: epilogue %d", epi);
  if (int rc = check_common(A, lda, W, M, N, K, dtype, "mtj_gemm_splitk")) return rc;
  const cut_t cut = cut_for(M, N, K, dtype, work, work_bytes);
  const int splits = cut.splits;
  // the reduce moves four columns at a time
  const bool rows_ok = out && ldo >= N && ldo % 4 == 0 && mtj_aligned16(out) && (!bias || mtj_aligned16(bias));
  const bool need = needs_ranges(M, N, K, dtype);
  MTJ_REQUIRE(rows_ok || !need, MTJ_EINVAL,
              "mtj_gemm_splitk: out needs ldo >= N, a multiple of 4, and 16-byte alignment (bias too)");
  if (splits == 1 || !rows_ok || (!need && !work_holds(cut, M, N, work, work_bytes)))
    return mtj_gemm(A, lda, W, bias, M, N, K, dtype, epi, out, ldo, out_dtype, nullptr, alpha, stream);
  MTJ_REQUIRE(epi == MTJ_EPI_RESID || mtj_is_dtype(out_dtype), MTJ_EDTYPE, "mtj_gemm_splitk: out_dtype %d", out_dtype);
  MTJ_REQUIRE(work_holds(cut, M, N, work, work_bytes), MTJ_EINVAL, "mtj_gemm_splitk: work must hold mtj_gemm_splitk_work_bytes() bytes");
  if (cut.front) {
    if (int rc = mtj_gemm(A, lda, W, bias, cut.front, N, K, dtype, epi, out, ldo, out_dtype, nullptr, alpha, stream)) return rc;
    A = rows_from(A, cut.front * lda, dtype);
    out = const_cast<void*>(rows_from(out, cut.front * ldo, epi == MTJ_EPI_RESID ? MTJ_F32 : out_dtype));
    M -= cut.front;
  }
  gemm_args a{};
  a.A = A; a.lda = lda; a.W = W; a.bias = nullptr; a.M = (int)M; a.N = (int)N; a.K = (int)K;
  a.out = work; a.ldo = N; a.out_dtype = MTJ_F32; a.alpha = alpha;
  a.splits = splits; a.split_stride = M * N;
  hipStream_t s = (hipStream_t)stream;
  if (int rc = dispatch_dtype(a, dtype, MTJ_EPI_STORE, s)) return rc;
  const int64_t quads = M * (N / 4);
  const unsigned grid = (unsigned)((quads + 255) / 256);
  if (epi == MTJ_EPI_RESID)
    splitk_reduce_kernel<MTJ_EPI_RESID><<<grid, 256, 0, s>>>((const float*)work, splits, M * N, (int)M, (int)N, bias, out, ldo, MTJ_F32);
  else
    splitk_reduce_kernel<MTJ_EPI_STORE><<<grid, 256, 0, s>>>((const float*)work, splits, M * N, (int)M, (int)N, bias, out, ldo, out_dtype);
  return mtj_check_launch("mtj_gemm_splitk");
}

extern "C" int mtj_gemm_splitk_ln(const void* A, int64_t lda, const void* W, const float* bias, int64_t M, int64_t N,
                                  int64_t K, int dtype, float* x, int64_t ldx, void* work, int64_t work_bytes,
                                  const float* ln_scale, const float* ln_offset, void* h, int64_t ldh, int h_dtype,
                                  float alpha, void* stream) {
  MTJ_REQUIRE(ln_scale && ln_offset && h && x, MTJ_EINVAL, "mtj_gemm_splitk_ln: null pointer");
  MTJ_REQUIRE(mtj_is_dtype(h_dtype), MTJ_EDTYPE, "mtj_gemm_splitk_ln: h_dtype %d", h_dtype);
  MTJ_REQUIRE(N % 4 == 0 && N <= 4 * RLN_Q * 1024 && ldh >= N && ldh % 4 == 0 && ldx >= N && ldx % 4 == 0 &&
                  mtj_aligned16(x) && mtj_aligned16(h) && mtj_aligned16(ln_scale) && mtj_aligned16(ln_offset) &&
                  (!bias || mtj_aligned16(bias)),
              MTJ_EINVAL, "mtj_gemm_splitk_ln: N a multiple of 4 and <= %d, rows of x and h 16-byte aligned", 4 * RLN_Q * 1024);
  if (int rc = check_common(A, lda, W, M, N, K, dtype, "mtj_gemm_splitk_ln")) return rc;
  const cut_t cut = cut_for(M, N, K, dtype, work, work_bytes);
  const int splits = cut.splits;
  // mtj_layernorm takes dense rows; pick_cut leaves none to it where needs_ranges holds (N <= 16384)
  const bool need = needs_ranges(M, N, K, dtype);
  MTJ_REQUIRE((ldx == N && ldh == N) || need, MTJ_EINVAL,
              "mtj_gemm_splitk_ln: x and h must be dense where one K range fills the chip");
  hipStream_t s = (hipStream_t)stream;
  if (splits == 1 || (!need && !work_holds(cut, M, N, work, work_bytes))) {      // no partials to reduce: the product with its own residual epilogue, then the plain LayerNorm
    if (int rc = mtj_gemm(A, lda, W, bias, M, N, K, dtype, MTJ_EPI_RESID, x, ldx, MTJ_F32, nullptr, alpha, stream)) return rc;
    return mtj_layernorm(x, ln_scale, ln_offset, M, N, h, h_dtype, stream);
  }
  MTJ_REQUIRE(work_holds(cut, M, N, work, work_bytes), MTJ_EINVAL, "mtj_gemm_splitk_ln: work must hold mtj_gemm_splitk_work_bytes() bytes");
  if (cut.front) {
    if (int rc = mtj_gemm(A, lda, W, bias, cut.front, N, K, dtype, MTJ_EPI_RESID, x, ldx, MTJ_F32, nullptr, alpha, stream)) return rc;
    if (int rc = mtj_layernorm(x, ln_scale, ln_offset, cut.front, N, h, h_dtype, stream)) return rc;
    A = rows_from(A, cut.front * lda, dtype);
    x += cut.front * ldx;
    h = const_cast<void*>(rows_from(h, cut.front * ldh, h_dtype));
    M -= cut.front;
  }
  gemm_args a{};
  a.A = A; a.lda = lda; a.W = W; a.bias = nullptr; a.M = (int)M; a.N = (int)N; a.K = (int)K;
  a.out = work; a.ldo = N; a.out_dtype = MTJ_F32; a.alpha = alpha;
  a.splits = splits; a.split_stride = M * N;
  if (int rc = dispatch_dtype(a, dtype, MTJ_EPI_STORE, s)) return rc;
  if (N <= 4096)
    splitk_reduce_ln_kernel<1><<<(unsigned)M, rln_threads(N), 0, s>>>((const float*)work, splits, M * N, (int)N, bias, x, ldx, ln_scale,
                                                                      ln_offset, h, ldh, h_dtype);
  else
    splitk_reduce_ln_kernel<RLN_Q><<<(unsigned)M, rln_threads(N), 0, s>>>((const float*)work, splits, M * N, (int)N, bias, x, ldx,
                                                                          ln_scale, ln_offset, h, ldh, h_dtype);
  return mtj_check_launch("mtj_gemm_splitk_ln");
}

extern "C" int64_t mtj_gemm_xent_work_bytes(int64_t M, int64_t N, int dtype) {
  if (M <= 0 || N <= 0 || !mtj_is_dtype(dtype)) return 0;
  const int64_t tiles_n = (N + xent_tile_n(M, N, dtype) - 1) / xent_tile_n(M, N, dtype);
  return (2 * tiles_n + 1) * M * (int64_t)sizeof(float);
}

extern "C" int mtj_gemm_xent(const void* A, int64_t lda, const void* W, const float* bias, int64_t M, int64_t N, int64_t K,
                             int dtype, float alpha, const int32_t* target, float* loss, uint8_t* correct, void* work,
                             int64_t work_bytes, void* stream) {
  if (int rc = check_common(A, lda, W, M, N, K, dtype, "mtj_gemm_xent")) return rc;
  MTJ_REQUIRE(target && loss && work, MTJ_EINVAL, "mtj_gemm_xent: null pointer");
  MTJ_REQUIRE(mtj_aligned16(work) && work_bytes >= mtj_gemm_xent_work_bytes(M, N, dtype), MTJ_EINVAL,
              "mtj_gemm_xent: work must hold mtj_gemm_xent_work_bytes() bytes");
  const int bn = xent_tile_n(M, N, dtype);
  const int64_t tiles_n = (N + bn - 1) / bn;
  gemm_args a{};
  a.A = A; a.lda = lda; a.W = W; a.bias = bias; a.M = (int)M; a.N = (int)N; a.K = (int)K;
  a.alpha = alpha; a.splits = 1;
  a.target = target;
  a.pmax = reinterpret_cast<float*>(work);
  a.psum = a.pmax + tiles_n * M;
  a.tlogit = a.psum + tiles_n * M;
  hipStream_t s = (hipStream_t)stream;
  if (int rc = dispatch_dtype(a, dtype, MTJ_EPI_XENT, s)) return rc;
  xent_merge_kernel<<<(unsigned)((M + XM_ROWS - 1) / XM_ROWS), XM_ROWS * XM_LANES, 0, s>>>(a.pmax, a.psum, a.tlogit, target, (int)M, (int)N, (int)tiles_n,
                                                              loss, correct);
  return mtj_check_launch("mtj_gemm_xent");
}
