// Error plumbing, weight packing, embedding gather and LayerNorm.
#include "mtj_common.h"

// ---------------------------------------------------------------- errors
static thread_local char g_err[512] = "";

int mtj_fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int mtj_check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return mtj_fail(MTJ_EHIP, "%s: %s", what, hipGetErrorString(e));
  return MTJ_OK;
}

extern "C" int mtj_version(void) { return MTJ_ABI_VERSION; }
extern "C" const char* mtj_last_error(void) { return g_err; }

// ---------------------------------------------------------------- pack: dst[(n_off+n)*Kt + k_off+k] = src[k*ld + n]
// 32x32 tiles through LDS so that both the read (along n) and the write (along k) are coalesced.
template <typename T>
__global__ __launch_bounds__(256) void pack_kernel(const T* __restrict__ src, int64_t ld, int64_t K, int64_t N,
                                                   T* __restrict__ dst, int64_t Kt, int64_t n_off, int64_t k_off) {
  __shared__ T tile[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  const int64_t n0 = (int64_t)blockIdx.x * 32, k0 = (int64_t)blockIdx.y * 32;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t k = k0 + ty + i * 8, n = n0 + tx;
    if (k < K && n < N) tile[ty + i * 8][tx] = src[k * ld + n];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t n = n0 + ty + i * 8, k = k0 + tx;
    if (k < K && n < N) dst[(n_off + n) * Kt + k_off + k] = tile[tx][ty + i * 8];
  }
}

// the same tiles with a change of type: dst = round(src * scale)
template <typename TS, typename TD>
__global__ __launch_bounds__(256) void pack_cvt_kernel(const TS* __restrict__ src, int64_t ld, int64_t K, int64_t N,
                                                       TD* __restrict__ dst, int64_t Kt, int64_t n_off, int64_t k_off,
                                                       float scale) {
  __shared__ float tile[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int64_t n0 = (int64_t)blockIdx.x * 32, k0 = (int64_t)blockIdx.y * 32;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t k = k0 + ty + i * 8, n = n0 + tx;
    if (k < K && n < N) tile[ty + i * 8][tx] = elem<TS>::load(src + k * ld + n) * scale;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t n = n0 + ty + i * 8, k = k0 + tx;
    if (k < K && n < N) elem<TD>::store(dst + (n_off + n) * Kt + k_off + k, tile[tx][ty + i * 8]);
  }
}

extern "C" int mtj_pack_weight_cvt(const void* src, int64_t src_ld, int64_t K, int64_t N, void* dst, int64_t K_total,
                                   int64_t n_off, int64_t k_off, int src_dtype, int dst_dtype, float scale, void* stream) {
  MTJ_REQUIRE(src && dst, MTJ_EINVAL, "mtj_pack_weight_cvt: null pointer");
  MTJ_REQUIRE(K > 0 && N > 0 && src_ld >= N && n_off >= 0 && k_off >= 0 && k_off + K <= K_total, MTJ_EINVAL,
              "mtj_pack_weight_cvt: bad shape K=%lld N=%lld ld=%lld K_total=%lld k_off=%lld", (long long)K, (long long)N,
              (long long)src_ld, (long long)K_total, (long long)k_off);
  MTJ_REQUIRE(scale > 0.f && scale < INFINITY, MTJ_EINVAL, "mtj_pack_weight_cvt: scale must be positive and finite");
  dim3 grid((unsigned)((N + 31) / 32), (unsigned)((K + 31) / 32));
  hipStream_t s = (hipStream_t)stream;
#define MTJ_CVT(SD, TS, DD, TD)                                                                                    \
  if (src_dtype == SD && dst_dtype == DD) {                                                                        \
    pack_cvt_kernel<TS, TD><<<grid, 256, 0, s>>>((const TS*)src, src_ld, K, N, (TD*)dst, K_total, n_off, k_off, scale); \
    return mtj_check_launch("mtj_pack_weight_cvt");                                                               \
  }
  MTJ_CVT(MTJ_BF16, bf16_t, MTJ_F16, f16_t)
  MTJ_CVT(MTJ_F32, float, MTJ_F16, f16_t)
  MTJ_CVT(MTJ_F32, float, MTJ_BF16, bf16_t)
  MTJ_CVT(MTJ_BF16, bf16_t, MTJ_F32, float)
  MTJ_CVT(MTJ_F16, f16_t, MTJ_F32, float)
#undef MTJ_CVT
  return mtj_fail(MTJ_EDTYPE, "mtj_pack_weight_cvt: no conversion from dtype %d to dtype %d", src_dtype, dst_dtype);
}

extern "C" int mtj_pack_weight(const void* src, int64_t src_ld, int64_t K, int64_t N, void* dst, int64_t K_total,
                               int64_t n_off, int64_t k_off, int dtype, void* stream) {
  MTJ_REQUIRE(src && dst, MTJ_EINVAL, "mtj_pack_weight: null pointer");
  MTJ_REQUIRE(K > 0 && N > 0 && src_ld >= N && n_off >= 0 && k_off >= 0 && k_off + K <= K_total, MTJ_EINVAL,
              "mtj_pack_weight: bad shape K=%lld N=%lld ld=%lld K_total=%lld k_off=%lld", (long long)K, (long long)N,
              (long long)src_ld, (long long)K_total, (long long)k_off);
  dim3 grid((unsigned)((N + 31) / 32), (unsigned)((K + 31) / 32));
  hipStream_t s = (hipStream_t)stream;
  if (dtype == MTJ_F32)
    pack_kernel<float><<<grid, 256, 0, s>>>((const float*)src, src_ld, K, N, (float*)dst, K_total, n_off, k_off);
  else if (dtype == MTJ_BF16 || dtype == MTJ_F16)
    pack_kernel<uint16_t><<<grid, 256, 0, s>>>((const uint16_t*)src, src_ld, K, N, (uint16_t*)dst, K_total, n_off, k_off);
  else
    return mtj_fail(MTJ_EDTYPE, "mtj_pack_weight: dtype %d", dtype);
  return mtj_check_launch("mtj_pack_weight");
}

// ---------------------------------------------------------------- embedding: one row per workgroup
template <typename T>
__global__ __launch_bounds__(256) void embed_kernel(const int32_t* __restrict__ tok, const T* __restrict__ W,
                                                    const float* __restrict__ b, int64_t V, int64_t d,
                                                    float* __restrict__ out) {
  const int64_t m = blockIdx.x;
  const int64_t t = (uint32_t)tok[m];
  const bool hit = t < V;  // an out-of-range id is an all-zero one-hot row
  for (int64_t c = threadIdx.x; c < d; c += blockDim.x) {
    const float w = hit ? elem<T>::load(W + t * d + c) : 0.0f;
    out[m * d + c] = w + b[c];
  }
}

extern "C" int mtj_embed(const int32_t* tok, int64_t M, const void* W, const float* b, int64_t n_vocab, int64_t d,
                         int dtype, float* out, void* stream) {
  MTJ_REQUIRE(tok && W && b && out, MTJ_EINVAL, "mtj_embed: null pointer");
  MTJ_REQUIRE(M > 0 && d > 0 && n_vocab > 0, MTJ_EINVAL, "mtj_embed: bad shape");
  hipStream_t s = (hipStream_t)stream;
  if (dtype == MTJ_F32)
    embed_kernel<float><<<(unsigned)M, 256, 0, s>>>(tok, (const float*)W, b, n_vocab, d, out);
  else if (dtype == MTJ_BF16)
    embed_kernel<bf16_t><<<(unsigned)M, 256, 0, s>>>(tok, (const bf16_t*)W, b, n_vocab, d, out);
  else if (dtype == MTJ_F16)
    embed_kernel<f16_t><<<(unsigned)M, 256, 0, s>>>(tok, (const f16_t*)W, b, n_vocab, d, out);
  else
    return mtj_fail(MTJ_EDTYPE, "mtj_embed: dtype %d", dtype);
  return mtj_check_launch("mtj_embed");
}

// ---------------------------------------------------------------- LayerNorm
// Two passes over a row that stays in registers (mean first, then centred variance, as the reference
// computes jnp.var); all statistics float32.
constexpr int LN_MAX = 4096;         // columns

// WG false: a wavefront per row, four rows per workgroup (up to 1024 columns); WG true: a workgroup of four wavefronts per row.
// Four float4 per lane either way.  Bound by memory: what matters is that a CU has other rows in flight while one is reduced,
// and for a few rows that a row is asked for at once.  With a wavefront per row of 4096 columns (64 registers for the row, 16
// loads one behind the other) 3 rows took 7.4 us, now 4.3; 511 10.3 -> 5.6, 2872 21.2 -> 16.8, 32736 214 -> 156 (5.2 TB/s); 50000
// rows of 512 columns 54 -> 29, 2000 of 2048 8.2 -> 6.9.
template <int OUT_DTYPE, bool WG>
__global__ __launch_bounds__(256) void layernorm_kernel(const float* __restrict__ x, const float* __restrict__ scale,
                                                        const float* __restrict__ offset, int64_t M, int d,
                                                        void* __restrict__ out) {
  constexpr int NT = WG ? 256 : 64, V = 4;
  __shared__ float red[2][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, at = WG ? threadIdx.x : lane;
  const int64_t row = WG ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * 4 + wave;
  if (row >= M) return;
  const float* xr = x + row * d;
  const int nvec = d >> 2;  // float4 chunks
  auto row_sum = [&](float s, int which) {
    s = wave_sum(s);
    if constexpr (WG) {
      if (lane == 0) red[which][wave] = s;
      __syncthreads();
      s = (red[which][0] + red[which][1]) + (red[which][2] + red[which][3]);
    }
    return s;
  };
  floatx4 v[V];
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = i * NT + at;
    if (c < nvec) {
      v[i] = *reinterpret_cast<const floatx4*>(xr + 4 * c);
      sum += (v[i].x + v[i].y) + (v[i].z + v[i].w);
    }
  }
  const float mean = row_sum(sum, 0) / (float)d;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = i * NT + at;
    if (c < nvec) {
      const floatx4 t = v[i] - mean;
      sq += (t.x * t.x + t.y * t.y) + (t.z * t.z + t.w * t.w);
    }
  }
  const float inv = rsqrtf(row_sum(sq, 1) / (float)d + 1e-5f);
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = i * NT + at;
    if (c < nvec) {
      const floatx4 sc = *reinterpret_cast<const floatx4*>(scale + 4 * c);
      const floatx4 of = *reinterpret_cast<const floatx4*>(offset + 4 * c);
      const floatx4 y = (sc * inv) * (v[i] - mean) + of;
      if (OUT_DTYPE == MTJ_F32) {
        *reinterpret_cast<floatx4*>(reinterpret_cast<float*>(out) + row * d + 4 * c) = y;
      } else {
        uint32x2 p;
        p.x = pack_16x2(y.x, y.y, OUT_DTYPE);
        p.y = pack_16x2(y.z, y.w, OUT_DTYPE);
        // streaming store: 16384 x 4096 rows in 81 us instead of 109 (the normalised rows are read again only by
        // the GEMM that follows, from the start, after all of them have been written)
        __builtin_nontemporal_store(p, reinterpret_cast<uint32x2*>(reinterpret_cast<uint16_t*>(out) + row * d + 4 * c));
      }
    }
  }
}

template <int OUT_DTYPE>
void launch_layernorm(const float* x, const float* scale, const float* offset, int64_t M, int d, void* out, hipStream_t s) {
  // a launch has less than 2^32 threads
  constexpr int64_t MOST = 1 << 23;
  const int esz = OUT_DTYPE == MTJ_F32 ? 4 : 2;
  for (int64_t m = 0; m < M; m += MOST, x += MOST * d, out = (char*)out + MOST * d * esz) {
    const int64_t rows = M - m < MOST ? M - m : MOST;
    if (d <= 1024) layernorm_kernel<OUT_DTYPE, false><<<(unsigned)((rows + 3) / 4), 256, 0, s>>>(x, scale, offset, rows, d, out);
    else layernorm_kernel<OUT_DTYPE, true><<<(unsigned)rows, 256, 0, s>>>(x, scale, offset, rows, d, out);
  }
}

extern "C" int mtj_layernorm(const float* x, const float* scale, const float* offset, int64_t M, int64_t d,
                             void* out, int out_dtype, void* stream) {
  MTJ_REQUIRE(x && scale && offset && out, MTJ_EINVAL, "mtj_layernorm: null pointer");
  MTJ_REQUIRE(M > 0 && d > 0 && d % 4 == 0 && d <= LN_MAX, MTJ_EINVAL,
              "mtj_layernorm: d=%lld must be a multiple of 4 and <= %d", (long long)d, LN_MAX);
  MTJ_REQUIRE(mtj_aligned16(x) && mtj_aligned16(scale) && mtj_aligned16(offset) && mtj_aligned16(out), MTJ_EALIGN,
              "mtj_layernorm: pointers must be 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  if (out_dtype == MTJ_F32) launch_layernorm<MTJ_F32>(x, scale, offset, M, (int)d, out, s);
  else if (out_dtype == MTJ_BF16) launch_layernorm<MTJ_BF16>(x, scale, offset, M, (int)d, out, s);
  else if (out_dtype == MTJ_F16) launch_layernorm<MTJ_F16>(x, scale, offset, M, (int)d, out, s);
  else
    return mtj_fail(MTJ_EDTYPE, "mtj_layernorm: out_dtype %d", out_dtype);
  return mtj_check_launch("mtj_layernorm");
}

// ---------------------------------------------------------------- rotary embedding + K/V window append on its own
// The epilogue of the fused input projection applied to rows that are already projected: element (m, c) of q, v, k
// [M, d] goes where inproj_store sends column c, d + c, 2d + c of row m (layers.py:261-273: interleaved rotation of
// the first rotary_dims of every head of q and k at position pos0[b] + t; layers.py:325-326: the window slot).
__global__ __launch_bounds__(256) void rope_append_kernel(const float* __restrict__ q, const float* __restrict__ v,
                                                          const float* __restrict__ k, int64_t M, const mtj_inproj ip) {
  const int d = ip.n_heads * ip.d_head;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= M * d) return;
  const int64_t m = i / d;
  const int c = (int)(i - m * d);
  const float* src[3] = {q, v, k};
#pragma unroll
  for (int seg = 0; seg < 3; ++seg) {
    if (!src[seg]) continue;
    inproj_store(ip, nullptr, m, (int64_t)seg * d + c, src[seg][m * d + c], src[seg][m * d + (c ^ 1)]);
  }
}

extern "C" int mtj_rope_append(const float* q, const float* v, const float* k, int64_t M, const mtj_inproj* ip, void* stream) {
  MTJ_REQUIRE(ip && M > 0 && (q || v || k), MTJ_EINVAL, "mtj_rope_append: nothing to do");
  MTJ_REQUIRE(!ip->rows && ip->n_heads > 0 && ip->d_head > 0 && ip->d_head % 2 == 0 && ip->rotary_dims % 2 == 0 &&
                  ip->rotary_dims >= 0 && ip->rotary_dims <= ip->d_head && ip->Tp > 0 && M % ip->Tp == 0 && ip->Tcap > 0 &&
                  ip->max_pos > 0 && ip->pos0 && ip->sin_tab && ip->cos_tab,
              MTJ_EINVAL, "mtj_rope_append: inconsistent geometry");
  MTJ_REQUIRE((!q || (ip->q && mtj_is_dtype(ip->q_dtype))) && (!v || ip->v_cache) && (!k || ip->k_cache) &&
                  ((!v && !k) || mtj_is_dtype(ip->kv_dtype)) && (!ip->v_t || ip->ldvt >= ip->Tp),
              MTJ_EINVAL, "mtj_rope_append: a destination is missing for a given source");
  const int64_t n = M * ip->n_heads * ip->d_head;
  MTJ_REQUIRE(n < (1ll << 39), MTJ_ELIMIT, "mtj_rope_append: too many elements");
  rope_append_kernel<<<(unsigned)((n + 255) / 256), 256, 0, (hipStream_t)stream>>>(q, v, k, M, *ip);
  return mtj_check_launch("mtj_rope_append");
}

// ---------------------------------------------------------------- cross entropy of a logits row
// ProjectionShard.loss (layers.py:569-593) on one shard: logits -= max; loss = log(sum exp) - logits[target];
// correct = (logits[target] == 0), i.e. the target holds the row maximum.  One 256-thread workgroup per row.
__global__ __launch_bounds__(256) void xent_kernel(const float* __restrict__ logits, const int32_t* __restrict__ target,
                                                   int64_t ld, int V, float* __restrict__ loss,
                                                   uint8_t* __restrict__ correct) {
  __shared__ float red[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* row = logits + (int64_t)blockIdx.x * ld;
  float m = -INFINITY;
  for (int i = tid; i < V; i += 256) m = fmaxf(m, row[i]);
  m = wave_max(m);
  if (lane == 0) red[wave] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  float s = 0.f;
  for (int i = tid; i < V; i += 256) s += expf(row[i] - m);
  s = wave_sum(s);
  if (lane == 0) red[wave] = s;
  __syncthreads();
  if (tid == 0) {
    const float total = (red[0] + red[1]) + (red[2] + red[3]);
    const int t = target[blockIdx.x];
    const float pred = ((uint32_t)t < (uint32_t)V) ? row[t] - m : 0.f;    // an all-zero one-hot row selects nothing
    loss[blockIdx.x] = logf(total) - pred;
    if (correct) correct[blockIdx.x] = (pred == 0.f) ? 1 : 0;
  }
}

extern "C" int mtj_xent(const float* logits, int64_t ld, const int32_t* target, int64_t M, int64_t V, float* loss,
                        uint8_t* correct, void* stream) {
  MTJ_REQUIRE(logits && target && loss, MTJ_EINVAL, "mtj_xent: null pointer");
  MTJ_REQUIRE(M > 0 && M < (1ll << 31) && V > 0 && V < (1ll << 31) && ld >= V, MTJ_EINVAL,
              "mtj_xent: bad shape M=%lld V=%lld ld=%lld", (long long)M, (long long)V, (long long)ld);
  xent_kernel<<<(unsigned)M, 256, 0, (hipStream_t)stream>>>(logits, target, ld, (int)V, loss, correct);
  return mtj_check_launch("mtj_xent");
}
