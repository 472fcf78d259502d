// The kvtc codec's passes over coefficients and token-matrix rows (scripts/kvtc.py:62-79 quantize_groups,
// :142-155 rung_errors, :246-274 the coding at the chosen rungs and the rebuilt caches), each one pass where the
// tensor operations they replace made a dozen per rung or layer.  Every element is computed with the reference's
// float32 operations, each rounded on its own.
#include "dkv_device.h"
#include "dkv_host.h"

namespace {

// ---------------------------------------------------------------------------
// The ladder quantizer.  16 lanes take a 64-component group, 4 components each, so a wave takes 4 groups with
// one 1 KB load and a group's extremes are four lane exchanges.
// ---------------------------------------------------------------------------
struct GroupRange {
  float lo, hi;  // NaN when the group holds one, as torch's amin / amax give
  half_t low;    // the fp16 shift (the group's minimum)
};

DKV_DEVICE GroupRange group_range(const float4& x, int lane) {
  GroupRange r;
  r.lo = -max16(fmaxf(fmaxf(-x.x, -x.y), fmaxf(-x.z, -x.w)));
  r.hi = max16(fmaxf(fmaxf(x.x, x.y), fmaxf(x.z, x.w)));
  const unsigned long long nan = __ballot(x.x != x.x || x.y != x.y || x.z != x.z || x.w != x.w);
  if ((nan >> (lane & 48)) & 0xffffu) r.lo = r.hi = __builtin_nanf("");
  r.low = (half_t)r.lo;
  return r;
}

// fp16 step of a width whose largest level is `top`: (max - shift) / top, at least 1e-8.
DKV_DEVICE half_t ladder_step(const GroupRange& r, float top) {
  const float v = (r.hi - (float)r.low) / top;
  return (half_t)(v < 1e-8f ? 1e-8f : v);
}

DKV_DEVICE float ladder_level(float x, float low, float step, float top) {
  const float q = rintf((x - low) / step);
  return q < 0.0f ? 0.0f : (q > top ? top : q);  // a NaN (a step that rounds to 0) stays one
}

DKV_DEVICE float level_value(float level, float low, float step) {
#pragma clang fp contract(off)
  const float prod = level * step;
  return prod + low;
}

DKV_DEVICE float square_error(float x, float value) {
#pragma clang fp contract(off)
  const float d = x - value;
  return d * d;
}

// Squared error of every token at every rung of a ladder: errors[t][r] = sum over the groups of the group's error at
// bits[r][g].  One wave per token; a group's errors at 0, 2, 4 and 8 bits are summed over its 16 lanes, and
// lane j of the 16 adds up rungs j, j + 16, ...  The rungs share their groups' errors, so the pass costs three
// quantizations whatever their number (the tensor operations it replaces ran one per rung).
constexpr int kErrorTok = 4;  // tokens (waves) per workgroup

template <int NR>
__global__ __launch_bounds__(kErrorTok * 64) void ladder_errors_kernel(const float* __restrict__ coef, int n, int G,
                                                                       const uint8_t* __restrict__ bits, int R,
                                                                       float* __restrict__ errors) {
  extern __shared__ uint8_t sbits[];  // [R][G]
  for (int e = threadIdx.x; e < R * G; e += kErrorTok * 64) sbits[e] = bits[e];
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const long t = (long)blockIdx.x * kErrorTok + (threadIdx.x >> 6);
  if (t >= n) return;
  const int j = lane & 15, sub = lane >> 4;
  const float4* row = (const float4*)(coef + t * (64L * G));
  float acc[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) acc[i] = 0.0f;
  for (int g0 = 0; g0 < G; g0 += 4) {
    const int g = g0 + sub;
    const bool live = g < G;
    const float4 x = row[(live ? g : G - 1) * 16 + j];
    const GroupRange r = group_range(x, lane);
    const float low = (float)r.low;
    const float xv[4] = {x.x, x.y, x.z, x.w};
    float e[4];  // at 0, 2, 4, 8 bits
    const float tops[3] = {3.0f, 15.0f, 255.0f};
    e[0] = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) e[0] += square_error(xv[i], 0.0f);
#pragma unroll
    for (int w = 0; w < 3; ++w) {
      const float step = (float)ladder_step(r, tops[w]);
      e[w + 1] = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        e[w + 1] += square_error(xv[i], level_value(ladder_level(xv[i], low, step, tops[w]), low, step));
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) e[w] = sum16(e[w]);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int rr = j + 16 * i;
      const int b = live && rr < R ? sbits[rr * G + g] : -1;
      acc[i] += b < 0 ? 0.0f : b == 2 ? e[1] : b == 4 ? e[2] : b == 8 ? e[3] : e[0];
    }
  }
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const float s = sum_xor32(sum_xor16(acc[i]));  // the four groups of a step
    if (lane < 16 && j + 16 * i < R) errors[t * R + j + 16 * i] = s;
  }
}

// Every token coded at its level: a rung of the ladder (codes, fp16 shift and step, and the dequantized
// coefficients), the level after the last (the coefficients as they are, no codes), or -1 (zeros).
__global__ __launch_bounds__(256) void ladder_code_kernel(const float* __restrict__ coef, int n, int G,
                                                          const uint8_t* __restrict__ bits, int R,
                                                          const int64_t* __restrict__ level, float* __restrict__ decoded,
                                                          uint8_t* __restrict__ codes, uint16_t* __restrict__ low,
                                                          uint16_t* __restrict__ step) {
  const int per = (G + 3) / 4;  // waves per token
  const long wv = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const long t = wv / per;
  if (t >= n) return;
  const int j = lane & 15, g = (int)(wv % per) * 4 + (lane >> 4);
  const bool live = g < G;
  const long tg = t * G + (live ? g : G - 1);
  const float4 x = *((const float4*)coef + tg * 16 + j);
  const int64_t rung = level[t];
  const int width = rung >= 0 && rung < R ? bits[rung * G + (live ? g : G - 1)] : 0;
  const int b = width == 2 || width == 4 || width == 8 ? width : 0;
  const GroupRange r = group_range(x, lane);
  const float top = b == 2 ? 3.0f : b == 4 ? 15.0f : 255.0f;
  const half_t st = ladder_step(r, top);
  const float xv[4] = {x.x, x.y, x.z, x.w};
  float v[4];
  uint32_t packed = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float q = ladder_level(xv[i], (float)r.low, (float)st, top);
    v[i] = b > 0 ? level_value(q, (float)r.low, (float)st) : (rung == R ? xv[i] : 0.0f);
    packed |= (b > 0 ? (uint32_t)q & 0xffu : 0u) << (8 * i);
  }
  if (!live) return;
  *((float4*)decoded + tg * 16 + j) = make_float4(v[0], v[1], v[2], v[3]);
  *((uint32_t*)codes + tg * 16 + j) = packed;
  if (j == 0) {
    uint16_t lb = 0, sb = 0;
    if (b > 0) {
      __builtin_memcpy(&lb, &r.low, 2);
      __builtin_memcpy(&sb, &st, 2);
    }
    low[tg] = lb;
    step[tg] = sb;
  }
}

int check_bits(const float* coef, int32_t n, int32_t G, const uint8_t* bits, int32_t R, const char* what) {
  DKV_REQUIRE(n >= 0 && G > 0 && R > 0 && R <= 64 && (long)R * G <= 65536, DKV_ESHAPE, "%s: bad shape (n=%d groups=%d rungs=%d)",
              what, n, G, R);
  DKV_REQUIRE(n == 0 || (coef && bits), DKV_EINVAL, "%s: null pointer", what);
  DKV_REQUIRE((uintptr_t)coef % 16 == 0, DKV_EINVAL, "%s: coefficients must be 16-byte aligned", what);
  return DKV_OK;
}

// ---------------------------------------------------------------------------
// Token-matrix rows back into per-layer caches [1][H][tokens][D] (the inverse of centred rows, scripts/kvtc.py:
// from_matrix with :46-47 rerotate): row i is token first + i (+ gap_len from gap_start on), keys rotated to it.
// One thread per 4 columns, or per 4 pairs of keys, of a row.
// ---------------------------------------------------------------------------
template <int T>
DKV_DEVICE void store_elem4(void* base, long idx, const float (&v)[4]) {
  if constexpr (T == DKV_F32) {
    *(float4*)((float*)base + idx) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    uint16_t e[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (T == DKV_BF16) {
        e[i] = float_to_bf16_bits(v[i]);
      } else {
        const half_t h = (half_t)v[i];
        __builtin_memcpy(&e[i], &h, 2);
      }
    }
    *(uint2*)((uint16_t*)base + idx) = make_uint2(e[0] | (uint32_t)e[1] << 16, e[2] | (uint32_t)e[3] << 16);
  }
}

DKV_DEVICE float rotated(float x, float rh, float c, float s) {
#pragma clang fp contract(off)
  const float a = x * c, b = rh * s;
  return a + b;
}

template <int T, bool ROTATE>
__global__ __launch_bounds__(256) void rows_to_caches_kernel(const float* __restrict__ rows, int n, int first, int gap_start,
                                                             int gap_len, const uint64_t* __restrict__ layer_ptrs, int L,
                                                             int H, int tokens, int D, const float* __restrict__ cos,
                                                             const float* __restrict__ sin, int col_blocks) {
  const int W = ROTATE ? D / 8 : D / 4;
  const int c = (int)(blockIdx.x % col_blocks) * 256 + threadIdx.x;
  if (c >= L * H * W) return;
  const int i = (int)(blockIdx.x / col_blocks);
  int t = first + i;
  if (t >= gap_start) t += gap_len;
  const int lh = c / W, d = 4 * (c % W), half = D / 2;
  const float* src = rows + (long)i * L * H * D + (long)lh * D + d;
  void* base = (void*)layer_ptrs[lh / H];
  const long at = ((long)(lh % H) * tokens + t) * D + d;
  const float4 x = *(const float4*)src;
  const float xv[4] = {x.x, x.y, x.z, x.w};
  if constexpr (ROTATE) {
    const float4 y = *(const float4*)(src + half);
    const float4 c0 = *(const float4*)(cos + (long)t * D + d), c1 = *(const float4*)(cos + (long)t * D + d + half);
    const float4 s0 = *(const float4*)(sin + (long)t * D + d), s1 = *(const float4*)(sin + (long)t * D + d + half);
    const float yv[4] = {y.x, y.y, y.z, y.w};
    const float a0[4] = {c0.x, c0.y, c0.z, c0.w}, b0[4] = {s0.x, s0.y, s0.z, s0.w};
    const float a1[4] = {c1.x, c1.y, c1.z, c1.w}, b1[4] = {s1.x, s1.y, s1.z, s1.w};
    float lo[4], hi[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      lo[e] = rotated(xv[e], -yv[e], a0[e], b0[e]);
      hi[e] = rotated(yv[e], xv[e], a1[e], b1[e]);
    }
    store_elem4<T>(base, at, lo);
    store_elem4<T>(base, at + half, hi);
  } else {
    store_elem4<T>(base, at, xv);
  }
}

// The tokens outside [skip, skip + skip_len) of per-layer caches, copied as they are (16 bytes per thread).
__global__ __launch_bounds__(256) void copy_tokens_kernel(const uint64_t* __restrict__ src, const uint64_t* __restrict__ dst,
                                                          int layers, int H, int tokens, int row_words, int skip, int skip_len) {
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  const int outside = tokens - skip_len;
  const int w = (int)(e % row_words);
  const long r = e / row_words;
  const int i = (int)(r % outside);
  const long lh = r / outside;
  const int l = (int)(lh / H), h = (int)(lh % H);
  if (l >= layers) return;
  const long at = ((long)h * tokens + (i < skip ? i : i + skip_len)) * row_words + w;
  ((uint4*)dst[l])[at] = ((const uint4*)src[l])[at];
}

// Which groups some row uses (scripts/kvtc.py:88-97): live[g] = 1 where any row's 64 coefficients of group g are not all
// 0 (a NaN is not 0); live starts at 0.  CODES: the coefficients are code * scale + low of ladder codes, each operation
// rounded on its own (scripts/kvtc_storage.py:119), and are written on the way.  16 lanes per (row, group), four
// members each.  Bound by its bytes: 5,964 x 2,048 from codes 14 us, 4,061 x 2,048 of coefficients 8 (4.2 TB/s); torch took
// 56 us for the latter's reduction alone, and three passes more for the former's coefficients.
template <bool CODES>
__global__ __launch_bounds__(256) void live_groups_kernel(const uint8_t* __restrict__ codes, const uint16_t* __restrict__ low,
                                                          const uint16_t* __restrict__ scale, float* __restrict__ coef,
                                                          long ngroups, int G, int32_t* __restrict__ live) {
  const long tg = (long)blockIdx.x * 16 + (threadIdx.x >> 4);
  const int j = threadIdx.x & 15;
  const bool ok = tg < ngroups;
  const long at = (ok ? tg : 0) * 64 + 4 * j;
  float4 v;
  if constexpr (CODES) {
    uint32_t c;
    __builtin_memcpy(&c, codes + at, 4);
    const float s = half_bits_to_float(scale[ok ? tg : 0]), l = half_bits_to_float(low[ok ? tg : 0]);
    {
#pragma clang fp contract(off)
      v.x = (float)(c & 0xffu) * s + l;
      v.y = (float)((c >> 8) & 0xffu) * s + l;
      v.z = (float)((c >> 16) & 0xffu) * s + l;
      v.w = (float)(c >> 24) * s + l;
    }
    if (ok) *(float4*)(coef + at) = v;
  } else {
    v = *(const float4*)(coef + at);
  }
  const bool any = ok && (v.x != 0.0f || v.y != 0.0f || v.z != 0.0f || v.w != 0.0f);
  const unsigned long long row = __ballot(any) >> (threadIdx.x & 48) & 0xffffull;
  // one lane a group, and only until the flag is seen: every writer stores the same 1
  if (j == 0 && row != 0 && live[(int)(tg % G)] == 0) live[(int)(tg % G)] = 1;
}

// The same tokens gathered into one buffer [layers][H][tokens - skip_len][row], the layers' addresses in the launch's
// arguments.  A progressive encode's sinks and recent window (16 layers x 8 heads x 36 tokens of 128 bytes): one launch
// a stream in place of a concatenation a layer, 16 launches of 7.4 us.
constexpr int kLaunchLayers = 128;
struct LayerPtrs {
  const void* p[kLaunchLayers];
};

__global__ __launch_bounds__(256) void outside_tokens_kernel(LayerPtrs src, uint4* __restrict__ dst, long layer_words, int tokens,
                                                             int row_words, int skip, int skip_len) {
  const int l = blockIdx.y;
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= layer_words) return;
  const int outside = tokens - skip_len;
  const int w = (int)(e % row_words);
  const long r = e / row_words;
  const int i = (int)(r % outside);
  dst[l * layer_words + e] = ((const uint4*)src.p[l])[(r / outside * tokens + (i < skip ? i : i + skip_len)) * row_words + w];
}

}  // namespace

extern "C" int dkv_live_groups(const uint8_t* codes, const uint16_t* low, const uint16_t* scale, float* coef, int64_t n,
                               int32_t groups, int32_t* live, void* stream) {
  DKV_REQUIRE(n >= 0 && groups > 0 && n < (1L << 31), DKV_ESHAPE, "dkv_live_groups: bad shape (n=%ld groups=%d)", (long)n, groups);
  if (n == 0) return DKV_OK;
  DKV_REQUIRE(coef && live && (!codes || (low && scale)), DKV_EINVAL, "dkv_live_groups: null pointer");
  const long ngroups = (long)n * groups, blocks = (ngroups + 15) / 16;
  DKV_REQUIRE(blocks < (1L << 31), DKV_ESHAPE, "dkv_live_groups: too many rows");
  if (codes)
    hipLaunchKernelGGL(live_groups_kernel<true>, dim3((unsigned)blocks), dim3(256), 0, dkv::as_stream(stream), codes, low, scale,
                       coef, ngroups, groups, live);
  else
    hipLaunchKernelGGL(live_groups_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, dkv::as_stream(stream), codes, low, scale,
                       coef, ngroups, groups, live);
  return dkv::check_launch("dkv_live_groups");
}

extern "C" int dkv_outside_tokens(const uint64_t* layer_ptrs, void* out, int32_t dtype, int32_t layers, int32_t heads,
                                  int32_t tokens, int32_t head_dim, int32_t skip, int32_t skip_len, void* stream) {
  DKV_REQUIRE(dtype == DKV_F32 || dtype == DKV_F16 || dtype == DKV_BF16, DKV_EINVAL,
              "dkv_outside_tokens: dtype %d not supported", dtype);
  DKV_REQUIRE(layers > 0 && heads > 0 && tokens >= 0 && head_dim > 0 && head_dim % 8 == 0 && skip >= 0 && skip_len >= 0 &&
                  (long)skip + skip_len <= tokens,
              DKV_ESHAPE, "dkv_outside_tokens: bad shape (layers=%d heads=%d tokens=%d head_dim=%d skip=%d+%d)", layers, heads,
              tokens, head_dim, skip, skip_len);
  const int row_words = head_dim * (dtype == DKV_F32 ? 4 : 2) / 16;
  const long layer_words = (long)heads * (tokens - skip_len) * row_words;
  if (layer_words == 0) return DKV_OK;
  DKV_REQUIRE(layer_ptrs && out, DKV_EINVAL, "dkv_outside_tokens: null pointer");
  DKV_REQUIRE((layer_words + 255) / 256 < (1L << 31), DKV_ESHAPE, "dkv_outside_tokens: too many tokens");
  for (int l0 = 0; l0 < layers; l0 += kLaunchLayers) {
    LayerPtrs src{};
    const int n = layers - l0 < kLaunchLayers ? layers - l0 : kLaunchLayers;
    for (int l = 0; l < n; ++l) src.p[l] = (const void*)layer_ptrs[l0 + l];
    hipLaunchKernelGGL(outside_tokens_kernel, dim3((unsigned)((layer_words + 255) / 256), n), dim3(256), 0,
                       dkv::as_stream(stream), src, (uint4*)out + l0 * layer_words, layer_words, tokens, row_words, skip, skip_len);
    const int rc = dkv::check_launch("dkv_outside_tokens");
    if (rc) return rc;
  }
  return DKV_OK;
}

extern "C" int dkv_ladder_errors(const float* coef, int32_t n, int32_t groups, const uint8_t* bits, int32_t rungs,
                                 float* errors, void* stream) {
  int rc = check_bits(coef, n, groups, bits, rungs, "dkv_ladder_errors");
  if (rc) return rc;
  if (n == 0) return DKV_OK;
  DKV_REQUIRE(errors, DKV_EINVAL, "dkv_ladder_errors: null pointer");
  const dim3 grid((unsigned)((n + kErrorTok - 1) / kErrorTok)), block(kErrorTok * 64);
  const size_t lds = (size_t)rungs * groups;
  hipStream_t st = dkv::as_stream(stream);
  if (rungs <= 16)
    hipLaunchKernelGGL(ladder_errors_kernel<1>, grid, block, lds, st, coef, n, groups, bits, rungs, errors);
  else
    hipLaunchKernelGGL(ladder_errors_kernel<4>, grid, block, lds, st, coef, n, groups, bits, rungs, errors);
  return dkv::check_launch("dkv_ladder_errors");
}

extern "C" int dkv_ladder_code(const float* coef, int32_t n, int32_t groups, const uint8_t* bits, int32_t rungs,
                               const int64_t* level, float* decoded, uint8_t* codes, uint16_t* low, uint16_t* scale,
                               void* stream) {
  int rc = check_bits(coef, n, groups, bits, rungs, "dkv_ladder_code");
  if (rc) return rc;
  if (n == 0) return DKV_OK;
  DKV_REQUIRE(level && decoded && codes && low && scale, DKV_EINVAL, "dkv_ladder_code: null pointer");
  const long waves = (long)n * ((groups + 3) / 4), blocks = (waves + 3) / 4;
  DKV_REQUIRE(blocks < (1L << 31), DKV_ESHAPE, "dkv_ladder_code: too many tokens");
  hipLaunchKernelGGL(ladder_code_kernel, dim3((unsigned)blocks), dim3(256), 0, dkv::as_stream(stream), coef, n, groups, bits,
                     rungs, level, decoded, codes, low, scale);
  return dkv::check_launch("dkv_ladder_code");
}

extern "C" int dkv_rows_to_caches(const float* rows, int32_t n, int32_t first, int32_t gap_start, int32_t gap_len,
                                  const uint64_t* layer_ptrs, int32_t dtype, int32_t layers, int32_t heads, int32_t tokens,
                                  int32_t head_dim, const float* cos, const float* sin, void* stream) {
  DKV_REQUIRE((cos == nullptr) == (sin == nullptr), DKV_EINVAL, "dkv_rows_to_caches: cos and sin go together");
  DKV_REQUIRE(dtype == DKV_F32 || dtype == DKV_F16 || dtype == DKV_BF16, DKV_EINVAL,
              "dkv_rows_to_caches: dtype %d not supported", dtype);
  DKV_REQUIRE(n >= 0 && layers > 0 && heads > 0 && head_dim > 0 && head_dim % 8 == 0 &&
                  (long)layers * heads * head_dim < (1L << 30),
              DKV_ESHAPE, "dkv_rows_to_caches: bad shape (rows=%d layers=%d heads=%d head_dim=%d)", n, layers, heads,
              head_dim);
  const long last = (long)first + n - 1;
  DKV_REQUIRE(first >= 0 && gap_len >= 0 && last + (last >= gap_start ? gap_len : 0) < tokens, DKV_ESHAPE,
              "dkv_rows_to_caches: rows %d.. of %d end past %d tokens", first, n, tokens);
  if (n == 0) return DKV_OK;
  DKV_REQUIRE(rows && layer_ptrs, DKV_EINVAL, "dkv_rows_to_caches: null pointer");
  const long cols = (long)layers * heads * (head_dim / (cos ? 8 : 4)), col_blocks = (cols + 255) / 256;
  DKV_REQUIRE(col_blocks * n < (1L << 31), DKV_ESHAPE, "dkv_rows_to_caches: too many rows");
  const dim3 grid((unsigned)(col_blocks * n));
  hipStream_t st = dkv::as_stream(stream);
#define DKV_ROWS(T_, R_)                                                                                             \
  hipLaunchKernelGGL((rows_to_caches_kernel<T_, R_>), grid, dim3(256), 0, st, rows, n, first, gap_start, gap_len,    \
                     layer_ptrs, layers, heads, tokens, head_dim, cos, sin, (int)col_blocks)
  const bool rot = cos != nullptr;
  if (dtype == DKV_F16) {
    if (rot) DKV_ROWS(DKV_F16, true); else DKV_ROWS(DKV_F16, false);
  } else if (dtype == DKV_BF16) {
    if (rot) DKV_ROWS(DKV_BF16, true); else DKV_ROWS(DKV_BF16, false);
  } else {
    if (rot) DKV_ROWS(DKV_F32, true); else DKV_ROWS(DKV_F32, false);
  }
#undef DKV_ROWS
  return dkv::check_launch("dkv_rows_to_caches");
}

extern "C" int dkv_copy_tokens(const uint64_t* src_ptrs, const uint64_t* dst_ptrs, int32_t dtype, int32_t layers,
                               int32_t heads, int32_t tokens, int32_t head_dim, int32_t skip, int32_t skip_len, void* stream) {
  DKV_REQUIRE(dtype == DKV_F32 || dtype == DKV_F16 || dtype == DKV_BF16, DKV_EINVAL, "dkv_copy_tokens: dtype %d not supported",
              dtype);
  DKV_REQUIRE(layers > 0 && heads > 0 && tokens >= 0 && head_dim > 0 && head_dim % 8 == 0 && skip >= 0 && skip_len >= 0 &&
                  (long)skip + skip_len <= tokens,
              DKV_ESHAPE, "dkv_copy_tokens: bad shape (layers=%d heads=%d tokens=%d head_dim=%d skip=%d+%d)", layers, heads,
              tokens, head_dim, skip, skip_len);
  const int row_words = head_dim * (dtype == DKV_F32 ? 4 : 2) / 16;
  const long total = (long)layers * heads * (tokens - skip_len) * row_words;
  if (total == 0) return DKV_OK;
  DKV_REQUIRE(src_ptrs && dst_ptrs, DKV_EINVAL, "dkv_copy_tokens: null pointer");
  DKV_REQUIRE((total + 255) / 256 < (1L << 31), DKV_ESHAPE, "dkv_copy_tokens: too many tokens");
  hipLaunchKernelGGL(copy_tokens_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, dkv::as_stream(stream), src_ptrs,
                     dst_ptrs, layers, heads, tokens, row_words, skip, skip_len);
  return dkv::check_launch("dkv_copy_tokens");
}
