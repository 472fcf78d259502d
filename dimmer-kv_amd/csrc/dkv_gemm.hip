// float32 matrix products on the fp16 matrix cores, for the codecs' projections onto the PCA basis and
// back (scripts/kvtc.py:88-97 inverse_transform and the projections of scripts/kvtc.py:189 and
// scripts/progressive.py:147-148, which the reference leaves to a float32 library product).
//
//   C[m][n] = sum_k A[m][k] B[n][k] (+ bias[n]),
//
// every operand element split into two fp16 pieces, x * 2^s = hi + lo with s from the row's largest
// magnitude, and the products hi hi + hi lo + lo hi summed in fp32.  hi + lo holds x to 2^-22 of itself down to 2^-17
// of its row's maximum and to 2^-39 of that maximum below (lo is then subnormal), the dropped lo lo is at most
// 2^-22 of a product, and the sums are 16 products wide, so the result lies closer to float64 than the float32
// library product does (its error is the fp32 accumulation of thousands of terms) wherever a row's elements
// that matter are within about 2^18 of each other.  A row whose result comes from elements further below its maximum,
// the maximum meeting zeros, keeps fewer bits: at K = 2,048 a relative error of 7.5e-7 with one element 2^20 above the
// others, 2.5e-6 with 2^22, 1.2e-5 with 2^24, against float32's 3.7e-7.
//
// Three fp16 products run at a third of the fp16 rate (about 1.4 PFLOP/s here), against 0.15 PFLOP/s of
// the float32 matrix instructions.  16,348 x 2,048 x 28,672 (the projection of a 16K-token 3B cache): 5,190 us
// with the splitting, 1.11 PFLOP/s of fp16 products, against 12,440 us of the library's float32 product (5,090 to 5,230
// straight from the caches, with the 627 us of their centred rows in it);
// 4,061 x 28,672 x 2,048 (back): 1,295 against 3,500 us.  Error against float64 2.0e-6 and 5.0e-7, against the
// library's 3.0e-6 and 8.1e-7.
#include <hip/hip_runtime.h>
#include <limits.h>

#include <algorithm>
#include <type_traits>

#include "dkv_device.h"
#include "dkv_host.h"

namespace {

// ---------------------------------------------------------------------------
// Split operands.  Rows are padded to whole 256-row tiles and K to whole pairs of 32-component blocks (zeros).
// One (row, 32-component block) is one 128-byte line of eight 16-byte pieces: hi of octets 0..3, lo of
// octets 0..3 (an octet is 8 consecutive k), piece i stored at i ^ (row & 7).  The lines of 32 rows are
// consecutive (4 KB), then the blocks along k, then the 32-row blocks.  A copy of a 4 KB block into LDS
// keeps this order, and the swizzle puts the eight lanes of a quarter of a 16-byte LDS read (eight
// consecutive rows, one octet) on distinct banks.
// ---------------------------------------------------------------------------
constexpr int kTile = 256;         // rows of A, and of B, per workgroup
constexpr int kLine = 128;         // bytes of one (row, 32-component block)
constexpr int kBlock = 32 * kLine; // bytes of one (32 rows, 32 components)
constexpr int kStage = 2 * 8 * kBlock;  // bytes of one stage: 256 rows of A and of B, 32 components
constexpr int kFlagged = INT_MIN;  // in place of the exponent of a row that holds an infinity or a NaN: its pieces are zeros

// Such rows of an operand, in any order: special_kernel's work.
struct Flagged {
  int* count;
  int* list;
  DKV_DEVICE void add(int row) const { list[atomicAdd(count, 1)] = row; }
};

inline long pad_to(long x, long m) { return (x + m - 1) / m * m; }

DKV_DEVICE long line_offset(long row, int kb, int KB) { return ((row >> 5) * KB + kb) * kBlock + (row & 31) * kLine; }

// The exponent s that takes a row whose largest magnitude has the bits `top` to [2^14, 2^15).
DKV_DEVICE int row_shift(uint32_t top) {
  if (top >= 0x7f800000u) return kFlagged;
  if (top == 0) return 0;
  const int e = top >= 0x00800000u ? (int)(top >> 23) - 127 : -118 - __clz(top);  // floor(log2)
  return 14 - e;
}

// Eight scaled floats -> their hi and lo pieces.
DKV_DEVICE void split8(const float (&x)[8], int shift, half8& hi, half8& lo) {
  if (shift == kFlagged) {
    hi = lo = half8{0, 0, 0, 0, 0, 0, 0, 0};
    return;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float v = __builtin_ldexpf(x[i], shift);
    const half_t h = (half_t)v;
    hi[i] = h;
    lo[i] = (half_t)(v - (float)h);
  }
}

DKV_DEVICE void store_octet(uint8_t* out, long row, int oct, int KB, const half8& hi, const half8& lo) {
  uint8_t* line = out + line_offset(row, oct >> 2, KB);
  const int r7 = (int)(row & 7), o = oct & 3;
  *(half8*)(line + ((o ^ r7) << 4)) = hi;
  *(half8*)(line + (((4 + o) ^ r7) << 4)) = lo;
}

DKV_DEVICE uint32_t abs_bits(float v) { return __float_as_uint(v) & 0x7fffffffu; }

__global__ __launch_bounds__(256) void clear_kernel(uint32_t* __restrict__ p, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// One workgroup per (padded) row of a row-major [rows][K] source.  A row of up to NT * OCT * 8 elements
// stays in registers between its maximum and its split (one read of the source); a longer row is read twice.
template <int NT, int OCT, bool VEC>
__global__ __launch_bounds__(NT) void split_rows_kernel(const float* __restrict__ src, long ld, int rows, int K, int KB,
                                                        uint8_t* __restrict__ out, int* __restrict__ shifts,
                                                        Flagged flagged) {
  __shared__ uint32_t wtop[NT / 64];
  const int tid = threadIdx.x;
  const long row = blockIdx.x;
  const bool live = row < rows;
  const float* r = src + (live ? row : 0) * ld;
  auto load = [&](int oct, float (&x)[8]) {
    const int k = oct * 8;
    if (VEC && live && k + 8 <= K) {
      const float4 a = *(const float4*)(r + k), b = *(const float4*)(r + k + 4);
      x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w; x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = live && k + i < K ? r[k + i] : 0.0f;
    }
  };
  float x[OCT][8];
  uint32_t top = 0;
#pragma unroll
  for (int j = 0; j < OCT; ++j) load(tid + j * NT, x[j]);
#pragma unroll
  for (int j = 0; j < OCT; ++j)
#pragma unroll
    for (int i = 0; i < 8; ++i) top = max(top, abs_bits(x[j][i]));
  const int octs = KB * 4;
  for (int o = tid + OCT * NT; o < octs; o += NT) {
    float y[8];
    load(o, y);
#pragma unroll
    for (int i = 0; i < 8; ++i) top = max(top, abs_bits(y[i]));
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) top = max(top, (uint32_t)__shfl_xor((int)top, o));
  if ((tid & 63) == 0) wtop[tid >> 6] = top;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) top = max(top, wtop[w]);
  const int shift = row_shift(top);
  if (tid == 0) {
    shifts[row] = shift == kFlagged ? 0 : shift;
    if (shift == kFlagged) flagged.add((int)row);
  }
  half8 hi, lo;
#pragma unroll
  for (int j = 0; j < OCT; ++j) {
    const int o = tid + j * NT;
    if (o >= octs) break;
    split8(x[j], shift, hi, lo);
    store_octet(out, row, o, KB, hi, lo);
  }
  for (int o = tid + OCT * NT; o < octs; o += NT) {
    float y[8];
    load(o, y);
    split8(y, shift, hi, lo);
    store_octet(out, row, o, KB, hi, lo);
  }
}

// Column maxima (as magnitude bits) of a row-major [K][N] source: a workgroup takes 64 columns of 128 rows.
__global__ __launch_bounds__(256) void column_top_kernel(const float* __restrict__ src, long ld, int K, int N,
                                                         uint32_t* __restrict__ top) {
  __shared__ uint32_t part[4][64];
  const int c = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int nb = (N + 63) / 64;  // column blocks, fastest in the grid
  const int n = (int)(blockIdx.x % nb) * 64 + c, k0 = (int)(blockIdx.x / nb) * 128;
  uint32_t t = 0;
  if (n < N)
#pragma unroll 8
    for (int k = k0 + w; k < min(k0 + 128, K); k += 4) t = max(t, abs_bits(src[(long)k * ld + n]));
  part[w][c] = t;
  __syncthreads();
  if (w == 0 && n < N) atomicMax(&top[n], max(max(part[0][c], part[1][c]), max(part[2][c], part[3][c])));
}

// The columns of a row-major [K][N] source as split rows: a workgroup turns 64 columns x 32 components.
__global__ __launch_bounds__(256) void split_columns_kernel(const float* __restrict__ src, long ld, int K, int N, int KB,
                                                            const uint32_t* __restrict__ top, uint8_t* __restrict__ out,
                                                            int* __restrict__ shifts, Flagged flagged) {
  __shared__ float t[32][65];
  const int tid = threadIdx.x;
  const int nb = gridDim.x / KB;  // column blocks, fastest in the grid
  const int n0 = (int)(blockIdx.x % nb) * 64, kb = (int)(blockIdx.x / nb);
  const int c = tid & 63, w = tid >> 6;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int k = kb * 32 + w + 4 * i;
    t[w + 4 * i][c] = n0 + c < N && k < K ? src[(long)k * ld + n0 + c] : 0.0f;
  }
  __syncthreads();
  const int nl = tid >> 2, o = tid & 3;
  const long n = n0 + nl;
  const int shift = row_shift(n < N ? top[n] : 0u);
  float x[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = t[8 * o + i][nl];
  half8 hi, lo;
  split8(x, shift, hi, lo);
  store_octet(out, n, 4 * kb + o, KB, hi, lo);
  if (kb == 0 && o == 0) {
    shifts[n] = shift == kFlagged ? 0 : shift;
    if (shift == kFlagged) flagged.add((int)n);
  }
}

// ---------------------------------------------------------------------------
// The product.  A workgroup takes a 256 x 256 tile of C over a range of 32-component blocks; wave (wm,
// wn) of the 4 x 2 takes 64 rows x 128 columns as 2 x 4 accumulators of 32 x 32.  A stage (32 components
// of 256 rows of A and B, hi and lo: 64 KB) is copied straight into one of two LDS buffers
// (global_load_lds, 1 KB per wave instruction) while the stage before is multiplied.
//
// What bounds it is the matrix pipe: per stage and wave 48 MFMAs (1,536 cycles; two waves per SIMD, so
// 3,072) against 64 KB of copies (about 1,800 cycles of a CU's load path) and 24 16-byte LDS operand
// reads per wave (192 KB per CU, about 1,500 cycles).  Three products per pair of operand fragments is what
// buys that balance: a plain fp16 product of this tile would do one.
//
// The operands of a 16-component step are read while the step before is multiplied, across the stage
// boundary too: a stage's copy is awaited, and its barrier stands, between the two steps of the stage
// before, so the matrix pipe has a full step in hand at every barrier.  (238 registers, none spilled; as the
// compiler orders it by itself, the reads stand behind the products they should run beside.)  16,348 x 2,048 x
// 28,672: 4,380 us in this kernel, 1.31 PFLOP/s; the library's plain fp16 product reaches 1.41 on 8,192^3 here.
// ---------------------------------------------------------------------------
struct GemmArgs {
  const uint8_t* a;  // split operands
  const uint8_t* b;
  const int* sa;     // their exponents
  const int* sb;
  const float* bias; // [N] or null
  float* c;          // [M][ldc], or with several splits the partial sums [splits][M][N]
  long ldc;
  int M, N, KB;      // K in 32-component blocks
  int mt, nt;        // tiles
  int splits, per_split;  // k ranges of per_split blocks
  int total, per_xcd;
};

typedef half8 Frag;

__global__ __launch_bounds__(512, 2) void gemm_split_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(1024))) uint8_t S0[kStage];
  __shared__ __attribute__((aligned(1024))) uint8_t S1[kStage];
  // consecutive workgroup indices of an XCD: bands of 8 row tiles, down the band first, so that the 32 tiles
  // it has in flight are about 8 x 4 and share their operands through its L2
  const int lin = (blockIdx.x & 7) * g.per_xcd + (blockIdx.x >> 3);
  if (lin >= g.total) return;
  const int tiles = g.mt * g.nt;
  const int z = lin / tiles, t = lin % tiles;
  const int band = t / (8 * g.nt);
  const int bm = min(8, g.mt - band * 8);
  const int ti = t - band * 8 * g.nt;
  const int tm = band * 8 + ti % bm, tn = ti / bm;
  const int kb0 = z * g.per_split, kb1 = min(g.KB, kb0 + g.per_split);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: the copies' LDS targets are scalar
  const int wm = wave & 3, wn = wave >> 2;
  const int l32 = lane & 31, lhi = lane >> 5;

  // this wave copies 32-row block `wave` of A and of B
  const uint8_t* ga = g.a + (long)(tm * 8 + wave) * g.KB * kBlock;
  const uint8_t* gb = g.b + (long)(tn * 8 + wave) * g.KB * kBlock;
  const uint32_t lane16 = lane * 16;
  auto copy = [&](int kb, uint8_t* S) {
    const uint8_t* pa = ga + (long)kb * kBlock;
    const uint8_t* pb = gb + (long)kb * kBlock;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_global_load_lds(pa + i * 1024 + lane16, S + wave * kBlock + i * 1024, 16, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_global_load_lds(pb + i * 1024 + lane16, S + 8 * kBlock + wave * kBlock + i * 1024, 16, 0, 0);
  };

  floatx16 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  // operand reads: piece (hl * 4 + step * 2 + lhi) ^ (row & 7) of the lane's row
  const int arow = (wm * 64 + l32) * kLine, brow = 8 * kBlock + (wn * 128 + l32) * kLine;
  const int p0 = lhi ^ (l32 & 7);
  struct Operands {
    Frag a[2][2], b[2][4];  // [hi, lo][32-row block]
  };
  auto read = [&](const uint8_t* S, int step, Operands& f) {
#pragma unroll
    for (int hl = 0; hl < 2; ++hl) {
      const int off = (p0 ^ (hl * 4 + step * 2)) << 4;
#pragma unroll
      for (int i = 0; i < 2; ++i) f.a[hl][i] = *(const Frag*)(S + arow + off + i * kBlock);
#pragma unroll
      for (int j = 0; j < 4; ++j) f.b[hl][j] = *(const Frag*)(S + brow + off + j * kBlock);
    }
  };
  auto multiply = [&](const Operands& f) {
#pragma unroll
    for (int p = 0; p < 3; ++p) {  // hi lo, lo hi, then hi hi
      const int ah = p == 1, bh = p == 0;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[ah][i], f.b[bh][j], acc[i][j], 0, 0, 0);
    }
  };
  // the copy of the next stage has landed and this stage's operand reads are done, in every wave
  auto meet = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  Operands f0, f1;
  // Stage kb in S (next: the other buffer).  In: f0 holds step 0 of this stage, the copy of stage kb + 1 into
  // `next` is under way.  COPY: stage kb + 2 exists; NEXT: stage kb + 1 does.  The scheduling groups spread the
  // reads and copies over the first products of a step (left alone the compiler puts them behind the products).
  auto stage = [&](int kb, uint8_t* S, uint8_t* next, auto copy_t, auto next_t) {
    constexpr bool COPY = decltype(copy_t)::value, NEXT = decltype(next_t)::value;
    read(S, 1, f1);
    multiply(f0);
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
    for (int i = 0; i < 12; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 11, 0);
    __builtin_amdgcn_sched_barrier(0);
    meet();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (COPY) copy(kb + 2, S);
    if constexpr (NEXT) read(next, 0, f0);
    multiply(f1);
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if constexpr (NEXT) {
#pragma unroll
      for (int i = 0; i < 12; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
    }
    if constexpr (COPY) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);  // copy
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 23 - (NEXT ? 12 : 0) - (COPY ? 8 : 0), 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  using T = std::true_type;
  using F = std::false_type;
  copy(kb0, S0);
  copy(kb0 + 1, S1);
  meet();
  read(S0, 0, f0);
  int kb = kb0;
  for (; kb + 2 < kb1; kb += 2) {  // an even number of stages (gemm_layout)
    stage(kb, S0, S1, T{}, T{});
    stage(kb + 1, S1, S0, T{}, T{});
  }
  stage(kb, S0, S1, F{}, T{});
  stage(kb + 1, S1, S0, F{}, F{});

  // acc[i][j][v]: row tm*256 + wm*64 + i*32 + 8*(v/4) + 4*lhi + (v&3), column tn*256 + wn*128 + j*32 + l32
  const bool part = g.splits > 1;
  float* c = part ? g.c + (long)z * g.M * g.N : g.c;
  const long ldc = part ? g.N : g.ldc;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = tn * kTile + wn * 128 + j * 32 + l32;
    if (n >= g.N) continue;
    const int sb = g.sb[n];
    const float bias = !part && g.bias ? g.bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = tm * kTile + wm * 64 + i * 32 + 8 * (v >> 2) + 4 * lhi + (v & 3);
        if (m >= g.M) continue;
        c[(long)m * ldc + n] = __builtin_ldexpf(acc[i][j][v], -(g.sa[m] + sb)) + bias;
      }
  }
}

// The k ranges' partial sums added in order.
__global__ __launch_bounds__(256) void sum_splits_kernel(const float* __restrict__ part, int splits, int M, int N,
                                                         const float* __restrict__ bias, float* __restrict__ c, long ldc) {
  const long e = (long)blockIdx.x * 256 + threadIdx.x, total = (long)M * N;
  if (e >= total) return;
  float s = 0.0f;
  for (int z = 0; z < splits; ++z) s += part[(long)z * total + e];
  const int n = (int)(e % N);
  c[(e / N) * ldc + n] = s + (bias ? bias[n] : 0.0f);
}

// A's rows as special_kernel reads them: as they lie, or a token's centred row from the caches.
struct PlainRows {
  const float* a;
  long lda;
  DKV_DEVICE float at(long m, int k) const { return a[m * lda + k]; }
};

template <int T>
DKV_DEVICE float load_elem(const void* base, long idx) {
  if constexpr (T == DKV_F32) return ((const float*)base)[idx];
  const uint16_t b = ((const uint16_t*)base)[idx];
  return T == DKV_BF16 ? bf16_bits_to_float(b) : half_bits_to_float(b);
}

template <int T>
DKV_DEVICE void load_elem8(const void* base, long idx, float (&x)[8]) {
  if constexpr (T == DKV_F32) {
    const float4 a = *(const float4*)((const float*)base + idx), b = *(const float4*)((const float*)base + idx + 4);
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w; x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
  } else {
    const uint4 w = *(const uint4*)((const uint16_t*)base + idx);
    const uint32_t e[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint16_t lo = (uint16_t)(e[i] & 0xffffu), hi = (uint16_t)(e[i] >> 16);
      x[2 * i] = T == DKV_BF16 ? bf16_bits_to_float(lo) : half_bits_to_float(lo);
      x[2 * i + 1] = T == DKV_BF16 ? bf16_bits_to_float(hi) : half_bits_to_float(hi);
    }
  }
}

struct CacheArgs {
  const uint64_t* layer_ptrs;
  const float* cos;  // with sin: keys, de-rotated
  const float* sin;
  const float* mean;
  int H, tokens, D, start, K;
};

template <int T, bool ROTATE>
struct CacheRows {
  CacheArgs c;
  DKV_DEVICE float at(long m, int f) const {
    const int lh = f / c.D, d = f % c.D, half = c.D / 2;
    const long t = c.start + m, row = ((long)(lh % c.H) * c.tokens + t) * c.D;
    const void* base = (const void*)c.layer_ptrs[lh / c.H];
    const float x = load_elem<T>(base, row + d);
    if constexpr (!ROTATE) return x - c.mean[f];
    const float y = load_elem<T>(base, row + (d < half ? d + half : d - half));
    return derotated(x, d < half ? -y : y, c.cos[t * c.D + d], c.sin[t * c.D + d], c.mean[f]);
  }
};

// The split form of the middle tokens' centred rows (centered_rows_kernel's arithmetic, then split_rows_kernel's)
// straight from the caches: a workgroup keeps a token's whole row in registers, 16 elements a unit (8 at d and the 8
// at d + D / 2 that rotate with them), so neither the rows nor a second read of them exist.  `energy`, when given,
// gets the row's sum of squares.  Bound by the lines it writes (4 bytes an element) beside the 2 it reads: 16,348 keys
// of 28,672 columns take 793 us, 3.5 TB/s (the two kernels 627 and 715; 878 with 1,024 threads, a single workgroup on a
// CU), 8,155 of 8,192 columns 116 against 84 and 95.
template <int T, bool ROTATE, int NT, int U>
__global__ __launch_bounds__(NT, NT == 512 ? 4 : 1) void split_caches_kernel(CacheArgs c, int rows, int KB, uint8_t* __restrict__ out,
                                                          int* __restrict__ shifts, Flagged flagged,
                                                          float* __restrict__ energy) {
  __shared__ uint32_t wtop[NT / 64];
  __shared__ float wsum[NT / 64];
  const int tid = threadIdx.x;
  const long row = blockIdx.x;
  const bool live = row < rows;
  const long t = c.start + (live ? row : 0);
  const int per_head = c.D / 16, half = c.D / 2, units = c.K / 16;
  float x[U][2][8];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int unit = min(tid + u * NT, units - 1);
    const int lh = unit / per_head, d = 8 * (unit % per_head);
    const void* base = (const void*)c.layer_ptrs[lh / c.H];
    const long at = ((long)(lh % c.H) * c.tokens + t) * c.D + d;
    load_elem8<T>(base, at, x[u][0]);
    load_elem8<T>(base, at + half, x[u][1]);
  }
  uint32_t top = 0;
  float sum = 0.0f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int unit = min(tid + u * NT, units - 1);
    const int f = unit / per_head * c.D + 8 * (unit % per_head), d = 8 * (unit % per_head);
    float m0[8], m1[8];
    load_elem8<DKV_F32>(c.mean, f, m0);
    load_elem8<DKV_F32>(c.mean, f + half, m1);
    if constexpr (ROTATE) {
      float c0[8], s0[8], c1[8], s1[8];
      load_elem8<DKV_F32>(c.cos, t * c.D + d, c0);
      load_elem8<DKV_F32>(c.sin, t * c.D + d, s0);
      load_elem8<DKV_F32>(c.cos, t * c.D + d + half, c1);
      load_elem8<DKV_F32>(c.sin, t * c.D + d + half, s1);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float a = x[u][0][i], b = x[u][1][i];
        x[u][0][i] = derotated(a, -b, c0[i], s0[i], m0[i]);
        x[u][1][i] = derotated(b, a, c1[i], s1[i], m1[i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        x[u][0][i] -= m0[i];
        x[u][1][i] -= m1[i];
      }
    }
    const bool mine = live && tid + u * NT < units;
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        x[u][e][i] = mine ? x[u][e][i] : 0.0f;
        top = max(top, abs_bits(x[u][e][i]));
        sum = __builtin_fmaf(x[u][e][i], x[u][e][i], sum);
      }
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    top = max(top, (uint32_t)__shfl_xor((int)top, o));
    sum += __shfl_xor(sum, o);
  }
  if ((tid & 63) == 0) {
    wtop[tid >> 6] = top;
    wsum[tid >> 6] = sum;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) top = max(top, wtop[w]);
  const int shift = row_shift(top);
  if (tid == 0) {
    shifts[row] = shift == kFlagged ? 0 : shift;
    if (shift == kFlagged) flagged.add((int)row);
    if (energy && live) {
      float s = 0.0f;
#pragma unroll
      for (int w = 0; w < NT / 64; ++w) s += wsum[w];
      energy[row] = s;
    }
  }
  half8 hi, lo;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int unit = tid + u * NT;
    if (unit >= units) break;
    const int oct = unit / per_head * (c.D / 8) + unit % per_head;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      split8(x[u][e], shift, hi, lo);
      store_octet(out, row, oct + e * (half / 8), KB, hi, lo);
    }
  }
  const half8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int o = c.K / 8 + tid; o < KB * 4; o += NT) store_octet(out, row, o, KB, zero, zero);
}

// Outputs of flagged rows.  One element that is not finite makes every output of its row infinite or NaN, whatever the
// finite terms are, so those are left out (zeros in the product above): a workgroup takes a flagged row of A (or of B),
// lists its elements that are not finite, 2,048 components at a time, and adds their products with every row of B (of A).
// A term of two such elements may be added from both sides, which changes nothing.  With nothing flagged every workgroup
// ends at once.  16,348 x 2,048 x 28,672, 4,945 us with nothing flagged: 4,961 with a flagged row, 5,060 with a flagged
// column, 4,376 with a NaN in every row (zeros are faster to multiply); from the caches, 5,054 us: 6,388 with an infinite
// channel of every token.
constexpr int kSpecialList = 2048;
constexpr int kSpecialGrid = 1024;  // workgroups at most

template <class Rows>
__global__ __launch_bounds__(256) void special_kernel(Rows a, const float* __restrict__ b, long ldb, int b_kn, int M, int N,
                                                      int K, const int* __restrict__ counts, const int* __restrict__ listed_a,
                                                      const int* __restrict__ listed_b, float* __restrict__ c, long ldc) {
  __shared__ int at[kSpecialList];
  __shared__ float value[kSpecialList];
  __shared__ int found;
  const int tid = threadIdx.x, na = counts[0], nb = counts[1];
  auto b_at = [&](int n, int k) { return b_kn ? b[(long)k * ldb + n] : b[(long)n * ldb + k]; };
  for (int it = blockIdx.x; it < na + nb; it += gridDim.x) {
    const bool of_a = it < na;
    const int row = of_a ? listed_a[it] : listed_b[it - na], others = of_a ? N : M;
    bool open = true;  // some output of this row is not NaN yet, as far as this workgroup knows
    for (int k0 = 0; k0 < K && open; k0 += kSpecialList) {
      float x[kSpecialList / 256];
#pragma unroll
      for (int i = 0; i < kSpecialList / 256; ++i) {
        const int k = min(k0 + tid + 256 * i, K - 1);
        x[i] = of_a ? a.at(row, k) : b_at(row, k);
      }
      __syncthreads();  // the segment before is added
      if (tid == 0) found = 0;
      __syncthreads();
#pragma unroll
      for (int i = 0; i < kSpecialList / 256; ++i) {
        const int k = k0 + tid + 256 * i;
        if (k < K && abs_bits(x[i]) >= 0x7f800000u) {
          const int j = atomicAdd(&found, 1);
          at[j] = k;
          value[j] = x[i];
        }
      }
      __syncthreads();
      const int count = found;
      if (count == 0) continue;
      bool mine = false;
      for (int o = tid; o < others; o += 256) {
        float s = 0.0f;
        for (int j = 0; j < count && s == s; ++j) s += value[j] * (of_a ? b_at(o, at[j]) : a.at(o, at[j]));
        atomicAdd(&c[of_a ? row * ldc + o : o * ldc + row], s);
        mine |= s == s;
      }
      open = __syncthreads_or(mine);
    }
  }
}

struct GemmLayout {
  int KB, mt, nt, splits, per_split;
  size_t a, b, sa, sb, top, listed, part, total;  // top: the column maxima and, after them, the flagged rows' counts
};

constexpr int kGemmCUs = 256;

GemmLayout gemm_layout(long M, long N, long K) {
  GemmLayout L{};
  L.KB = (int)(pad_to(K, 64) / 32);
  L.mt = (int)(pad_to(M, kTile) / kTile);
  L.nt = (int)(pad_to(N, kTile) / kTile);
  // Products whose tiles leave CUs idle are cut along k, as long as a cut keeps 16 blocks (its copies and
  // the extra pass over the partial sums stay small beside its products).
  const long tiles = (long)L.mt * L.nt;
  L.splits = (int)std::max(1L, std::min(kGemmCUs / std::max(1L, tiles), (long)L.KB / 16));
  L.per_split = (int)pad_to((L.KB + L.splits - 1) / L.splits, 2);
  L.splits = (L.KB + L.per_split - 1) / L.per_split;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += (bytes + 255) & ~(size_t)255;
    return at;
  };
  L.a = take((size_t)L.mt * kTile * L.KB * kLine);
  L.b = take((size_t)L.nt * kTile * L.KB * kLine);
  L.sa = take((size_t)L.mt * kTile * 4);
  L.sb = take((size_t)L.nt * kTile * 4);
  L.top = take((size_t)(N + 2) * 4);
  L.listed = take((size_t)(M + N) * 4);  // the flagged rows of A, then of B
  L.part = take(L.splits > 1 ? (size_t)L.splits * M * N * 4 : 0);
  L.total = off;
  return L;
}

void launch_split_rows(const float* src, long ld, long rows, long rows_pad, int K, int KB, uint8_t* out, int* shifts,
                       Flagged flagged, hipStream_t st) {
  const bool vec = ld % 4 == 0 && (uintptr_t)src % 16 == 0;
  const dim3 grid((unsigned)rows_pad);
#define DKV_SPLIT(NT_, OCT_)                                                                                        \
  do {                                                                                                              \
    if (vec)                                                                                                        \
      hipLaunchKernelGGL((split_rows_kernel<NT_, OCT_, true>), grid, dim3(NT_), 0, st, src, ld, (int)rows, K, KB,   \
                         out, shifts, flagged);                                                                     \
    else                                                                                                            \
      hipLaunchKernelGGL((split_rows_kernel<NT_, OCT_, false>), grid, dim3(NT_), 0, st, src, ld, (int)rows, K, KB,  \
                         out, shifts, flagged);                                                                     \
  } while (0)
  if (KB * 4 <= 256)
    DKV_SPLIT(256, 1);
  else
    DKV_SPLIT(1024, 4);
#undef DKV_SPLIT
}

int check_gemm(int64_t M, int64_t N, int64_t K, const char* what) {
  DKV_REQUIRE(M > 0 && N > 0 && K > 0 && M < (1L << 24) && N < (1L << 24) && K < (1L << 24), DKV_ESHAPE,
              "%s: bad shape (M=%ld N=%ld K=%ld)", what, (long)M, (long)N, (long)K);
  const GemmLayout L = gemm_layout(M, N, K);
  DKV_REQUIRE((long)L.mt * L.nt * L.splits < (1L << 28) && (long)L.nt * (kTile / 64) * L.KB < (1L << 31) && M * N < (1L << 38),
              DKV_ESHAPE, "%s: too many tiles", what);
  return DKV_OK;
}

}  // namespace

extern "C" size_t dkv_matmul_f32_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (check_gemm(M, N, K, "dkv_matmul_f32_workspace_bytes")) return 0;
  return gemm_layout(M, N, K).total;
}

namespace {

// The product of A's split rows, once `split_a` has launched their split into the workspace.
template <class Rows, class SplitA>
int launch_product(const char* what, Rows rows, SplitA&& split_a, const float* b, long ldb, int b_is_kn, const float* bias, long M,
                   long N, long K, float* c, long ldc, void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_gemm(M, N, K, what);
  if (rc) return rc;
  DKV_REQUIRE(ldb >= (b_is_kn ? N : K) && ldc >= N, DKV_ESHAPE, "%s: bad row strides", what);
  const GemmLayout L = gemm_layout(M, N, K);
  DKV_REQUIRE(workspace && workspace_bytes >= L.total, DKV_EWORKSPACE, "%s: workspace %zu B < required %zu B", what,
              workspace_bytes, L.total);
  uint8_t* ws = (uint8_t*)workspace;
  hipStream_t st = dkv::as_stream(stream);
  int *sa = (int*)(ws + L.sa), *sb = (int*)(ws + L.sb);
  uint32_t* top = (uint32_t*)(ws + L.top);
  int *counts = (int*)(top + N), *listed = (int*)(ws + L.listed);
  hipLaunchKernelGGL(clear_kernel, dim3((unsigned)((N + 2 + 255) / 256)), dim3(256), 0, st, top, (int)N + 2);
  split_a(L, ws + L.a, sa, Flagged{counts, listed}, st);
  const Flagged flagged{counts + 1, listed + M};
  if (b_is_kn) {
    hipLaunchKernelGGL(column_top_kernel, dim3((unsigned)((N + 63) / 64 * ((K + 127) / 128))), dim3(256), 0, st, b,
                       ldb, (int)K, (int)N, top);
    hipLaunchKernelGGL(split_columns_kernel, dim3((unsigned)((long)L.nt * (kTile / 64) * L.KB)), dim3(256), 0, st, b, ldb,
                       (int)K, (int)N, L.KB, top, ws + L.b, sb, flagged);
  } else {
    launch_split_rows(b, ldb, N, (long)L.nt * kTile, (int)K, L.KB, ws + L.b, sb, flagged, st);
  }
  rc = dkv::check_launch(what);
  if (rc) return rc;
  GemmArgs g{};
  g.a = ws + L.a;
  g.b = ws + L.b;
  g.sa = sa;
  g.sb = sb;
  g.bias = bias;
  g.c = L.splits > 1 ? (float*)(ws + L.part) : c;
  g.ldc = ldc;
  g.M = (int)M;
  g.N = (int)N;
  g.KB = L.KB;
  g.mt = L.mt;
  g.nt = L.nt;
  g.splits = L.splits;
  g.per_split = L.per_split;
  g.total = L.mt * L.nt * L.splits;
  g.per_xcd = (g.total + 7) / 8;
  hipLaunchKernelGGL(gemm_split_kernel, dim3(8u * (unsigned)g.per_xcd), dim3(512), 0, st, g);
  rc = dkv::check_launch(what);
  if (rc) return rc;
  if (L.splits > 1)
    hipLaunchKernelGGL(sum_splits_kernel, dim3((unsigned)((M * N + 255) / 256)), dim3(256), 0, st,
                       (const float*)(ws + L.part), L.splits, (int)M, (int)N, bias, c, ldc);
  hipLaunchKernelGGL(special_kernel<Rows>, dim3((unsigned)std::min(M + N, (long)kSpecialGrid)), dim3(256), 0, st, rows, b,
                     ldb, b_is_kn, (int)M, (int)N, (int)K, counts, listed, listed + M, c, ldc);
  return dkv::check_launch(what);
}

template <int T, bool ROTATE>
int launch_project(const CacheArgs& c, const float* b, long ldb, int b_is_kn, long M, long N, float* out, long ldo, float* energy,
                   void* workspace, size_t workspace_bytes, void* stream) {
  auto split = [&](const GemmLayout& L, uint8_t* lines, int* sa, Flagged flagged, hipStream_t st) {
    const dim3 grid((unsigned)(L.mt * kTile));
    if (c.K <= 8192)
      hipLaunchKernelGGL((split_caches_kernel<T, ROTATE, 256, 2>), grid, dim3(256), 0, st, c, (int)M, L.KB, lines, sa, flagged,
                         energy);
    else
      hipLaunchKernelGGL((split_caches_kernel<T, ROTATE, 512, 4>), grid, dim3(512), 0, st, c, (int)M, L.KB, lines, sa, flagged,
                         energy);
  };
  return launch_product("dkv_project_caches", CacheRows<T, ROTATE>{c}, split, b, ldb, b_is_kn, nullptr, M, N, c.K, out, ldo,
                        workspace, workspace_bytes, stream);
}

}  // namespace

extern "C" int dkv_project_caches(const uint64_t* layer_ptrs, int32_t dtype, int32_t layers, int32_t heads, int32_t tokens,
                                  int32_t head_dim, const float* cos, const float* sin, const float* mean, int32_t start,
                                  int32_t end, const float* basis, int64_t ldb, int32_t b_is_kn, int64_t rank, float* out,
                                  int64_t ldo, float* energy, void* workspace, size_t workspace_bytes, void* stream) {
  DKV_REQUIRE(layer_ptrs && mean && basis && out, DKV_EINVAL, "dkv_project_caches: null pointer");
  DKV_REQUIRE((cos == nullptr) == (sin == nullptr), DKV_EINVAL, "dkv_project_caches: cos and sin go together");
  DKV_REQUIRE(dtype == DKV_F32 || dtype == DKV_F16 || dtype == DKV_BF16, DKV_EINVAL,
              "dkv_project_caches: dtype %d not supported", dtype);
  DKV_REQUIRE(layers > 0 && heads > 0 && tokens >= 0 && head_dim > 0 && head_dim % 16 == 0 &&
                  (long)layers * heads * head_dim <= 32768,
              DKV_ESHAPE, "dkv_project_caches: bad shape (layers=%d heads=%d tokens=%d head_dim=%d)", layers, heads, tokens,
              head_dim);
  DKV_REQUIRE(0 <= start && start < end && end <= tokens, DKV_ESHAPE, "dkv_project_caches: rows %d..%d outside 0..%d", start,
              end, tokens);
  const CacheArgs c{layer_ptrs, cos, sin, mean, heads, tokens, head_dim, start, layers * heads * head_dim};
#define DKV_PROJECT(T_, R_) \
  return launch_project<T_, R_>(c, basis, ldb, b_is_kn, end - start, rank, out, ldo, energy, workspace, workspace_bytes, stream)
  if (dtype == DKV_F32) {
    if (cos) DKV_PROJECT(DKV_F32, true);
    DKV_PROJECT(DKV_F32, false);
  } else if (dtype == DKV_F16) {
    if (cos) DKV_PROJECT(DKV_F16, true);
    DKV_PROJECT(DKV_F16, false);
  }
  if (cos) DKV_PROJECT(DKV_BF16, true);
  DKV_PROJECT(DKV_BF16, false);
#undef DKV_PROJECT
}

extern "C" int dkv_matmul_f32(const float* a, int64_t lda, const float* b, int64_t ldb, int32_t b_is_kn,
                              const float* bias, int64_t M, int64_t N, int64_t K, float* c, int64_t ldc,
                              void* workspace, size_t workspace_bytes, void* stream) {
  DKV_REQUIRE(a && b && c, DKV_EINVAL, "dkv_matmul_f32: null pointer");
  DKV_REQUIRE(lda >= K, DKV_ESHAPE, "dkv_matmul_f32: bad row strides");
  auto split = [&](const GemmLayout& L, uint8_t* lines, int* sa, Flagged flagged, hipStream_t st) {
    launch_split_rows(a, lda, M, (long)L.mt * kTile, (int)K, L.KB, lines, sa, flagged, st);
  };
  return launch_product("dkv_matmul_f32", PlainRows{a, lda}, split, b, ldb, b_is_kn, bias, M, N, K, c, ldc, workspace,
                        workspace_bytes, stream);
}
