// Packing, K1 unpack/dequantize, cold-plane gather (K4c) and basis layouts.
//
// Reference behaviour replaced here (SrikanthBalaaji/Dimmer-KV):
//   scripts/progressive.py:47-55   dequantize
//   scripts/progressive.py:103-110 TokenStore (codes kept unpacked; only counted)
//   scripts/progressive.py:185-194 hot/cold byte accounting
//   scripts/progressive.py:224-236 ProgressiveCache.refine (cold pieces of the top tokens)
#include <string>

#include "dkv_device.h"
#include "dkv_host.h"

namespace dkv {
static thread_local std::string g_error;
void set_error(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_error = buf;
}
}  // namespace dkv

extern "C" int dkv_abi_version(void) { return DKV_ABI_VERSION; }
extern "C" const char* dkv_last_error(void) { return dkv::g_error.c_str(); }

// ---------------------------------------------------------------------------
// Pack: one thread per (token, group, half).  Byte i of the half's code word w is the coefficient of plane bit
// w + 8 i (before the plane's rotation by 25 + p), so plane word p gathers bit 7 - p of all 32 bytes: an 8 x 8 bit
// transpose of the eight words, byte by byte, in three rounds of masked swaps.  A plane's two words (halves) go
// out side by side from neighbouring lanes.  8,155 tokens x 16 groups with the cold tier: 8.6 us (49 with one wave per
// (token, group), eight shuffles and ballots each).
// ---------------------------------------------------------------------------
// Exchanges the bits of a under `mask << shift` with those of b under `mask`.
DKV_DEVICE void swap_bits(uint32_t& a, uint32_t& b, int shift, uint32_t mask) {
  const uint32_t d = ((a >> shift) ^ b) & mask;
  b ^= d;
  a ^= d << shift;
}

// In every byte lane: bit p of word w <-> bit w of word p.
DKV_DEVICE void transpose_bits(uint32_t (&v)[8]) {
#pragma unroll
  for (int w = 0; w < 4; ++w) swap_bits(v[w], v[w + 4], 4, 0x0f0f0f0fu);
#pragma unroll
  for (int w = 0; w < 8; w += 4) {
    swap_bits(v[w], v[w + 2], 2, 0x33333333u);
    swap_bits(v[w + 1], v[w + 3], 2, 0x33333333u);
  }
#pragma unroll
  for (int w = 0; w < 8; w += 2) swap_bits(v[w], v[w + 1], 1, 0x55555555u);
}

__global__ __launch_bounds__(256) void pack_kernel(const uint8_t* __restrict__ codes, const uint16_t* __restrict__ low,
                                                   const uint16_t* __restrict__ span,
                                                   const int16_t* __restrict__ pieces, int n, dkv_order_t order,
                                                   uint8_t* __restrict__ hot, const int64_t* __restrict__ hot_off,
                                                   uint8_t* __restrict__ cold,
                                                   const int64_t* __restrict__ cold_tok_off) {
  const int G = order.groups;
  const long id = (long)blockIdx.x * 256 + threadIdx.x;
  const long gw = id >> 1;
  const int h = (int)(id & 1);
  if (gw >= (long)n * G) return;
  const int t = (int)(gw / G), g = (int)(gw % G);
  uint32_t v[8];
  __builtin_memcpy(v, codes + gw * 64 + h * 32, 32);  // (a caller's buffer may lie at any byte)
  const int k = pieces[t];
  const int m = order.planes[(long)k * G + g];
  const int m_full = order.planes[(long)order.pieces * G + g];
  const uint32_t header = (uint32_t)low[gw] | ((uint32_t)span[gw] << 16);
  transpose_bits(v);
  uint32_t words[8];
#pragma unroll
  for (int p = 0; p < 8; ++p) words[p] = __builtin_rotateright32(v[7 - p], (25 + p) & 31);
  if (m > 0) {
    uint32_t* dst = (uint32_t*)(hot + hot_off[t] + order.seg_off[(long)k * G + g]);
    if (h == 0) dst[0] = header;
#pragma unroll
    for (int p = 0; p < 8; ++p)
      if (p < m) dst[1 + 2 * p + h] = words[p];
  }
  if (cold != nullptr && m < m_full) {
    uint32_t* dst = (uint32_t*)(cold + cold_tok_off[t] + order.cold_off[(long)k * G + g]);
    if (m == 0) {
      if (h == 0) dst[0] = header;
      dst += 1;
    }
#pragma unroll
    for (int p = 0; p < 8; ++p)
      if (p >= m && p < m_full) dst[2 * (p - m) + h] = words[p];
  }
}

extern "C" int dkv_pack_planes(const uint8_t* codes, const uint16_t* low, const uint16_t* span, const int16_t* pieces,
                               int32_t n, dkv_order_t order, uint8_t* hot, const int64_t* hot_off, uint8_t* cold,
                               const int64_t* cold_off, void* stream) {
  DKV_REQUIRE(n >= 0, DKV_ESHAPE, "dkv_pack_planes: n < 0");
  int rc = dkv::check_order(order, "dkv_pack_planes");
  if (rc) return rc;
  if (n == 0) return DKV_OK;
  DKV_REQUIRE(codes && low && span && pieces && hot && hot_off, DKV_EINVAL, "dkv_pack_planes: null pointer");
  DKV_REQUIRE(!cold || (cold_off && order.cold_off), DKV_EINVAL, "dkv_pack_planes: cold needs cold offsets");
  const long blocks = ((long)n * order.groups * 2 + 255) / 256;
  DKV_REQUIRE(blocks < (1L << 31), DKV_ESHAPE, "dkv_pack_planes: too many tokens");
  hipLaunchKernelGGL(pack_kernel, dim3((unsigned)blocks), dim3(256), 0, dkv::as_stream(stream), codes, low, span,
                     pieces, n, order, hot, hot_off, cold, cold_off);
  return dkv::check_launch("dkv_pack_planes");
}

// ---------------------------------------------------------------------------
// Ladder pack: one thread per (token, group, half).  The 32 codes of the half
// are squeezed to b bits each, LSB-first (code j at bit b*j), into b words;
// the thread of half 0 also writes the [low][scale] header.
// ---------------------------------------------------------------------------
DKV_DEVICE uint32_t gather_nibbles(uint32_t c) {  // 4 bytes < 16 -> 16 bits
  return (c & 0xfu) | ((c >> 4) & 0xf0u) | ((c >> 8) & 0xf00u) | ((c >> 12) & 0xf000u);
}

DKV_DEVICE uint32_t gather_pairs(uint32_t c) {  // 4 bytes < 4 -> 8 bits
  return (c & 0x3u) | ((c >> 6) & 0xcu) | ((c >> 12) & 0x30u) | ((c >> 18) & 0xc0u);
}

__global__ __launch_bounds__(256) void pack_ladder_kernel(const uint8_t* __restrict__ codes,
                                                          const uint16_t* __restrict__ low,
                                                          const uint16_t* __restrict__ scale,
                                                          const int16_t* __restrict__ rung, int n, dkv_ladder_t lad,
                                                          uint8_t* __restrict__ blob,
                                                          const int64_t* __restrict__ tok_off) {
  const int G = lad.groups;
  const long id = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (long)n * G * 2) return;
  const int h = (int)(id & 1);
  const long tg = id >> 1;
  const int t = (int)(tg / G), g = (int)(tg % G);
  const int r = rung[t];
  if (r < 0 || r >= lad.rungs) return;
  const int b = lad.bits[(long)r * G + g];
  if (b != 2 && b != 4 && b != 8) return;
  uint32_t* seg = (uint32_t*)(blob + tok_off[t] + lad.seg_off[(long)r * G + g]);
  if (h == 0) seg[0] = (uint32_t)low[tg] | ((uint32_t)scale[tg] << 16);
  const uint4* src = (const uint4*)(codes + tg * 64 + h * 32);
  const uint4 c0 = src[0], c1 = src[1];
  const uint32_t cw[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
  uint32_t* dst = seg + 1 + b * h;
  if (b == 8) {
#pragma unroll
    for (int k = 0; k < 8; ++k) dst[k] = cw[k];
  } else if (b == 4) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      dst[k] = gather_nibbles(cw[2 * k] & 0x0f0f0f0fu) | (gather_nibbles(cw[2 * k + 1] & 0x0f0f0f0fu) << 16);
  } else {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      uint32_t wv = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) wv |= gather_pairs(cw[4 * k + j] & 0x03030303u) << (8 * j);
      dst[k] = wv;
    }
  }
}

extern "C" int dkv_pack_ladder(const uint8_t* codes, const uint16_t* low, const uint16_t* scale, const int16_t* rung,
                               int32_t n, dkv_ladder_t ladder, uint8_t* blob, const int64_t* tok_off, void* stream) {
  DKV_REQUIRE(n >= 0, DKV_ESHAPE, "dkv_pack_ladder: n < 0");
  int rc = dkv::check_ladder(ladder, "dkv_pack_ladder");
  if (rc) return rc;
  if (n == 0) return DKV_OK;
  DKV_REQUIRE(codes && low && scale && rung && blob && tok_off, DKV_EINVAL, "dkv_pack_ladder: null pointer");
  const long threads = (long)n * ladder.groups * 2;
  const long blocks = (threads + 255) / 256;
  DKV_REQUIRE(blocks < (1L << 31), DKV_ESHAPE, "dkv_pack_ladder: too many tokens");
  hipLaunchKernelGGL(pack_ladder_kernel, dim3((unsigned)blocks), dim3(256), 0, dkv::as_stream(stream), codes, low,
                     scale, rung, n, ladder, blob, tok_off);
  return dkv::check_launch("dkv_pack_ladder");
}

// ---------------------------------------------------------------------------
// Byte storage.  One thread per (token, group, half): the half's 32 codes are
// 4b bytes of the (token, group)'s code run, which starts at a byte boundary
// (64 b-bit codes are 8b bytes), so halves never share a byte.  Storage
// positions carry no alignment (the sections follow byte-sized rung ids), so
// the storage side moves single bytes; the code/shift/scale side is aligned.
// ---------------------------------------------------------------------------
struct WireSpot {
  long code, low, scale;  // byte positions of the half's codes and of the group's shift and scale
  int b;                  // width, 0 = nothing to move
};

DKV_DEVICE int width_index(int b) { return b == 2 ? 0 : (b == 4 ? 1 : 2); }

DKV_DEVICE WireSpot wire_spot(const int16_t* __restrict__ rung, const dkv_ladder_t& lad, const dkv_wire_t& w, int t,
                              int g, int h) {
  WireSpot s{0, 0, 0, 0};
  const int G = lad.groups;
  const int r = rung[t];
  if (r < 0 || r >= lad.rungs) return s;
  const int b = lad.bits[(long)r * G + g];
  if (b != 2 && b != 4 && b != 8) return s;
  const int wi = width_index(b);
  const long cnt = w.count[r], nw = w.nwidth[3 * r + wi];
  const long k = w.rank[t], j = w.slot[(long)r * G + g];
  if (k < 0 || k >= cnt || j < 0 || j >= nw) return s;
  const long base = w.section[3 * r + wi];
  const long item = k * nw + j;
  s.code = base + item * 8 * b + 4 * b * h;
  s.low = base + cnt * nw * 8 * b + item * 2;
  s.scale = base + cnt * nw * (8 * b + 2) + item * 2;
  if (base < 0 || s.scale + 2 > w.bytes) return s;  // outside the storage buffer: leave it alone
  s.b = b;
  return s;
}

__global__ __launch_bounds__(256) void wire_pack_kernel(const uint8_t* __restrict__ codes,
                                                        const uint16_t* __restrict__ low,
                                                        const uint16_t* __restrict__ scale,
                                                        const int16_t* __restrict__ rung, int n, dkv_ladder_t lad,
                                                        dkv_wire_t w, uint8_t* __restrict__ out) {
  const int G = lad.groups;
  const long id = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (long)n * G * 2) return;
  const int h = (int)(id & 1);
  const long tg = id >> 1;
  const int t = (int)(tg / G), g = (int)(tg % G);
  const WireSpot s = wire_spot(rung, lad, w, t, g, h);
  if (s.b == 0) return;
  const uint4* src = (const uint4*)(codes + tg * 64 + h * 32);
  const uint4 c0 = src[0], c1 = src[1];
  const uint32_t cw[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
  uint32_t pw[8];
  if (s.b == 8) {
#pragma unroll
    for (int k = 0; k < 8; ++k) pw[k] = cw[k];
  } else if (s.b == 4) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      pw[k] = gather_nibbles(cw[2 * k] & 0x0f0f0f0fu) | (gather_nibbles(cw[2 * k + 1] & 0x0f0f0f0fu) << 16);
  } else {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      uint32_t wv = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) wv |= gather_pairs(cw[4 * k + j] & 0x03030303u) << (8 * j);
      pw[k] = wv;
    }
  }
  uint8_t* dst = out + s.code;
#pragma unroll
  for (int k = 0; k < 8; ++k)  // b words = 4b bytes
    if (k < s.b)
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[4 * k + i] = (uint8_t)(pw[k] >> (8 * i));
  if (h == 0) {
    const uint16_t lo = low[tg], sc = scale[tg];
    out[s.low] = (uint8_t)lo;
    out[s.low + 1] = (uint8_t)(lo >> 8);
    out[s.scale] = (uint8_t)sc;
    out[s.scale + 1] = (uint8_t)(sc >> 8);
  }
}

// The 32 codes of a half from its 4B storage bytes (code i at bit B*i), one code per byte of cw.
template <int B>
DKV_DEVICE void wire_codes_half(const uint8_t* __restrict__ src, uint32_t (&cw)[8]) {
  uint32_t pw[B];
#pragma unroll
  for (int k = 0; k < B; ++k)
    pw[k] = (uint32_t)src[4 * k] | ((uint32_t)src[4 * k + 1] << 8) | ((uint32_t)src[4 * k + 2] << 16) |
            ((uint32_t)src[4 * k + 3] << 24);
  constexpr uint32_t kMask = (1u << B) - 1u;
#pragma unroll
  for (int k = 0; k < 8; ++k) {  // codes 4k .. 4k+3
    uint32_t v = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int bit = (4 * k + i) * B;
      v |= ((pw[bit >> 5] >> (bit & 31)) & kMask) << (8 * i);
    }
    cw[k] = v;
  }
}

__global__ __launch_bounds__(256) void wire_unpack_kernel(const uint8_t* __restrict__ in,
                                                          const int16_t* __restrict__ rung, int n, dkv_ladder_t lad,
                                                          dkv_wire_t w, uint8_t* __restrict__ codes,
                                                          uint16_t* __restrict__ low, uint16_t* __restrict__ scale) {
  const int G = lad.groups;
  const long id = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (long)n * G * 2) return;
  const int h = (int)(id & 1);
  const long tg = id >> 1;
  const int t = (int)(tg / G), g = (int)(tg % G);
  const WireSpot s = wire_spot(rung, lad, w, t, g, h);
  if (s.b == 0) return;
  uint32_t cw[8];
  if (s.b == 8) {
    wire_codes_half<8>(in + s.code, cw);
  } else if (s.b == 4) {
    wire_codes_half<4>(in + s.code, cw);
  } else {
    wire_codes_half<2>(in + s.code, cw);
  }
  uint4* dst = (uint4*)(codes + tg * 64 + h * 32);
  dst[0] = make_uint4(cw[0], cw[1], cw[2], cw[3]);
  dst[1] = make_uint4(cw[4], cw[5], cw[6], cw[7]);
  if (h == 0) {
    low[tg] = (uint16_t)(in[s.low] | (in[s.low + 1] << 8));
    scale[tg] = (uint16_t)(in[s.scale] | (in[s.scale + 1] << 8));
  }
}

static int check_wire(const dkv_wire_t& w, int32_t n, const char* what) {
  if (!w.section || !w.count || !w.slot || !w.nwidth || (n > 0 && !w.rank) || w.bytes < 0) {
    dkv::set_error("%s: storage tables must be non-null and bytes >= 0", what);
    return DKV_EINVAL;
  }
  return DKV_OK;
}

extern "C" int dkv_wire_pack(const uint8_t* codes, const uint16_t* low, const uint16_t* scale, const int16_t* rung,
                             int32_t n, dkv_ladder_t ladder, dkv_wire_t wire, uint8_t* out, void* stream) {
  DKV_REQUIRE(n >= 0, DKV_ESHAPE, "dkv_wire_pack: n < 0");
  int rc = dkv::check_ladder(ladder, "dkv_wire_pack");
  if (rc) return rc;
  if ((rc = check_wire(wire, n, "dkv_wire_pack"))) return rc;
  if (n == 0) return DKV_OK;
  DKV_REQUIRE(codes && low && scale && rung && out, DKV_EINVAL, "dkv_wire_pack: null pointer");
  const long blocks = ((long)n * ladder.groups * 2 + 255) / 256;
  DKV_REQUIRE(blocks < (1L << 31), DKV_ESHAPE, "dkv_wire_pack: too many tokens");
  hipLaunchKernelGGL(wire_pack_kernel, dim3((unsigned)blocks), dim3(256), 0, dkv::as_stream(stream), codes, low, scale,
                     rung, n, ladder, wire, out);
  return dkv::check_launch("dkv_wire_pack");
}

extern "C" int dkv_wire_unpack(const uint8_t* in, const int16_t* rung, int32_t n, dkv_ladder_t ladder,
                               dkv_wire_t wire, uint8_t* codes, uint16_t* low, uint16_t* scale, void* stream) {
  DKV_REQUIRE(n >= 0, DKV_ESHAPE, "dkv_wire_unpack: n < 0");
  int rc = dkv::check_ladder(ladder, "dkv_wire_unpack");
  if (rc) return rc;
  if ((rc = check_wire(wire, n, "dkv_wire_unpack"))) return rc;
  if (n == 0) return DKV_OK;
  DKV_REQUIRE(in && rung && codes && low && scale, DKV_EINVAL, "dkv_wire_unpack: null pointer");
  const long blocks = ((long)n * ladder.groups * 2 + 255) / 256;
  DKV_REQUIRE(blocks < (1L << 31), DKV_ESHAPE, "dkv_wire_unpack: too many tokens");
  hipLaunchKernelGGL(wire_unpack_kernel, dim3((unsigned)blocks), dim3(256), 0, dkv::as_stream(stream), in, rung, n,
                     ladder, wire, codes, low, scale);
  return dkv::check_launch("dkv_wire_unpack");
}

// ---------------------------------------------------------------------------
// K1: one thread per (token, group, half): 32 coefficients.
// ---------------------------------------------------------------------------
// Ladder streams: code * scale + low in fp32 (scripts/kvtc.py:78), then the
// output cast.  A rung outside the ladder decodes to zeros.
template <int DT>
DKV_DEVICE void unpack_ladder_half(const dkv_stream_t& s, int t, int g, int h, long base, void* __restrict__ out) {
  const int G = s.ladder.groups;
  const int r = s.pieces[t];
  const bool ok = r >= 0 && r < s.ladder.rungs;
  const int b = ok ? s.ladder.bits[(long)r * G + g] : 0;
  const uint8_t* seg = s.blob + s.tok_off[t] + (ok ? s.ladder.seg_off[(long)r * G + g] : 0);
  uint32_t cw[8], header;
  load_ladder_half(seg, b, h, cw, header);
  const float low = half_bits_to_float((uint16_t)(header & 0xffffu));
  const float scale = half_bits_to_float((uint16_t)(header >> 16));
#pragma unroll
  for (int w = 0; w < 8; ++w)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      store_from_float(out, base + 4 * w + i, DT, ladder_value((cw[w] >> (8 * i)) & 0xffu, low, scale));
}

template <int DT>
__global__ __launch_bounds__(256) void unpack_dequant_kernel(dkv_stream_t s, int t0, int nt, void* __restrict__ out) {
  const int G = dkv_groups(s);
  const long id = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (long)nt * G * 2) return;
  const int h = (int)(id & 1);
  const long tg = id >> 1;
  const int tt = (int)(tg / G), g = (int)(tg % G);
  const int t = t0 + tt;
  if (s.format == DKV_FMT_LADDER) {
    unpack_ladder_half<DT>(s, t, g, h, (long)tt * (64L * G) + g * 64 + h * 32, out);
    return;
  }
  const int k = s.pieces[t];
  const int m = s.order.planes[(long)k * G + g];
  const uint8_t* seg = s.blob + s.tok_off[t] + s.order.seg_off[(long)k * G + g];
  uint32_t pl[8], header;
  load_segment(seg, m, h, pl, header);
  const float low = half_bits_to_float((uint16_t)(header & 0xffffu));
  const float span = half_bits_to_float((uint16_t)(header >> 16));
  const float inv_bins = __builtin_ldexpf(1.0f, -m);
  uint32_t cw[8];
  cw[0] = assemble_codes<0>(pl);
  cw[1] = assemble_codes<1>(pl);
  cw[2] = assemble_codes<2>(pl);
  cw[3] = assemble_codes<3>(pl);
  cw[4] = assemble_codes<4>(pl);
  cw[5] = assemble_codes<5>(pl);
  cw[6] = assemble_codes<6>(pl);
  cw[7] = assemble_codes<7>(pl);
  const long base = (long)tt * (64L * G) + g * 64 + h * 32;
  if (DT == DKV_F32) {
    float4* o = (float4*)((float*)out + base);
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      float4 v;
      v.x = dequant_exact(cw[w] & 0xffu, m, low, span, inv_bins);
      v.y = dequant_exact((cw[w] >> 8) & 0xffu, m, low, span, inv_bins);
      v.z = dequant_exact((cw[w] >> 16) & 0xffu, m, low, span, inv_bins);
      v.w = dequant_exact(cw[w] >> 24, m, low, span, inv_bins);
      o[w] = v;
    }
  } else {
#pragma unroll
    for (int w = 0; w < 8; ++w) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        store_from_float(out, base + 4 * w + i, DT, dequant_exact((cw[w] >> (8 * i)) & 0xffu, m, low, span, inv_bins));
    }
  }
}

extern "C" int dkv_unpack_dequant(const dkv_stream_t* s, int32_t t0, int32_t nt, void* out, int32_t out_dtype,
                                  void* stream) {
  int rc = dkv::check_stream(s, "dkv_unpack_dequant");
  if (rc) return rc;
  DKV_REQUIRE(out, DKV_EINVAL, "dkv_unpack_dequant: out is null");
  DKV_REQUIRE(t0 >= 0 && nt >= 0, DKV_ESHAPE, "dkv_unpack_dequant: bad token range");
  DKV_REQUIRE(out_dtype == DKV_F32 || out_dtype == DKV_F16 || out_dtype == DKV_BF16, DKV_EINVAL,
              "dkv_unpack_dequant: bad dtype %d", out_dtype);
  if (nt == 0) return DKV_OK;
  const long threads = (long)nt * dkv::stream_groups(*s) * 2;
  const unsigned blocks = (unsigned)((threads + 255) / 256);
  hipStream_t st = dkv::as_stream(stream);
  if (out_dtype == DKV_F32)
    hipLaunchKernelGGL(unpack_dequant_kernel<DKV_F32>, dim3(blocks), dim3(256), 0, st, *s, t0, nt, out);
  else if (out_dtype == DKV_F16)
    hipLaunchKernelGGL(unpack_dequant_kernel<DKV_F16>, dim3(blocks), dim3(256), 0, st, *s, t0, nt, out);
  else
    hipLaunchKernelGGL(unpack_dequant_kernel<DKV_BF16>, dim3(blocks), dim3(256), 0, st, *s, t0, nt, out);
  return dkv::check_launch("dkv_unpack_dequant");
}

// Reference dequantize on unpacked codes (progressive.py:47-55).
__global__ __launch_bounds__(256) void dequantize_codes_kernel(const uint8_t* __restrict__ codes,
                                                               const uint16_t* __restrict__ low,
                                                               const uint16_t* __restrict__ span,
                                                               const uint8_t* __restrict__ planes, int planes_rows,
                                                               int n, int G, float* __restrict__ out) {
  const long id = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (long)n * G * 64) return;
  const long tg = id >> 6;
  const int t = (int)(tg / G), g = (int)(tg % G);
  const int m = planes[(long)(planes_rows == 1 ? 0 : t) * G + g];
  const float lo = half_bits_to_float(low[tg]);
  const float sp = half_bits_to_float(span[tg]);
  out[id] = dequant_exact(codes[id], m, lo, sp, __builtin_ldexpf(1.0f, -m));
}

extern "C" int dkv_dequantize_codes(const uint8_t* codes, const uint16_t* low, const uint16_t* span,
                                    const uint8_t* planes, int32_t planes_rows, int32_t n, int32_t groups, float* out,
                                    void* stream) {
  DKV_REQUIRE(codes && low && span && planes && out, DKV_EINVAL, "dkv_dequantize_codes: null pointer");
  DKV_REQUIRE(n >= 0 && groups > 0 && (planes_rows == 1 || planes_rows == n), DKV_ESHAPE,
              "dkv_dequantize_codes: bad shape (n=%d groups=%d planes_rows=%d)", n, groups, planes_rows);
  if (n == 0) return DKV_OK;
  const long total = (long)n * groups * 64;
  hipLaunchKernelGGL(dequantize_codes_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                     dkv::as_stream(stream), codes, low, span, planes, planes_rows, n, groups, out);
  return dkv::check_launch("dkv_dequantize_codes");
}

// ---------------------------------------------------------------------------
// Encoder: quantize8 (progressive.py:37-44) and the squared error of the codes cut to 0..8 planes
// (progressive.py:152-158) in one pass over the coefficients.  16 lanes per (token, group), four members
// a lane (one 16-byte load, one word of codes): the group's min and max are reductions over the 16
// lanes; low = f16(min), span = f16(max(max - low, 1e-8)), code = clamp(floor((x - low) / span * 256), 0, 255)
// with the division correctly rounded (a NaN from a zero fp16 span gives code 0); then every lane's
// squared errors against the reference's dequantize at each plane count, summed over the lanes.
//
// quantize8_kernel writes the codes and, asked for, the table of a group's nine errors; rung_errors_kernel writes
// the codes and what the allocator takes instead of the table: a token's error at every rung of the order (the
// sum over its groups of the table entry at the rung's planes) and its energy (the errors at no planes), a wave
// per token.  8,155 tokens x 1,024, codes and errors at 7 rungs: 26 us, bound by the errors' arithmetic (its bytes take
// 8; 53 us with the table at one wave per group before, and torch's gather and sums over it besides).
// ---------------------------------------------------------------------------
template <int CTRL>
DKV_DEVICE float lanes_dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// Over the 16 lanes of a DPP row, in every lane: xor 1, xor 2, then the mirrored half row and row.
DKV_DEVICE float row_sum(float v) {
  v += lanes_dpp<0xB1>(v);
  v += lanes_dpp<0x4E>(v);
  v += lanes_dpp<0x141>(v);
  return v + lanes_dpp<0x140>(v);
}

DKV_DEVICE float row_max(float v) {
  v = fmaxf(v, lanes_dpp<0xB1>(v));
  v = fmaxf(v, lanes_dpp<0x4E>(v));
  v = fmaxf(v, lanes_dpp<0x141>(v));
  return fmaxf(v, lanes_dpp<0x140>(v));
}

struct QuadCodes {
  float lo, sp;
  uint32_t codes;  // byte i: member 4 * (lane & 15) + i
};

DKV_DEVICE uint16_t half_bits(float v) {
  const half_t h = (half_t)v;
  uint16_t b;
  __builtin_memcpy(&b, &h, 2);
  return b;
}

DKV_DEVICE QuadCodes quantize_quad(const float (&x)[4]) {
  QuadCodes q;
  const float amin = -row_max(fmaxf(fmaxf(-x[0], -x[1]), fmaxf(-x[2], -x[3])));
  const float amax = row_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
  q.lo = (float)(half_t)amin;
  q.sp = (float)(half_t)fmaxf(amax - q.lo, 1e-8f);
  q.codes = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float v;
    {
#pragma clang fp contract(off)
      v = floorf(((x[i] - q.lo) / q.sp) * 256.0f);
    }
    v = (v != v) ? 0.0f : fminf(fmaxf(v, 0.0f), 255.0f);
    q.codes |= (uint32_t)v << (8 * i);
  }
  return q;
}

// The group's squared error at `lane & 15` planes (0 in lanes past 8).  dequant_exact's value at m planes,
// low + ((code >> (8 - m)) + 0.5) * span / 2^m, with the code's low bits cleared instead of shifted out: the factor
// has at most 9 bits and the fp16 span 11, so their product is exact and one fma rounds the sum as the separate
// operations do.
DKV_DEVICE float quad_error(const float (&x)[4], const QuadCodes& q) {
  const int j = threadIdx.x & 15;
  const float step = q.sp * (1.0f / 256.0f);
  float mine = 0.0f;
#pragma unroll
  for (int m = 0; m <= 8; ++m) {
    const uint32_t cut = q.codes & (0x01010101u * (0xffu & (0xff00u >> m)));
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float c = (float)((cut >> (8 * i)) & 0xffu) + __builtin_ldexpf(0.5f, 8 - m);
      const float d = m == 0 ? x[i] : x[i] - __builtin_fmaf(c, step, q.lo);
      s = __builtin_fmaf(d, d, s);
    }
    s = row_sum(s);
    mine = j == m ? s : mine;
  }
  return mine;
}

__global__ __launch_bounds__(256) void quantize8_kernel(const float* __restrict__ coef, long ngroups,
                                                        uint8_t* __restrict__ codes, uint16_t* __restrict__ low,
                                                        uint16_t* __restrict__ span, float* __restrict__ errors) {
  const long tg = (long)blockIdx.x * 16 + (threadIdx.x >> 4);
  const int j = threadIdx.x & 15;
  if (tg >= ngroups) return;  // whole rows of 16 lanes
  float x[4];
  __builtin_memcpy(x, coef + tg * 64 + 4 * j, 16);  // (callers' buffers may lie at any element)
  const QuadCodes q = quantize_quad(x);
  __builtin_memcpy(codes + tg * 64 + 4 * j, &q.codes, 4);
  if (j == 0) {
    low[tg] = half_bits(q.lo);
    span[tg] = half_bits(q.sp);
  }
  if (!errors) return;
  const float e = quad_error(x, q);
  if (j <= 8) errors[tg * 9 + j] = e;
}

constexpr int kRungChunks = 8;  // 16 rungs each

template <int CHUNKS>
__global__ __launch_bounds__(256) void rung_errors_kernel(const float* __restrict__ coef, int n, int G,
                                                          const uint8_t* __restrict__ planes, int rungs,
                                                          uint8_t* __restrict__ codes, uint16_t* __restrict__ low,
                                                          uint16_t* __restrict__ span, float* __restrict__ errors,
                                                          float* __restrict__ energy) {
  extern __shared__ uint8_t at_rung[];  // [rungs][G]
  for (int e = threadIdx.x; e < rungs * G; e += 256) at_rung[e] = min((int)planes[e], 8);
  __syncthreads();
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= n) return;
  const int lane = threadIdx.x & 63, j = lane & 15, row = lane >> 4;
  float sum[CHUNKS], total = 0.0f;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) sum[c] = 0.0f;
  const float* src = coef + (long)t * G * 64 + lane * 4;
  float next[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (row < G) __builtin_memcpy(next, src, 16);
  for (int g0 = 0; g0 < G; g0 += 4) {
    const int g = g0 + row;  // past the last group: zeros, not stored, not summed
    float x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = g < G ? next[i] : 0.0f;
    if (g + 4 < G) __builtin_memcpy(next, src + (long)(g0 + 4) * 64, 16);
    const QuadCodes q = quantize_quad(x);
    const float e = quad_error(x, q);
    const long tg = (long)t * G + g;
    if (g < G) {
      __builtin_memcpy(codes + tg * 64 + 4 * j, &q.codes, 4);
      if (j == 0) {
        low[tg] = half_bits(q.lo);
        span[tg] = half_bits(q.sp);
        total += e;  // lane 0 of the row holds the error at no planes
      }
    }
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int r = min(c * 16 + j, rungs - 1);
      const float v = __shfl(e, (lane & 48) + at_rung[r * G + min(g, G - 1)], 64);
      sum[c] += g < G ? v : 0.0f;
    }
  }
  // the four rows' groups
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    float v = sum[c];
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    if (row == 0 && c * 16 + j < rungs) errors[(long)t * rungs + c * 16 + j] = v;
  }
  total += __shfl_xor(total, 16, 64);
  total += __shfl_xor(total, 32, 64);
  if (lane == 0) energy[t] = total;
}

extern "C" int dkv_quantize8(const float* coef, int32_t n, int32_t groups, uint8_t* codes, uint16_t* low,
                             uint16_t* span, float* errors, void* stream) {
  DKV_REQUIRE(coef && codes && low && span, DKV_EINVAL, "dkv_quantize8: null pointer");
  DKV_REQUIRE(n >= 0 && groups > 0, DKV_ESHAPE, "dkv_quantize8: bad shape (n=%d groups=%d)", n, groups);
  if (n == 0) return DKV_OK;
  const long ngroups = (long)n * groups;
  hipLaunchKernelGGL(quantize8_kernel, dim3((unsigned)((ngroups + 15) / 16)), dim3(256), 0, dkv::as_stream(stream),
                     coef, ngroups, codes, low, span, errors);
  return dkv::check_launch("dkv_quantize8");
}

extern "C" int dkv_quantize8_rungs(const float* coef, int32_t n, int32_t groups, const uint8_t* planes, int32_t rungs,
                                   uint8_t* codes, uint16_t* low, uint16_t* span, float* errors, float* energy,
                                   void* stream) {
  DKV_REQUIRE(n >= 0 && groups > 0 && rungs > 0 && rungs <= 16 * kRungChunks && (long)rungs * groups <= 65536, DKV_ESHAPE,
              "dkv_quantize8_rungs: bad shape (n=%d groups=%d rungs=%d)", n, groups, rungs);
  if (n == 0) return DKV_OK;
  DKV_REQUIRE(coef && planes && codes && low && span && errors && energy, DKV_EINVAL, "dkv_quantize8_rungs: null pointer");
  const dim3 grid((unsigned)((n + 3) / 4));
  const size_t lds = (size_t)rungs * groups;
  if (rungs <= 16)
    hipLaunchKernelGGL(rung_errors_kernel<1>, grid, dim3(256), lds, dkv::as_stream(stream), coef, n, groups, planes, rungs,
                       codes, low, span, errors, energy);
  else
    hipLaunchKernelGGL(rung_errors_kernel<kRungChunks>, grid, dim3(256), lds, dkv::as_stream(stream), coef, n, groups, planes,
                       rungs, codes, low, span, errors, energy);
  return dkv::check_launch("dkv_quantize8_rungs");
}

// ---------------------------------------------------------------------------
// Centred token-matrix rows of the middle tokens, the encoders' input to the PCA projection
// (scripts/kvtc.py:137-140 to_matrix with :40-43 derotate and :50-53 token_matrix, then
// (matrix[start:end] - mean), :189 and scripts/progressive.py:147-148): row t - start, column
// f = (l * H + h) * D + d holds x - mean[f], x the cache element [l][0][h][t][d] as fp32 and, for
// keys, first de-rotated at position t: (k * cos - rotate_half(k) * sin) / (cos^2 + sin^2).  Every
// operation is rounded on its own, as the reference's separate tensor operations round them (no
// contraction), so the rows are bit-identical to that torch arithmetic.
//
// Bound by the rows it writes (4 bytes an element; it reads 2 of an fp16 cache).  A thread keeps its columns
// (4 at d, and for keys the 4 at d + D/2 that rotate with them, so every cache element is loaded once) over
// kRowTok tokens whose loads go out together; the column arithmetic is 32-bit and done once.  16,348 tokens x
// 28,672 columns from fp16 keys: 952 -> 627 us (4.5 TB/s; the card copies at 5.2), 8,155 x 8,192: keys 133 -> 84
// us, values 98 -> 68 (one thread per 4 columns and token before, with 64-bit index divisions and each key
// element loaded twice).
// ---------------------------------------------------------------------------
template <int T>
DKV_DEVICE float4 load_elem4(const void* base, long idx) {
  if constexpr (T == DKV_F32) {
    return *(const float4*)((const float*)base + idx);
  } else {
    const uint2 w = *(const uint2*)((const uint16_t*)base + idx);
    const uint16_t e[4] = {(uint16_t)(w.x & 0xffffu), (uint16_t)(w.x >> 16), (uint16_t)(w.y & 0xffffu),
                           (uint16_t)(w.y >> 16)};
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = T == DKV_BF16 ? bf16_bits_to_float(e[i]) : half_bits_to_float(e[i]);
    return make_float4(v[0], v[1], v[2], v[3]);
  }
}

constexpr int kRowTok = 4;  // tokens per thread

template <int T, bool ROTATE>
__global__ __launch_bounds__(256) void centered_rows_kernel(const uint64_t* __restrict__ layer_ptrs, int L, int H,
                                                            int tokens, int D, const float* __restrict__ cos,
                                                            const float* __restrict__ sin,
                                                            const float* __restrict__ mean, int start, int end,
                                                            int col_blocks, float* __restrict__ out) {
  const int W = ROTATE ? D / 8 : D / 4;  // threads per head: 4 columns, or 4 pairs
  const int c = (int)(blockIdx.x % col_blocks) * 256 + threadIdx.x;
  if (c >= L * H * W) return;
  const int t0 = start + (int)(blockIdx.x / col_blocks) * kRowTok;
  const int lh = c / W, d = 4 * (c % W);
  const int l = lh / H, h = lh % H;
  const void* base = (const void*)layer_ptrs[l];
  const long F = (long)L * H * D, f = (long)lh * D + d;
  const int half = D / 2;
  const float4 mu = *(const float4*)(mean + f);
  float4 x[kRowTok], y[kRowTok], c0[kRowTok], s0[kRowTok], c1[kRowTok], s1[kRowTok];
#pragma unroll
  for (int i = 0; i < kRowTok; ++i) {
    const long t = min(t0 + i, end - 1);
    const long row = ((long)h * tokens + t) * D;  // the cache element [l][0][h][t][.]
    x[i] = load_elem4<T>(base, row + d);
    if constexpr (ROTATE) {
      y[i] = load_elem4<T>(base, row + d + half);
      c0[i] = *(const float4*)(cos + t * D + d);
      s0[i] = *(const float4*)(sin + t * D + d);
      c1[i] = *(const float4*)(cos + t * D + d + half);
      s1[i] = *(const float4*)(sin + t * D + d + half);
    }
  }
  float4 mu1 = mu;
  if constexpr (ROTATE) mu1 = *(const float4*)(mean + f + half);
#pragma unroll
  for (int i = 0; i < kRowTok; ++i) {
    if (t0 + i >= end) break;
    float* o = out + (long)(t0 + i - start) * F + f;
    if constexpr (ROTATE) {
      const float xv[4] = {x[i].x, x[i].y, x[i].z, x[i].w}, yv[4] = {y[i].x, y[i].y, y[i].z, y[i].w};
      const float a0[4] = {c0[i].x, c0[i].y, c0[i].z, c0[i].w}, b0[4] = {s0[i].x, s0[i].y, s0[i].z, s0[i].w};
      const float a1[4] = {c1[i].x, c1[i].y, c1[i].z, c1[i].w}, b1[4] = {s1[i].x, s1[i].y, s1[i].z, s1[i].w};
      const float m0[4] = {mu.x, mu.y, mu.z, mu.w}, m1[4] = {mu1.x, mu1.y, mu1.z, mu1.w};
      float lo[4], hi[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo[e] = derotated(xv[e], -yv[e], a0[e], b0[e], m0[e]);
        hi[e] = derotated(yv[e], xv[e], a1[e], b1[e], m1[e]);
      }
      *(float4*)o = make_float4(lo[0], lo[1], lo[2], lo[3]);
      *(float4*)(o + half) = make_float4(hi[0], hi[1], hi[2], hi[3]);
    } else {
      *(float4*)o = make_float4(x[i].x - mu.x, x[i].y - mu.y, x[i].z - mu.z, x[i].w - mu.w);
    }
  }
}

extern "C" int dkv_centered_rows(const uint64_t* layer_ptrs, int32_t dtype, int32_t layers, int32_t heads,
                                 int32_t tokens, int32_t head_dim, const float* cos, const float* sin,
                                 const float* mean, int32_t start, int32_t end, float* out, void* stream) {
  DKV_REQUIRE(layer_ptrs && mean && out, DKV_EINVAL, "dkv_centered_rows: null pointer");
  DKV_REQUIRE((cos == nullptr) == (sin == nullptr), DKV_EINVAL, "dkv_centered_rows: cos and sin go together");
  DKV_REQUIRE(dtype == DKV_F32 || dtype == DKV_F16 || dtype == DKV_BF16, DKV_EINVAL,
              "dkv_centered_rows: dtype %d not supported", dtype);
  DKV_REQUIRE(layers > 0 && heads > 0 && tokens >= 0 && head_dim > 0 && head_dim % 8 == 0, DKV_ESHAPE,
              "dkv_centered_rows: bad shape (layers=%d heads=%d tokens=%d head_dim=%d)", layers, heads, tokens,
              head_dim);
  DKV_REQUIRE(0 <= start && start <= end && end <= tokens, DKV_ESHAPE,
              "dkv_centered_rows: rows %d..%d outside 0..%d", start, end, tokens);
  if (end == start) return DKV_OK;
  const long cols = (long)layers * heads * (head_dim / (cos ? 8 : 4));
  const long col_blocks = (cols + 255) / 256, blocks = col_blocks * ((end - start + kRowTok - 1) / kRowTok);
  DKV_REQUIRE((long)layers * heads * head_dim < (1L << 30) && blocks < (1L << 31), DKV_ESHAPE,
              "dkv_centered_rows: too many rows or columns");
  const dim3 grid((unsigned)blocks);
  hipStream_t st = dkv::as_stream(stream);
#define DKV_CENTERED(T_, R_)                                                                                    \
  hipLaunchKernelGGL((centered_rows_kernel<T_, R_>), grid, dim3(256), 0, st, layer_ptrs, layers, heads, tokens, \
                     head_dim, cos, sin, mean, start, end, (int)col_blocks, out)
  const bool rot = cos != nullptr;
  if (dtype == DKV_F16) {
    if (rot) DKV_CENTERED(DKV_F16, true); else DKV_CENTERED(DKV_F16, false);
  } else if (dtype == DKV_BF16) {
    if (rot) DKV_CENTERED(DKV_BF16, true); else DKV_CENTERED(DKV_BF16, false);
  } else {
    if (rot) DKV_CENTERED(DKV_F32, true); else DKV_CENTERED(DKV_F32, false);
  }
#undef DKV_CENTERED
  return dkv::check_launch("dkv_centered_rows");
}

// ---------------------------------------------------------------------------
// K4c: merge hot + cold segments of selected tokens into full blobs.
// One workgroup per selected token; one thread per group.
// ---------------------------------------------------------------------------
// Merges token t's hot and cold segments into the full blob at refined + r * full_bytes and points the
// stream at it (one workgroup; one thread per group).
DKV_DEVICE void gather_token(const dkv_stream_t& s, const uint8_t* __restrict__ cold,
                             const int64_t* __restrict__ cold_tok_off, int t, int r, uint8_t* __restrict__ refined,
                             int64_t refined_base_off, int64_t* tok_off, int16_t* pieces) {
  const int G = s.order.groups, K = s.order.pieces;
  const int k = pieces[t];
  const int64_t off = tok_off[t];
  const int full_bytes = s.order.prefix_bytes[K];
  uint8_t* dst_tok = refined + (long)r * full_bytes;
  // One group per thread.  The full segment is the header and m_full plane words (at most 17
  // 32-bit words); word i comes from the hot segment (header and planes below m_hot) or the cold
  // one (the header when m_hot = 0, then planes m_hot..).  Every word's source is selected first
  // and all loads go out together (words past the segment re-read the header and are not stored).
  for (int g = threadIdx.x; g < G; g += blockDim.x) {
    const int m_hot = s.order.planes[(long)k * G + g];
    const int m_full = s.order.planes[(long)K * G + g];
    if (m_full == 0) continue;
    uint32_t* dst = (uint32_t*)(dst_tok + s.order.seg_off[(long)K * G + g]);
    const uint32_t* hseg = (const uint32_t*)(s.blob + off + s.order.seg_off[(long)k * G + g]);
    const uint32_t* cseg = (const uint32_t*)(cold + cold_tok_off[t] + s.order.cold_off[(long)k * G + g]);
    const uint32_t* head = m_hot > 0 ? hseg : cseg;
    const uint32_t* cplanes = m_hot > 0 ? cseg : cseg + 1;  // the cold part's plane words
    const int words = 1 + 2 * m_full;
    uint32_t v[17];
    v[0] = head[0];
#pragma unroll
    for (int i = 1; i < 17; ++i) {
      const int p = (i - 1) >> 1, j = (i - 1) & 1;
      const uint32_t* src = i >= words ? head : p < m_hot ? hseg + 1 + 2 * p + j : cplanes + 2 * (p - m_hot) + j;
      v[i] = *src;
    }
#pragma unroll
    for (int i = 0; i < 17; ++i)
      if (i < words) dst[i] = v[i];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    tok_off[t] = refined_base_off + (int64_t)r * full_bytes;
    pieces[t] = (int16_t)K;
  }
}


__global__ __launch_bounds__(64) void gather_cold_kernel(dkv_stream_t s, const uint8_t* __restrict__ cold,
                                                         const int64_t* __restrict__ cold_tok_off,
                                                         const int32_t* __restrict__ idx, uint8_t* __restrict__ refined,
                                                         int64_t refined_base_off, int64_t* tok_off,
                                                         int16_t* pieces) {
  gather_token(s, cold, cold_tok_off, idx[blockIdx.x], blockIdx.x, refined, refined_base_off, tok_off, pieces);
}

// ---------------------------------------------------------------------------
// K4c over any token list, without a host round trip.  refine_prepare_kernel:
// one thread per entry r of rows; in-range entries add the reference's cold
// bytes (full size - hot prefix of the token's current pieces,
// progressive.py:232) to fetched[0] and claim the token in owner[t] with the
// key (version << 32) | (2^31 - 1 - r): the largest key of this version is the
// token's first entry, and older versions' keys are smaller, so owner never
// needs clearing.  An entry outside 0..n-1 sets fetched[1].  The gather then
// runs one workgroup per entry and merges a token only from its first entry,
// and none at all if fetched[1] is set.  Integer sums: the result does not
// depend on the order in which entries are added.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void refine_prepare_kernel(const int32_t* __restrict__ rows, int k, int n,
                                                             const int16_t* __restrict__ pieces,
                                                             const int32_t* __restrict__ prefix_bytes, int K,
                                                             int64_t* owner, int64_t version, int64_t* fetched) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= k) return;
  const int t = rows[r];
  if (t < 0 || t >= n) {
    atomicOr((unsigned long long*)&fetched[1], 1ull);
    return;
  }
  const int64_t bytes = (int64_t)prefix_bytes[K] - prefix_bytes[pieces[t]];
  atomicAdd((unsigned long long*)&fetched[0], (unsigned long long)bytes);
  atomicMax((unsigned long long*)&owner[t], (unsigned long long)((version << 32) | (int64_t)(0x7fffffff - r)));
}

__global__ __launch_bounds__(64) void gather_owned_kernel(dkv_stream_t s, const uint8_t* __restrict__ cold,
                                                          const int64_t* __restrict__ cold_tok_off,
                                                          const int32_t* __restrict__ rows, int n,
                                                          uint8_t* __restrict__ refined, int64_t refined_base_off,
                                                          int64_t* tok_off, int16_t* pieces,
                                                          const int64_t* __restrict__ owner, int64_t version,
                                                          const int64_t* __restrict__ fetched) {
  const int r = blockIdx.x;
  const int t = rows[r];
  // uniform per workgroup: a bad list changes nothing; a repeated token is merged from its first entry
  if (fetched[1] != 0 || t < 0 || t >= n) return;
  if (owner[t] != ((version << 32) | (int64_t)(0x7fffffff - r))) return;
  gather_token(s, cold, cold_tok_off, t, r, refined, refined_base_off, tok_off, pieces);
}

extern "C" int dkv_gather_cold(const dkv_stream_t* s, const uint8_t* cold, const int64_t* cold_tok_off,
                               const int32_t* idx, int32_t k, uint8_t* refined, int64_t refined_base_off,
                               int64_t* tok_off, int16_t* pieces, void* stream) {
  int rc = dkv::check_stream(s, "dkv_gather_cold");
  if (rc) return rc;
  DKV_REQUIRE(s->format == DKV_FMT_PLANES, DKV_EINVAL, "dkv_gather_cold: only bit-plane streams have a cold tier");
  DKV_REQUIRE(cold && cold_tok_off && idx && refined && tok_off && pieces && s->order.cold_off, DKV_EINVAL,
              "dkv_gather_cold: null pointer");
  DKV_REQUIRE(k >= 0 && refined_base_off >= 0, DKV_ESHAPE, "dkv_gather_cold: bad k / offset");
  if (k == 0) return DKV_OK;
  dkv_stream_t view = *s;
  hipLaunchKernelGGL(gather_cold_kernel, dim3(k), dim3(64), 0, dkv::as_stream(stream), view, cold, cold_tok_off, idx,
                     refined, refined_base_off, tok_off, pieces);
  return dkv::check_launch("dkv_gather_cold");
}

extern "C" int dkv_refine_rows(const dkv_stream_t* s, int32_t n, const uint8_t* cold, const int64_t* cold_tok_off,
                               const int32_t* rows, int32_t k, uint8_t* refined, int64_t refined_base_off,
                               int64_t* tok_off, int16_t* pieces, int64_t* owner, int32_t version, int64_t* fetched,
                               void* stream) {
  int rc = dkv::check_stream(s, "dkv_refine_rows");
  if (rc) return rc;
  DKV_REQUIRE(s->format == DKV_FMT_PLANES, DKV_EINVAL, "dkv_refine_rows: only bit-plane streams have a cold tier");
  DKV_REQUIRE(cold && cold_tok_off && rows && refined && tok_off && pieces && owner && fetched && s->order.cold_off,
              DKV_EINVAL, "dkv_refine_rows: null pointer");
  DKV_REQUIRE(n >= 0 && k >= 0 && refined_base_off >= 0 && version > 0, DKV_ESHAPE,
              "dkv_refine_rows: bad n / k / offset / version");
  if (k == 0) return DKV_OK;
  const hipStream_t st = dkv::as_stream(stream);
  hipLaunchKernelGGL(refine_prepare_kernel, dim3((unsigned)((k + 255) / 256)), dim3(256), 0, st, rows, k, n,
                     (const int16_t*)pieces, s->order.prefix_bytes, s->order.pieces, owner, (int64_t)version, fetched);
  rc = dkv::check_launch("dkv_refine_rows");
  if (rc) return rc;
  dkv_stream_t view = *s;
  hipLaunchKernelGGL(gather_owned_kernel, dim3(k), dim3(64), 0, st, view, cold, cold_tok_off, rows, n, refined,
                     refined_base_off, tok_off, pieces, (const int64_t*)owner, (int64_t)version, (const int64_t*)fetched);
  return dkv::check_launch("dkv_refine_rows");
}

// ---------------------------------------------------------------------------
// Basis layouts.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void key_basis_kernel(const float* __restrict__ basis, int L, int H, int D, int R,
                                                        uint16_t* __restrict__ out) {
  const long id = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = (long)L * H * D * R;
  if (id >= total) return;
  // out index = (((l*G + g)*H + h)*D + dd)*64 + kk
  const int G = R / 64;
  const int kk = (int)(id & 63);
  long rest = id >> 6;
  const int dd = (int)(rest % D);
  rest /= D;
  const int h = (int)(rest % H);
  rest /= H;
  const int g = (int)(rest % G);
  const int l = (int)(rest / G);
  const float v = basis[((long)(l * H + h) * D + dd) * R + g * 64 + kk];
  half_t hv = (half_t)v;
  uint16_t bits;
  __builtin_memcpy(&bits, &hv, 2);
  out[id] = bits;
}

__global__ __launch_bounds__(256) void value_basis_kernel(const float* __restrict__ basis, int L, int H, int D, int R,
                                                          uint16_t* __restrict__ out) {
  const long id = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = (long)L * H * D * R;
  if (id >= total) return;
  // out index = ((l*H + h)*R + k)*D + dd
  const int dd = (int)(id % D);
  long rest = id / D;
  const int k = (int)(rest % R);
  const long lh = rest / R;
  const float v = basis[(lh * D + dd) * R + k];
  half_t hv = (half_t)v;
  uint16_t bits;
  __builtin_memcpy(&bits, &hv, 2);
  out[id] = bits;
}

static int check_basis_args(const float* basis, int L, int H, int D, int R, const uint16_t* out, const char* what) {
  DKV_REQUIRE(basis && out, DKV_EINVAL, "%s: null pointer", what);
  DKV_REQUIRE(L > 0 && H > 0 && D > 0 && R > 0 && R % 64 == 0, DKV_ESHAPE, "%s: bad shape L=%d H=%d D=%d R=%d", what,
              L, H, D, R);
  return DKV_OK;
}

extern "C" int dkv_prepare_key_basis(const float* basis, int32_t layers, int32_t kv_heads, int32_t head_dim,
                                     int32_t rank, uint16_t* out, void* stream) {
  int rc = check_basis_args(basis, layers, kv_heads, head_dim, rank, out, "dkv_prepare_key_basis");
  if (rc) return rc;
  const long total = (long)layers * kv_heads * head_dim * rank;
  hipLaunchKernelGGL(key_basis_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, dkv::as_stream(stream),
                     basis, layers, kv_heads, head_dim, rank, out);
  return dkv::check_launch("dkv_prepare_key_basis");
}

extern "C" int dkv_prepare_value_basis(const float* basis, int32_t layers, int32_t kv_heads, int32_t head_dim,
                                       int32_t rank, uint16_t* out, void* stream) {
  int rc = check_basis_args(basis, layers, kv_heads, head_dim, rank, out, "dkv_prepare_value_basis");
  if (rc) return rc;
  const long total = (long)layers * kv_heads * head_dim * rank;
  hipLaunchKernelGGL(value_basis_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, dkv::as_stream(stream),
                     basis, layers, kv_heads, head_dim, rank, out);
  return dkv::check_launch("dkv_prepare_value_basis");
}
