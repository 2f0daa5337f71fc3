// skinny.hip -- quantized-weight product for a few rows of x on MFMA (gfx950): 3 <= M <= 16, Q4_K, Q5_K
// and int4 (group a multiple of 128), plain or gated (SwiGLU / GELU-erf); 17 <= M <= 64, Q4_K and Q5_K.
//
// Role: Light's matmul_q and int4_gemv for small batches (ops/matmul_q.go:61-75,
// ops/int4.go:87-99) and its gated MLP projection (models/llama.go:1306-1328): a decode batch or
// a speculative step, where each weight is used M times.
//
// The int8-dot GEMV pays its dot products, scale arithmetic and a re-read of the weights (four
// rows of x per pass) once per row.  A wave here multiplies a tile of 16 weight rows by up to 16 rows of
// x with v_mfma_f32_16x16x32_f16, so the weight bytes are unpacked once whatever M is.  Q4_K, M = 6,
// layers replayed from a graph, that GEMV / this: gate/up 14336 x 4096 46.9 / 21.2 us (66 MB), down
// 4096 x 14336 33.1 / 16.8 (33 MB, the launch for the long rows' x among them).
// What bounds it now, by counters of these calls.  Gate/up: VALU issues on 60 % of a SIMD's cycles (3.4
// instructions per weight and lane; the unpacking's nine per eight weights are a third of them), MFMA
// is busy on a tenth, LDS bank conflicts fill a quarter of a CU's.  Down: VALU 37 %, MFMA 7 %; seven of
// ten requests to L2 are not for weights but for the records of x, which every CU reads, and waves wait.
//  * B holds exact integers in f16: sc * q (6-bit scale times quant, at most 63 * 31) for the K
//    formats, q for int4.  A nibble pair becomes (1024 + q) by one v_and_or_b32, and one packed
//    FMA by (sc, -1024 sc) leaves sc * q without rounding (high nibbles in place: 1024 + 16 q
//    with sc / 16).  d, dmin, s and z stay f32 and are applied to the f32 sums of a unit.
//  * A holds x as f16 under a power-of-two scale per row and unit (256 elements; int4 128), so
//    no x overflows and no element down to 2^-24 of its unit's largest is lost.  XM = kXPair (M <= 8)
//    splits x into two f16 (rows 0-7 the high parts, rows 8-15 the remainders): 22 bits, for the calls
//    whose int8 form keeps two levels.  XM = kXDup (M <= 8): rows 8-15 repeat rows 0-7, one f16 level
//    (2^-12, against 2^-8 of q8_1's single level).  XM = kX16: sixteen rows, one level.
//  * The lane group g = lane / 16 of a fragment holds the unit's g-th quarter (Q4_K: pair g),
//    so a lane unpacks only its own quarter's scales.  The minimum term is one more MFMA per
//    unit: minima (integers) against the sub-block sums of the rounded x, split in two f16.
//  * Waves split K; their 16 x 16 sums meet in LDS in wave order (deterministic).
//  * Weights reach LDS by direct loads of whole row runs.  (The MFMA operand order -- lane l reads
//    row l % 16 -- as plain loads touches a cache line per lane: 33 MB in 9.4 us against 6.9 us.)
#include "actq.hpp"
#include "decode.hpp"
#include "dma.hpp"
#include "internal.hpp"

#include <algorithm>
#include <atomic>

namespace hq {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kXDup = 0, kXPair = 1, kX16 = 2;  // how the sixteen A rows hold x
constexpr int kX64 = 3;                         // records of up to 64 rows (skinny_mid_kernel)

constexpr uint32_t K1024 = 0x64006400u;  // f16 pair (1024, 1024)

__device__ __forceinline__ f16x2 as_h2(uint32_t u) {
  f16x2 h;
  __builtin_memcpy(&h, &u, 4);
  return h;
}
__device__ __forceinline__ uint32_t as_u32(f16x2 h) {
  uint32_t u;
  __builtin_memcpy(&u, &h, 4);
  return u;
}
__device__ __forceinline__ f16x8 as_h8(u32x4 u) {
  f16x8 h;
  __builtin_memcpy(&h, &u, 16);
  return h;
}
// (w & mask) | (1024, 1024), as one v_and_or_b32 (VOP3 takes no literals: the mask in a scalar
// register, the bias in a vector one).
__device__ __forceinline__ f16x2 and_1024(uint32_t w, uint32_t mask, uint32_t bias) {
  uint32_t o;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(o) : "v"(w), "s"(mask), "v"(bias));
  return as_h2(o);
}
__device__ __forceinline__ f16x2 splat(float v) {
  const _Float16 h = (_Float16)v;
  return f16x2{h, h};
}

}  // namespace

// A source of x besides the dtypes: prepared activations (act layout).
constexpr int kXAct = -1;

struct SkinnyArgs {
  const void *x;           // (M, K) of x's dtype, or prepared activations
  int64_t in_q2, in_d;     // kXAct: offsets of q2 and (d, e)
  const uint8_t *xf;       // prepared x (skinny_x_kernel), long rows only
  const uint8_t *w0, *w1;  // weights (N, K); w1 = up projection (gated)
  const float *s, *z;      // int4 scales / zeros (N, K / G)
  void *out;               // (M, N)
  int M, N, K, nun, tiles, act;
  int xdt;                 // x's dtype (F32, BF16, F16; kXAct)
  int gpr, gunits;         // int4: groups per row, units per group
  uint32_t row_bytes, last;  // last: N row_bytes - 16
  // skinny_kernel's plan: groups of 256 k per chunk, chunks, pieces of a staged row, tile sets.
  int cg, nch, pr, tsets;
};

namespace {

// ---- weight formats -----------------------------------------------------------------
// A unit of KU weights of one row, ST MFMA steps of 32 k; lane group g holds the unit's weights
// [g KU / 4, (g + 1) KU / 4), eight per step.  Step i, slot j <-> weight KU / 4 * g + kofs(i, j).

// Q4_K / Q5_K super-block; lane group g: pair g (sub-blocks 2g, 2g + 1).  Step i covers quant
// bytes 4i .. 4i + 3 of the pair: slots 0-3 their low nibbles (bytes 0, 2, 1, 3), 4-7 the high.
template <bool Q5>
struct SkQk {
  static constexpr bool INT4 = false;
  static constexpr int DT = Q5 ? Q5_K : Q4_K;
  static constexpr int KU = 256, ST = 8, BB = Q5 ? 176 : 144, QO = Q5 ? 48 : 16;
  struct Raw {
    u32x4 hd, q0, q1, h0, h1;  // h0, h1: Q5_K's fifth bits
  };
  struct Sc {
    f16x2 a, am, b, bm;
    float d, dmin;
    u32x4 mn;
  };
  // The unit from a staged row of pr 16-byte pieces, piece j at position (j + rotation) % pr;
  // j0: the unit's first piece plus the rotation.
  __device__ static void load_lds(const uint8_t *row, int j0, int pr, int g, Raw &r) {
    auto at = [&](int j) __attribute__((always_inline)) {
      j += j0;
      j = j < pr ? j : j - pr;
      return *reinterpret_cast<const u32x4 *>(row + (j << 4));
    };
    r.hd = at(0);
    r.q0 = at(QO / 16 + 2 * g);
    r.q1 = at(QO / 16 + 1 + 2 * g);
    if constexpr (Q5) {
      r.h0 = at(1);
      r.h1 = at(2);
    }
  }
  __device__ static Sc decode(const Raw &r, int g) {
    Sc s;
    s.d = h2f(r.hd[0] & 0xffffu);
    s.dmin = h2f(r.hd[0] >> 16);
    // 6-bit (scale, min) of sub-blocks 2g, 2g + 1 (getScaleMinK4, quant/q4_k.go:83-89): g < 2
    // the low six bits of scales[j] / scales[j + 4]; g >= 2 nibbles of scales[j + 4] with the
    // top two bits of scales[j - 4] / scales[j].
    const int sh = 16 * (g & 1);
    const uint32_t t1 = (r.hd[1] >> sh) & 0xffffu, t2 = (r.hd[2] >> sh) & 0xffffu, t3 = (r.hd[3] >> sh) & 0xffffu;
    const uint32_t sel = g < 2 ? ~0u : 0u, mlo = g < 2 ? 0x3F3Fu : 0x0F0Fu, mhi = g < 2 ? 0u : 0x3030u;
    const uint32_t srcS = (t1 & sel) | (t3 & ~sel), srcM = (t2 & sel) | ((t3 >> 4) & ~sel);
    const uint32_t scp = (srcS & mlo) | ((t1 >> 2) & mhi), mnp = (srcM & mlo) | ((t2 >> 2) & mhi);
    const float sA = (float)(scp & 0xffu), sB = (float)(scp >> 8);
    s.a = splat(sA);
    s.am = splat(-1024.f * sA);
    if constexpr (Q5) {
      s.b = splat(sB);
      s.bm = splat(-1024.f * sB);
    } else {
      s.b = splat(0.0625f * sB);
      s.bm = splat(-64.f * sB);
    }
    const uint32_t mp = as_u32(f16x2{(_Float16)(float)(mnp & 0xffu), (_Float16)(float)(mnp >> 8)});
    s.mn = u32x4{mp, mp, 0, 0};
    return s;
  }
  __device__ static f16x8 frag(const Raw &r, const Sc &s, int g, int i) {
    const uint32_t w = i < 4 ? r.q0[i & 3] : r.q1[i & 3];
    u32x4 o;
    if constexpr (Q5) {
      const uint32_t hb = (i < 4 ? r.h0[i & 3] : r.h1[i & 3]) >> (2 * g);
      const uint32_t l = (w & 0x0F0F0F0Fu) | ((hb & 0x01010101u) << 4);
      const uint32_t h = ((w >> 4) & 0x0F0F0F0Fu) | ((hb & 0x02020202u) << 3);
      constexpr uint32_t B64 = 0x64646464u;  // (byte b, 0x64) = f16 1024 + b
      o[0] = as_u32(__builtin_elementwise_fma(as_h2(__builtin_amdgcn_perm(B64, l, 0x04020400u)), s.a, s.am));
      o[1] = as_u32(__builtin_elementwise_fma(as_h2(__builtin_amdgcn_perm(B64, l, 0x04030401u)), s.a, s.am));
      o[2] = as_u32(__builtin_elementwise_fma(as_h2(__builtin_amdgcn_perm(B64, h, 0x04020400u)), s.b, s.bm));
      o[3] = as_u32(__builtin_elementwise_fma(as_h2(__builtin_amdgcn_perm(B64, h, 0x04030401u)), s.b, s.bm));
    } else {
      const uint32_t t = w >> 8;
      o[0] = as_u32(__builtin_elementwise_fma(and_1024(w, 0x000F000Fu, K1024), s.a, s.am));
      o[1] = as_u32(__builtin_elementwise_fma(and_1024(t, 0x000F000Fu, K1024), s.a, s.am));
      o[2] = as_u32(__builtin_elementwise_fma(and_1024(w, 0x00F000F0u, K1024), s.b, s.bm));
      o[3] = as_u32(__builtin_elementwise_fma(and_1024(t, 0x00F000F0u, K1024), s.b, s.bm));
    }
    return as_h8(o);
  }
};

// int4 (quant.Int4): 128 codes of one row, one group's scale and zero; lane group g: code words
// 4g .. 4g + 3.  Step i is word 4g + i: slots hold nibbles 0, 4, 2, 6, 1, 5, 3, 7.
struct SkI4 {
  static constexpr bool INT4 = true;
  static constexpr int KU = 128, ST = 4, BB = 64;
  struct Raw {
    u32x4 q;
  };
  struct Sc {};
  __device__ static void load_lds(const uint8_t *row, int j0, int pr, int g, Raw &r) {
    int j = j0 + g;
    j = j < pr ? j : j - pr;
    r.q = *reinterpret_cast<const u32x4 *>(row + (j << 4));
  }
  __device__ static Sc decode(const Raw &, int) { return {}; }
  __device__ static f16x8 frag(const Raw &r, const Sc &, int, int i) {
    const uint32_t w = r.q[i], t = w >> 8;
    const f16x2 k = splat(-1024.f), k16 = splat(-64.f), i16 = splat(0.0625f);
    const u32x4 o = {as_u32(and_1024(w, 0x000F000Fu, K1024) + k), as_u32(and_1024(t, 0x000F000Fu, K1024) + k),
                     as_u32(__builtin_elementwise_fma(and_1024(w, 0x00F000F0u, K1024), i16, k16)),
                     as_u32(__builtin_elementwise_fma(and_1024(t, 0x00F000F0u, K1024), i16, k16))};
    return as_h8(o);
  }
};

// ---- x: rows of a unit in A fragment order ----------------------------------------------
// Record of one unit for P rows: fragments [ST][4][P] x 16 B, then (K formats) sub-block sums
// [4][P] x 8 B = (hi 2g, hi 2g+1, lo 2g, lo 2g+1), then by A row xs f32 [16] (the row's power of
// two; kX64: [64]) and (int4) sx f32 [16] (the unit's sum).  In memory P is M (kXPair: 2 M), so that a CU
// fetches no padding (every CU reads all of x from L2); in LDS the A rows, 8 or 16.
template <class F, int XM>
struct XRec {
  static constexpr int ROWS = XM == kXDup ? 8 : 16;
  __host__ __device__ static constexpr int rows(int M) { return XM == kXPair ? 2 * M : M; }
  __host__ __device__ static constexpr int mins(int P) { return F::ST * 4 * P * 16; }
  __host__ __device__ static constexpr int xs(int P) { return mins(P) + (F::INT4 ? 0 : 32 * P); }
  __host__ __device__ static constexpr int bytes(int P) { return xs(P) + (XM == kX64 ? 256 : F::INT4 ? 128 : 64); }
  static constexpr int BYTES = bytes(ROWS);
};

template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
template <int CTRL>
__device__ __forceinline__ uint32_t dppu(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}
__device__ __forceinline__ float fdot2(f16x2 a, f16x2 b, float c) { return __builtin_amdgcn_fdot2(a, b, c, false); }

// 256 consecutive elements of x row m (four per lane) into the record(s) for P rows at `rec`: one
// unit of a K format, or two int4 units (lanes 32-63 the second).
template <class F, int XM>
__device__ __forceinline__ void convert_row(const float (&v)[4], int m, int lane, uint8_t *rec, int P) {
  using R = XRec<F, XM>;
  // Magnitudes compare as integers (a NaN above Inf, so no canonicalising max).
  auto mag = [](float y) { return __float_as_uint(y) & 0x7fffffffu; };
  auto umax = [](uint32_t p, uint32_t q) { return p > q ? p : q; };
  uint32_t mx = umax(umax(mag(v[0]), mag(v[1])), umax(mag(v[2]), mag(v[3])));
  mx = umax(mx, dppu<0xB1>(mx));
  mx = umax(mx, dppu<0x4E>(mx));
  mx = umax(mx, dppu<0x141>(mx));
  mx = umax(mx, dppu<0x140>(mx));
  auto at = [&](int l) { return (uint32_t)__builtin_amdgcn_readlane((int)mx, l); };
  const uint32_t m01 = umax(at(0), at(16)), m23 = umax(at(32), at(48));
  // The largest |x| scaled to [2^9, 2^10): a sum of 32 stays below f16's range.  (Inf: unscaled;
  // below 2^-117: the largest scale.)
  auto expo = [](uint32_t u) { return u >= 0x7f800000u ? 136u : (u < (10u << 23) ? 10u : u >> 23); };
  uint32_t e;
  if constexpr (F::INT4) {
    const uint32_t e01 = expo(m01), e23 = expo(m23);
    e = lane < 32 ? e01 : e23;
  } else {
    e = expo(umax(m01, m23));
  }
  const float f = __uint_as_float((263u - e) << 23), xs = __uint_as_float((e - 9u) << 23);
  const f16x2 ones = {(_Float16)1.f, (_Float16)1.f};
  _Float16 hi[4], lo[4];
  float sl = 0.f;
#pragma unroll
  for (int j = 0; j < 4; j++) hi[j] = (_Float16)__fmaf_rn(v[j], f, 0.f);
  const float sh = fdot2(f16x2{hi[2], hi[3]}, ones, fdot2(f16x2{hi[0], hi[1]}, ones, 0.f));
  if constexpr (XM == kXPair) {
#pragma unroll
    for (int j = 0; j < 4; j++) lo[j] = (_Float16)__fmaf_rn(v[j], f, -(float)hi[j]);
    sl = fdot2(f16x2{lo[2], lo[3]}, ones, fdot2(f16x2{lo[0], lo[1]}, ones, 0.f));
  }
  auto put = [&](const _Float16 (&h)[4], float s, int row, int arow) __attribute__((always_inline)) {
    s += dppf<0xB1>(s);
    s += dppf<0x4E>(s);
    s += dppf<0x141>(s);  // the sum over eight lanes (32 elements), in each of them
    if constexpr (F::INT4) {
      uint8_t *rc = rec + (lane >> 5) * R::bytes(P);
      const int l5 = lane & 31, g = l5 >> 3, i = (l5 >> 1) & 3;
      // Word i's nibbles 0-3 (even lane) and 4-7 (odd): slots 0-3 are 0, 4, 2, 6, slots 4-7
      // 1, 5, 3, 7, so each lane of the pair writes one half.
      const uint32_t a02 = as_u32(f16x2{h[0], h[2]}), a13 = as_u32(f16x2{h[1], h[3]});
      const bool odd = lane & 1;
      const uint32_t mine = odd ? a13 : a02, give = odd ? a02 : a13;
      const uint32_t got = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)give, 0xB1, 0xF, 0xF, false);
      // even: (0, 2) with (4, 6); odd: (1, 3) of the partner with its own (5, 7)
      const uint32_t first = odd ? got : mine, second = odd ? mine : got;
      const u32x2 o = {__builtin_amdgcn_perm(second, first, 0x05040100u), __builtin_amdgcn_perm(second, first, 0x07060302u)};
      *reinterpret_cast<u32x2 *>(rc + ((i * 4 + g) * P + row) * 16 + (odd ? 8 : 0)) = o;
      s += dppf<0x140>(s);  // sixteen lanes
      s += __shfl_xor(s, 16, 64);
      if (l5 == 0) {
        *reinterpret_cast<float *>(rc + R::xs(P) + 4 * arow) = xs;
        *reinterpret_cast<float *>(rc + R::xs(P) + 64 + 4 * arow) = s;
      }
    } else {
      const int g = lane >> 4, e16 = lane & 15, i = e16 & 7;
      const u32x2 o = {as_u32(f16x2{h[0], h[2]}), as_u32(f16x2{h[1], h[3]})};
      *reinterpret_cast<u32x2 *>(rec + ((i * 4 + g) * P + row) * 16 + (e16 & 8)) = o;
      if ((lane & 7) == 0) {
        const _Float16 a = (_Float16)s, b = (_Float16)(s - (float)a);
        _Float16 *mp = reinterpret_cast<_Float16 *>(rec + R::mins(P) + (g * P + row) * 8) + ((lane >> 3) & 1);
        mp[0] = a;
        mp[2] = b;
      }
      if (lane == 0) *reinterpret_cast<float *>(rec + R::xs(P) + 4 * arow) = xs;
    }
  };
  put(hi, sh, m, m);
  if constexpr (XM == kXPair) put(lo, sl, P / 2 + m, m + 8);
}

// Elements k .. k + 3 of x row m (k % 4 == 0).
template <int XDT>
__device__ __forceinline__ void load_x4(const SkinnyArgs &a, int m, int64_t k, float (&v)[4]) {
  const int64_t i = (int64_t)m * a.K + k;
  if constexpr (XDT == F32) {
    const f32x4 f = *reinterpret_cast<const f32x4 *>(static_cast<const float *>(a.x) + i);
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = f[j];
  } else if constexpr (XDT == kXAct) {
    const uint8_t *p = static_cast<const uint8_t *>(a.x);
    const uint32_t q1 = *reinterpret_cast<const uint32_t *>(p + i), q2 = *reinterpret_cast<const uint32_t *>(p + a.in_q2 + i);
    const float2 de = reinterpret_cast<const float2 *>(p + a.in_d)[i >> 5];
#pragma unroll
    for (int j = 0; j < 4; j++)
      v[j] = __fmaf_rn(de.y, (float)(int8_t)(q2 >> (8 * j)), __fmul_rn(de.x, (float)(int8_t)(q1 >> (8 * j))));
  } else {
    const u32x2 u = *reinterpret_cast<const u32x2 *>(static_cast<const uint16_t *>(a.x) + i);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t h = (j & 1) ? u[j >> 1] >> 16 : u[j >> 1] & 0xffffu;
      v[j] = XDT == BF16 ? bf2f(h) : h2f(h);
    }
  }
}

// A wave's view of one unit of x.
template <class F>
struct XFrag {
  u32x4 f[F::ST];
  u32x2 mn;
  f32x4 xs, sx;
};

template <class F, int XM>
__device__ __forceinline__ void load_frag(const uint8_t *rec, int lane, XFrag<F> &x) {
  using R = XRec<F, XM>;
  const int g = lane >> 4, r = lane & (R::ROWS - 1);
#pragma unroll
  for (int i = 0; i < F::ST; i++) x.f[i] = *reinterpret_cast<const u32x4 *>(rec + ((i * 4 + g) * R::ROWS + r) * 16);
  const int q = XM == kXDup ? g & 1 : g;  // D rows 4g .. 4g + 3 of this lane
  x.xs = *reinterpret_cast<const f32x4 *>(rec + R::xs(R::ROWS) + 16 * q);
  if constexpr (F::INT4)
    x.sx = *reinterpret_cast<const f32x4 *>(rec + R::xs(R::ROWS) + 64 + 16 * q);
  else
    x.mn = *reinterpret_cast<const u32x2 *>(rec + R::mins(R::ROWS) + (g * R::ROWS + r) * 8);
}

// The same from a record in memory for P = rows(M) rows (A rows past M repeat row M - 1).  No load
// sits in a branch, so the compiler's wait counts stay exact.
template <class F, int XM>
__device__ __forceinline__ void load_frag_rows(const uint8_t *rec, int lane, int M, XFrag<F> &x) {
  using R = XRec<F, XM>;
  const int g = lane >> 4, r = lane & 15, P = R::rows(M);
  const bool low = XM == kXPair && r >= 8;
  const int k = low ? r - 8 : r, pr = (k < M ? k : M - 1) + (low ? M : 0);
#pragma unroll
  for (int i = 0; i < F::ST; i++) x.f[i] = *reinterpret_cast<const u32x4 *>(rec + i * (64 * P) + (g * P + pr) * 16);
  x.xs = *reinterpret_cast<const f32x4 *>(rec + R::xs(P) + 16 * g);
  if constexpr (F::INT4)
    x.sx = *reinterpret_cast<const f32x4 *>(rec + R::xs(P) + 64 + 16 * g);
  else
    x.mn = *reinterpret_cast<const u32x2 *>(rec + R::mins(P) + (g * P + pr) * 8);
}

// acc += one unit of a 16-row tile (s, z: int4 scale and zero of the lane's row).
template <class F>
__device__ __forceinline__ void unit_mma(const typename F::Raw &w, const XFrag<F> &x, int g, float s, float z, f32x4 &acc) {
  const typename F::Sc sc = F::decode(w, g);
  f32x4 q = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < F::ST; i++)
    q = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_h8(x.f[i]), F::frag(w, sc, g, i), q, 0, 0, 0);
  if constexpr (F::INT4) {
#pragma unroll
    for (int r = 0; r < 4; r++) acc[r] = __fmaf_rn(s * x.xs[r], __fmaf_rn(-z, x.sx[r], q[r]), acc[r]);
  } else {
    f32x4 m = {0.f, 0.f, 0.f, 0.f};
    m = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_h8(u32x4{x.mn[0], x.mn[1], 0, 0}), as_h8(sc.mn), m, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; r++) acc[r] = __fmaf_rn(x.xs[r], __fmaf_rn(sc.d, q[r], -(sc.dmin * m[r])), acc[r]);
  }
}

// x's non-finite elements of row m in [k0, k1) times their weights of row n, if there are any.  An
// infinite x meets the split weights (sc * q and a minimum; int4: q and z) as Inf - Inf, so an output
// that is not finite is worked out again from these, as f32 arithmetic has it (the finite elements add
// nothing to them): by one pass at the kernel's end, for the threads that saw such an output.
template <class F>
__device__ __forceinline__ bool nonfinite_sum(const SkinnyArgs &a, const uint8_t *w, int m, int n, int k0, int k1, float &s) {
  s = 0.f;
  bool any = false;
#pragma unroll 1
  for (int k = k0; k < k1 && s == s; k += 8) {  // (NaN stays NaN)
    const int64_t i = (int64_t)m * a.K + k;
    float v[8];
    if (a.xdt == F32) {
      const f32x4 *p = reinterpret_cast<const f32x4 *>(static_cast<const float *>(a.x) + i);
      const f32x4 p0 = p[0], p1 = p[1];
#pragma unroll
      for (int j = 0; j < 8; j++) v[j] = j < 4 ? p0[j] : p1[j - 4];
    } else {
      const u32x4 p = *reinterpret_cast<const u32x4 *>(static_cast<const uint16_t *>(a.x) + i);
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const uint32_t h = (j & 1) ? p[j >> 1] >> 16 : p[j >> 1] & 0xffffu;
        v[j] = a.xdt == BF16 ? bf2f(h) : h2f(h);
      }
    }
    bool bad = false;
#pragma unroll
    for (int j = 0; j < 8; j++) bad |= !__builtin_isfinite(v[j]);
    if (!bad) continue;
    any = true;
    float d[8];
    if constexpr (F::INT4) {
      const int64_t gi = (int64_t)n * a.gpr + k / (128 * a.gunits);
      const uint32_t q = reinterpret_cast<const uint32_t *>(w + (int64_t)n * a.row_bytes)[k >> 3];
#pragma unroll
      for (int j = 0; j < 8; j++) d[j] = a.s[gi] * ((float)((q >> (4 * j)) & 15) - a.z[gi]);
    } else {
      decode8<F::DT>(w + (int64_t)n * a.row_bytes, k >> 3, d);
    }
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (!__builtin_isfinite(v[j])) s += v[j] * d[j];
  }
  return any;
}

template <int ODT>
__device__ __forceinline__ void store_y(void *out, int64_t i, float y) {
  if constexpr (ODT == F32)
    static_cast<float *>(out)[i] = y;
  else if constexpr (ODT == BF16)
    static_cast<uint16_t *>(out)[i] = f2bf_rne(y);
  else
    static_cast<uint16_t *>(out)[i] = f2h_rne(y);
}

// Output (m, n) again, where row m of x holds a non-finite element (gate and up both have it then).
template <class F, bool GATED, int ODT>
__device__ __forceinline__ void settle(const SkinnyArgs &a, int m, int n) {
  float y, u;
  if (m >= a.M || n >= a.N || !nonfinite_sum<F>(a, a.w0, m, n, 0, a.K, y)) return;
  if constexpr (GATED) {
    nonfinite_sum<F>(a, a.w1, m, n, 0, a.K, u);
    y = gate_act(y, a.act) * u;
  }
  store_y<ODT>(a.out, (int64_t)m * a.N + n, y);
}

// A direct load of 16 bytes per lane from base + off (base uniform).
__device__ __forceinline__ void dma16s(const uint8_t *base, uint32_t off, uint32_t lds_base) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds_base) : "memory", "m0");
#pragma clang diagnostic pop
}

// At most n (0 .. 4, wave-uniform) vector-memory operations outstanding.
__device__ __forceinline__ void wait_few(int n) {
  if (n >= 4)
    wait_vm<4>();
  else if (n == 3)
    wait_vm<3>();
  else if (n == 2)
    wait_vm<2>();
  else if (n == 1)
    wait_vm<1>();
  else
    wait_vm<0>();
}

// Byte offset, from its first row, of LDS piece p of staged rows of pr pieces: piece
// (p % pr - rot (row % 16)) mod pr of row p / pr.
__device__ __forceinline__ uint32_t piece_off(int p, int pr, float ipr, int rot, uint32_t row_bytes) {
  const int row = (int)(((float)p + 0.5f) * ipr);  // p / pr: p < 2^12, so the quotient is exact
  int j = p - row * pr - rot * (row & 15);
  j = j < 0 ? j + pr : j;
  return (uint32_t)row * row_bytes + (uint32_t)j * 16;
}

// acc += the wave's group (number kg of the stage, units u0 ..) of the staged 16-row tile.
// int4: scales at stage + raw, SU per row, zeros ZO floats on.
template <class F, int SU, int ZO = 512, int UPG>
__device__ __forceinline__ void group_mma(const uint8_t *stage, int raw_bytes, int row, int kg, int u0, int nun, int pr, int rot,
                                          int g, const XFrag<F> (&x)[UPG], f32x4 &acc) {
#pragma unroll
  for (int q = 0; q < UPG; q++) {
    if (u0 + q >= nun) continue;  // wave-uniform
    typename F::Raw raw;
    float us = 0.f, uz = 0.f;
    F::load_lds(stage + (row * pr << 4), (kg * UPG + q) * (F::BB / 16) + rot * (row & 15), pr, g, raw);
    if constexpr (F::INT4) {
      const float *sp = reinterpret_cast<const float *>(stage + raw_bytes) + row * SU + kg * UPG + q;
      us = sp[0];
      uz = sp[ZO];
    }
    unit_mma<F>(raw, x[q], g, us, uz, acc);
  }
}

// Sums KW parts (1 KB apart: [16 weight rows][16 A rows]) of (weight row c, x row m).
template <int KW, int XM>
__device__ __forceinline__ float sum_parts(const float *p, int c, int m) {
  float y = 0.f;
#pragma unroll
  for (int k = 0; k < KW; k++) {
    float v = p[k * 256 + c * 16 + m];
    if constexpr (XM == kXPair) v += p[k * 256 + c * 16 + m + 8];
    y += v;
  }
  return y;
}

// LDS of skinny_kernel (bytes).  A stage holds one item: up to 256 row-groups of 256 k (16 rows x
// 16 groups, or 16 TG rows x KW groups) of raw weights, and int4's scales and zeros of its rows.
template <class F, int XM>
struct SkinnyLds {
  static constexpr int UPG = 256 / F::KU, GB = UPG * F::BB;  // units and bytes of a row group
  static constexpr int RAW = 256 * GB;
  static constexpr int STAGE = RAW + (F::INT4 ? 2 * 512 * 4 : 0);
  static constexpr int PARTS = 2 * 16 * 1024;
  // The conversion of resident x: eight or sixteen waves at a time, in the place of the last
  // stage and the parts (or of the parts alone).
  static constexpr int CW = XRec<F, XM>::ROWS == 8 ? 16 : 8;
  static constexpr int CONV = CW * UPG * XRec<F, XM>::BYTES;
  static constexpr int S3 = 2 * STAGE + (STAGE + PARTS > CONV ? STAGE + PARTS : CONV);
  static constexpr int S2 = 2 * STAGE + (PARTS > CONV ? PARTS : CONV);
  static constexpr int NS = S3 <= 160 * 1024 ? 3 : 2;
  static constexpr int BYTES = NS == 3 ? S3 : S2;
  static_assert(BYTES <= 160 * 1024, "LDS");
};

}  // namespace

// K <= 4096.  One 1024-thread workgroup per CU.  A tile is 16 weight rows; the sixteen waves are KW
// parts of K (one group of 256 k each, its x converted into registers once) times TG = 16 / KW
// tiles.  An item is a tile set's rows of one weight; tile sets are dealt in grid order.  Items
// are staged in LDS by direct loads of whole rows (the pieces of a row rotated by the row, so
// that the sixteen rows' reads fall into different banks), NS - 1 ahead; one barrier per item
// publishes a stage, frees the one before and hands over the item's parts.
template <class F, int KW, bool GATED, int XM, int XR, int XDT, int ODT>
__global__ __launch_bounds__(1024) void skinny_kernel(SkinnyArgs a) {
  using R = XRec<F, XM>;
  using T = SkinnyLds<F, XM>;
  constexpr int TG = 16 / KW, NW = GATED ? 2 : 1, NS = T::NS, UPG = T::UPG;
  constexpr int XROWS = XM == kX16 ? 16 : 8;
  constexpr int NO = (TG * 16 * XROWS + 1023) / 1024;  // outputs per thread and item
  extern __shared__ __align__(16) uint8_t smem[];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int g = lane >> 4, r = lane & 15;
  const int kw = wave % KW, tg = wave / KW;
  const int nkg = (a.K + 255) >> 8, pr = a.pr;
  const int rot = pr & 1 || pr < 16 ? 0 : 1;
  const int npiece = 16 * TG * pr;
  const int nd = (((npiece + 63) >> 6) - wave + 15) >> 4;  // this wave's direct loads per item (at most 3)

  // This wave's pieces: load q = wave + 16 k, lane's LDS piece 64 q + lane holds piece
  // (jj - rot * row) of its row.
  uint32_t poff[3];
  const float ipr = 1.0f / (float)pr;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    int p = (wave + 16 * k) * 64 + lane;
    p = p < npiece ? p : npiece - 1;
    poff[k] = piece_off(p, pr, ipr, rot, a.row_bytes);
  }
  const int niter = (a.tsets - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
  auto row0_of = [&](int it) __attribute__((always_inline)) {
    return ((int)blockIdx.x + it * (int)gridDim.x) * TG * 16;
  };
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  auto issue = [&](int it, int j, int slot) __attribute__((always_inline)) {
    if (it >= niter) it = niter - 1;  // (the ring's last loads repeat)
    const int row0 = row0_of(it);
    const uint8_t *w = GATED && j ? a.w1 : a.w0;
    const uint32_t base = (uint32_t)row0 * a.row_bytes;
    const uint32_t dst = lds0 + slot * T::STAGE;
#pragma unroll
    for (int k = 0; k < 3; k++)
      if (k < nd) {  // wave-uniform
        uint32_t o = base + poff[k];
        o = o < a.last ? o : a.last;  // rows past N: any valid bytes
        dma16s(w, o, __builtin_amdgcn_readfirstlane(dst + (wave + k * 16) * 1024));
      }
    if constexpr (F::INT4) {
      // 512 scales (waves 0-7) and zeros (8-15): [row][unit of the row's 2 KW].
      const int f = (wave & 7) * 64 + lane, lr = f / (2 * KW);
      int row = row0 + lr, u = f - lr * (2 * KW);
      row = row < a.N ? row : a.N - 1;
      u = u < a.nun ? u : a.nun - 1;
      if (a.gunits != 1) u = (int)((uint32_t)u / (uint32_t)a.gunits);
      dma4(((wave < 8 ? a.s : a.z) + (int64_t)row * a.gpr) + u, __builtin_amdgcn_readfirstlane(dst + T::RAW + wave * 256));
    }
  };
  const int ndi = nd + (F::INT4 ? 1 : 0);
#pragma unroll
  for (int i = 0; i < NS - 1; i++) issue(i / NW, i % NW, i);

  // The wave's group of x (units kw UPG ..).  Rows are converted without a branch between them, so that
  // their chains interleave (rows past M repeat row M - 1).
  XFrag<F> xf[UPG];
  {
    uint8_t *conv = smem + 2 * T::STAGE;
    int64_t k = (int64_t)kw * 256 + lane * 4;
    k = k < a.K ? k : a.K - 4;
    auto load_frags = [&](const uint8_t *rec) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < UPG; q++) load_frag<F, XM>(rec + q * R::BYTES, lane, xf[q]);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    if constexpr (TG > 1) {
      // The TG waves of a group convert XR / TG of its rows each (M = 16, 4345 x 256: 12.6 us with every
      // wave converting all rows of its group, 5.6 so; M = 9, 12357 x 512, Q5_K: 12.7, 6.1).
      constexpr int RW = (XR + TG - 1) / TG;
      uint8_t *rec = conv + kw * (UPG * R::BYTES);
      float xv[RW][4];
#pragma unroll
      for (int i = 0; i < RW; i++) load_x4<XDT>(a, tg + i * TG < a.M ? tg + i * TG : a.M - 1, k, xv[i]);
      if (XR >= TG || tg < XR) {
#pragma unroll
        for (int i = 0; i < RW; i++) convert_row<F, XM>(xv[i], tg + i * TG, lane, rec, R::ROWS);
      }
      __syncthreads();
      load_frags(rec);
      __syncthreads();  // the stage and the parts take the place
    } else {
      float xv[XR][4];
#pragma unroll
      for (int m = 0; m < XR; m++) load_x4<XDT>(a, m < a.M ? m : a.M - 1, k, xv[m]);
#pragma unroll
      for (int ph = 0; ph < 16 / T::CW; ph++) {
        if (wave / T::CW == ph) {
          uint8_t *rec = conv + (wave % T::CW) * (UPG * R::BYTES);
#pragma unroll
          for (int m = 0; m < XR; m++) convert_row<F, XM>(xv[m], m, lane, rec, R::ROWS);
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          load_frags(rec);
        }
        __syncthreads();  // the next waves' records, then the stage and the parts, take the place
      }
    }
  }

  float *part = reinterpret_cast<float *>(smem + NS * T::STAGE);
  float gs[NO];
  bool bad = false;  // an output of this thread is not finite
  // Outputs of (iteration, weight j): sums the KW parts of (tile, x row, weight row) in order; the
  // gate's sums wait in registers for the up weight's.
  auto reduce = [&](int it, int j, int buf) __attribute__((always_inline)) {
    const int row0 = row0_of(it);
    const float *pb = part + buf * (16 * 256);
#pragma unroll
    for (int k = 0; k < NO; k++) {
      const int o = t + 1024 * k;
      if (o >= TG * 16 * XROWS) continue;
      const int c = o & 15, m = (o >> 4) & (XROWS - 1), q = (o >> 4) / XROWS;
      float y = sum_parts<KW, XM>(pb + q * KW * 256, c, m);
      const int col = row0 + q * 16 + c;
      if (GATED && j == 0) {
        gs[k] = y;
      } else if (m < a.M && col < a.N) {
        if constexpr (GATED) y = gate_act(gs[k], a.act) * y;
        bad |= !__builtin_isfinite(y);
        store_y<ODT>(a.out, (int64_t)m * a.N + col, y);
      }
    }
  };
  const bool have = kw < nkg;
  int slot = 0, nslot = NS - 1;
  for (int it = 0; it < niter; it++) {
#pragma unroll
    for (int j = 0; j < NW; j++) {
      if constexpr (NS == 3)
        wait_few(ndi);  // the next item's loads may be in flight
      else
        wait_vm<0>();
      __syncthreads();
      issue(it + (j + NS - 1) / NW, (j + NS - 1) % NW, nslot);
      if (NW == 2 && j == 1)
        reduce(it, 0, 0);
      else if (it > 0)
        reduce(it - 1, NW - 1, NW == 2 ? 1 : (it - 1) & 1);
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      if (have)
        group_mma<F, 2 * KW>(smem + slot * T::STAGE, T::RAW, tg * 16 + r, kw, kw * UPG, a.nun, pr, rot, g, xf, acc);
      *reinterpret_cast<f32x4 *>(part + (NW == 2 ? j : it & 1) * (16 * 256) + wave * 256 + r * 16 + 4 * g) = acc;
      slot = slot + 1 == NS ? 0 : slot + 1;
      nslot = nslot + 1 == NS ? 0 : nslot + 1;
    }
  }
  __syncthreads();
  reduce(niter - 1, NW - 1, NW == 2 ? 1 : (niter - 1) & 1);
  wait_vm<0>();  // the last (repeated) stages have landed before the LDS is given up
  if constexpr (XDT >= 0)
    if (bad) {
#pragma unroll 1
      for (int it = 0; it < niter; it++)
#pragma unroll 1
        for (int o = t; o < TG * 16 * XROWS; o += 1024)
          settle<F, GATED, ODT>(a, (o >> 4) & (XROWS - 1), row0_of(it) + (o >> 4) / XROWS * 16 + (o & 15));
    }
}

// Longer rows: RT tiles per workgroup, x from skinny_x_kernel's records.  Items are (K chunk of up
// to 14 groups, tile, weight), one group per compute wave (14); two more waves issue every
// direct load, NS - 1 items ahead, because a wave's wait counts its loads in order: a wave that
// loads x into registers cannot leave newer weight loads in flight when it uses them.
template <class F>
struct SkinnyLongLds {
  static constexpr int CG = 14, UPG = 256 / F::KU, GB = UPG * F::BB;
  static constexpr int RAW = (16 * CG * GB + 1023) / 1024 * 1024;
  static constexpr int SC = F::INT4 ? 16 * CG * 2 / 64 : 0;  // direct loads of scales (and of zeros)
  static constexpr int STAGE = RAW + 2 * SC * 256;
  static constexpr int ND = (RAW / 1024 + 1) / 2 + SC;  // a loading wave's loads per item
  static constexpr int NS = 4 * STAGE <= 160 * 1024 ? 4 : 3;
  static constexpr int BYTES = NS * STAGE;
  static_assert((NS - 2) * ND < 64 && 2 * 14 * 1024 <= BYTES, "wait counts; the parts reuse the stages");
};

template <class F, int RT, bool GATED, int XM, int ODT>
__global__ __launch_bounds__(1024) void skinny_long_kernel(SkinnyArgs a) {
  using R = XRec<F, XM>;
  using T = SkinnyLongLds<F>;
  constexpr int NW = GATED ? 2 : 1, NT = RT * NW, NS = T::NS, UPG = T::UPG, CW = T::CG;
  constexpr int XROWS = XM == kX16 ? 16 : 8;
  extern __shared__ __align__(16) uint8_t smem[];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int g = lane >> 4, r = lane & 15;
  const int nch = a.nch, cg = a.cg, pr = a.pr;
  const int rot = pr & 1 || pr < 16 ? 0 : 1;
  const int nitem = nch * NT;
  auto row0_of = [&](int i) __attribute__((always_inline)) { return ((int)blockIdx.x * RT + i) * 16; };

  f32x4 acc[NT];
#pragma unroll
  for (int i = 0; i < NT; i++) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (wave >= CW) {
    // ---- loads ----
    const int pw = wave - CW;
    const int npiece = 16 * pr, ninst = (npiece + 63) >> 6;
    const float ipr = 1.0f / (float)pr;
    constexpr int NDW = T::ND - T::SC;
    uint32_t poff[NDW];
#pragma unroll
    for (int k = 0; k < NDW; k++) {
      int q = pw + 2 * k;
      q = q < ninst ? q : ninst - 1;
      int p = q * 64 + lane;
      p = p < npiece ? p : npiece - 1;
      poff[k] = piece_off(p, pr, ipr, rot, a.row_bytes);
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    int ic = 0, ik = 0, islot = 0;  // the next item to request: chunk, tile x weight, slot
    auto issue = [&]() __attribute__((always_inline)) {
      const int c = ic < nch ? ic : nch - 1;  // (the ring's last loads repeat)
      const int row0 = row0_of(ik / NW);
      const uint8_t *w = GATED && (ik & 1) ? a.w1 : a.w0;
      const uint32_t base = (uint32_t)row0 * a.row_bytes + (uint32_t)(c * cg * T::GB);
      const uint32_t dst = lds0 + islot * T::STAGE;
#pragma unroll
      for (int k = 0; k < NDW; k++) {
        int q = pw + 2 * k;
        q = q < ninst ? q : ninst - 1;  // (a shorter chunk repeats its last load: the same bytes, the same place)
        uint32_t o = base + poff[k];
        o = o < a.last ? o : a.last;  // rows past N, groups past K: any valid bytes
        dma16s(w, o, __builtin_amdgcn_readfirstlane(dst + q * 1024));
      }
#pragma unroll
      for (int k = 0; k < T::SC; k++) {
        // Scales (the first loading wave) and zeros (the second): [16 rows][2 CG units].
        const int f = k * 64 + lane, lr = f / (2 * T::CG);
        int row = row0 + lr, u = c * cg * 2 + f - lr * (2 * T::CG);
        row = row < a.N ? row : a.N - 1;
        u = u < a.nun ? u : a.nun - 1;
        if (a.gunits != 1) u = (int)((uint32_t)u / (uint32_t)a.gunits);
        dma4(((pw ? a.z : a.s) + (int64_t)row * a.gpr) + u,
             __builtin_amdgcn_readfirstlane(dst + T::RAW + (pw * T::SC + k) * 256));
      }
      islot = islot + 1 == NS ? 0 : islot + 1;
      if (++ik == NT) ik = 0, ic++;
    };
#pragma unroll
    for (int i = 0; i < NS - 1; i++) issue();
    for (int i = 0; i < nitem; i++) {
      wait_vm<(NS - 2) * T::ND>();
      __syncthreads();  // item i is staged; item i - 1 is done
      issue();
    }
    wait_vm<0>();
  } else {
    // ---- products ----
    // Two register sets of x where they fit (one tile, without Q5_K's fifth bits); else the next
    // chunk's x is requested when this one's has been used.
    constexpr bool TWO = NT == 1 && F::BB != 176;
    XFrag<F> x0[UPG], x1[TWO ? UPG : 1];
    auto load_x = [&](int c, auto &x) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < UPG; q++) {
        int u = (c * cg + wave) * UPG + q;
        u = u < a.nun ? u : a.nun - 1;
        load_frag_rows<F, XM>(a.xf + (int64_t)u * R::bytes(R::rows(a.M)), lane, a.M, x[q]);
      }
    };
    int slot = 0;
    auto chunk = [&](int c, const XFrag<F> (&x)[UPG]) __attribute__((always_inline)) {
#pragma unroll
      for (int k = 0; k < NT; k++) {
        __syncthreads();
        if (wave < cg)
          group_mma<F, 2 * T::CG, T::SC * 64>(smem + slot * T::STAGE, T::RAW, r, wave, (c * cg + wave) * UPG, a.nun, pr, rot, g,
                                             x, acc[k]);
        slot = slot + 1 == NS ? 0 : slot + 1;
      }
    };
    load_x(0, x0);
    // (Unconditional loads: a load that may not have been issued costs a full wait.)
    auto clampc = [&](int c) __attribute__((always_inline)) { return c < nch ? c : nch - 1; };
    if constexpr (TWO) {
#pragma unroll 1
      for (int c = 0; c < nch; c += 2) {
        load_x(clampc(c + 1), x1);
        chunk(c, x0);
        load_x(clampc(c + 2), x0);
        if (c + 1 < nch) chunk(c + 1, x1);
      }
    } else {
#pragma unroll 1
      for (int c = 0; c < nch; c++) {
        chunk(c, x0);
        load_x(clampc(c + 1), x0);
      }
    }
  }
  float *part = reinterpret_cast<float *>(smem);
  float gs = 0.f;
  bool bad = false;
#pragma unroll
  for (int k = 0; k < NT; k++) {
    __syncthreads();  // (first: every wave is done with the stages; then: the part before was summed)
    if (wave < CW) *reinterpret_cast<f32x4 *>(part + wave * 256 + r * 16 + 4 * g) = acc[k];
    __syncthreads();
    if (t < 16 * XROWS) {
      const int c = t & 15, m = t >> 4, col = row0_of(k / NW) + c;
      float y = sum_parts<CW, XM>(part, c, m);
      if (GATED && k % NW == 0) {
        gs = y;
      } else if (m < a.M && col < a.N) {
        if constexpr (GATED) y = gate_act(gs, a.act) * y;
        bad |= !__builtin_isfinite(y);
        store_y<ODT>(a.out, (int64_t)m * a.N + col, y);
      }
    }
  }
  if (bad && a.xdt >= 0) {
#pragma unroll 1
    for (int i = 0; i < RT; i++) settle<F, GATED, ODT>(a, t >> 4, row0_of(i) + (t & 15));
  }
}

// x (M, K) -> one record per unit: a wave per (row, 256 elements).
template <class F, int XM, int XDT>
__global__ __launch_bounds__(256) void skinny_x_kernel(SkinnyArgs a, uint8_t *xf) {
  using R = XRec<F, XM>;
  constexpr int UPC = F::INT4 ? 2 : 1;
  const int lane = threadIdx.x & 63;
  const int chunks = (a.K + 255) / 256;
  const int id = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (id >= chunks * a.M) return;
  const int c = id / a.M, m = id - c * a.M;
  int64_t k = (int64_t)c * 256 + lane * 4;
  k = k < a.K ? k : a.K - 4;  // (int4, an odd unit count: the record past the end is allocated)
  float v[4];
  load_x4<XDT>(a, m, k, v);
  const int P = R::rows(a.M);
  convert_row<F, XM>(v, m, lane, xf + (int64_t)c * (UPC * R::bytes(P)), P);
}

// ---- 17 to 64 rows ---------------------------------------------------------------------------
// Eight tiles of 16 weight rows per workgroup, one per wave, over one of S parts of K (F32 partials,
// added by splitk_reduce_kernel).  All waves multiply the same unit, so x's record (up to 64 rows,
// 34 KB) is staged in LDS once per workgroup, and each unpacked weight fragment meets MT of its
// row tiles.  Per unit: wait for this wave's direct loads, one barrier, request the next unit, work.
// What bounds it, by counters of 14336 x 4096 at M = 40: no unit alone -- VALU issues on 40 % of a SIMD's
// cycles, MFMA is busy on 19 %, LDS on a third of a CU's with its bank conflicts -- but the chain through
// them with two waves a SIMD.
template <class F>
struct SkinnyMidLds {
  static constexpr int WST = (16 * F::BB + 1023) / 1024 * 1024;  // a wave's weights of one unit
  static constexpr int NW = WST / 1024;
  static constexpr int XST = (XRec<F, kX64>::bytes(64) + 1023) / 1024 * 1024;
  static constexpr int STAGE = XST + 8 * WST, BYTES = 2 * STAGE;
  static_assert(BYTES <= 160 * 1024, "LDS");
};

template <class F, int MT>
__global__ __launch_bounds__(512) void skinny_mid_kernel(SkinnyArgs a) {
  using R = XRec<F, kX64>;
  using T = SkinnyMidLds<F>;
  constexpr int PR = F::BB / 16;  // pieces of a row's unit
  extern __shared__ __align__(16) uint8_t smem[];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int g = lane >> 4, r = lane & 15;
  const int S = (int)gridDim.y;
  const int u0 = a.nun * (int)blockIdx.y / S, u1 = a.nun * ((int)blockIdx.y + 1) / S;  // u0 < u1: S <= nun
  const int P = a.M, rec = R::bytes(P);
  const int row0 = ((int)blockIdx.x * 8 + wave) * 16;
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  // The record's direct loads of this wave: 1 KB each, wave + 8 k (at most five), the last shifted
  // back to end with the record.
  const int nx = (rec + 1023) >> 10, ndx = (nx - wave + 7) >> 3;
  uint32_t woff[T::NW];
#pragma unroll
  for (int k = 0; k < T::NW; k++) {
    int p = k * 64 + lane;
    p = p < 16 * PR ? p : 16 * PR - 1;
    const int row = row0 + p / PR;
    woff[k] = (uint32_t)(row < a.N ? row : a.N - 1) * a.row_bytes + (uint32_t)(p % PR) * 16;
  }
  auto issue = [&](int u, int buf) __attribute__((always_inline)) {
    u = u < u1 ? u : u1 - 1;  // (the last request repeats)
    const uint32_t dst = lds0 + buf * T::STAGE;
    const uint8_t *xr = a.xf + (int64_t)u * rec;
    for (int k = 0; k < ndx; k++) {  // wave-uniform
      const int o = (wave + 8 * k) * 1024, oc = o + 1024 <= rec ? o : rec - 1024;
      dma16s(xr, (uint32_t)(oc + lane * 16), __builtin_amdgcn_readfirstlane(dst + oc));
    }
#pragma unroll
    for (int k = 0; k < T::NW; k++)
      dma16s(a.w0, woff[k] + (uint32_t)(u * F::BB), __builtin_amdgcn_readfirstlane(dst + T::XST + wave * T::WST + k * 1024));
  };
  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; m++) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  issue(u0, 0);
  for (int u = u0; u < u1; u++) {
    const int buf = (u - u0) & 1;
    wait_vm<0>();
    __syncthreads();  // unit u is staged; every wave is done with the other buffer
    issue(u + 1, buf ^ 1);
    const uint8_t *x = smem + buf * T::STAGE;
    typename F::Raw raw;
    F::load_lds(x + T::XST + wave * T::WST + r * F::BB, 0, PR, g, raw);
    const typename F::Sc sc = F::decode(raw, g);
    f32x4 q[MT], mn[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) q[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint8_t *xa[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) {
      const int row = m * 16 + r;
      xa[m] = x + (g * P + (row < P ? row : P - 1)) * 16;
    }
#pragma unroll
    for (int i = 0; i < F::ST; i++) {
      const f16x8 b = F::frag(raw, sc, g, i);
#pragma unroll
      for (int m = 0; m < MT; m++)
        q[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_h8(*reinterpret_cast<const u32x4 *>(xa[m] + i * (64 * P))), b, q[m], 0,
                                                       0, 0);
    }
#pragma unroll
    for (int m = 0; m < MT; m++) {
      const int row = m * 16 + r;
      const u32x2 xm = *reinterpret_cast<const u32x2 *>(x + R::mins(P) + (g * P + (row < P ? row : P - 1)) * 8);
      mn[m] = f32x4{0.f, 0.f, 0.f, 0.f};
      mn[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_h8(u32x4{xm[0], xm[1], 0, 0}), as_h8(sc.mn), mn[m], 0, 0, 0);
    }
#pragma unroll
    for (int m = 0; m < MT; m++) {
      const f32x4 xs = *reinterpret_cast<const f32x4 *>(x + R::xs(P) + (m * 16 + 4 * g) * 4);
#pragma unroll
      for (int j = 0; j < 4; j++) acc[m][j] = __fmaf_rn(xs[j], __fmaf_rn(sc.d, q[m][j], -(sc.dmin * mn[m][j])), acc[m][j]);
    }
  }
  wait_vm<0>();
  float *out = static_cast<float *>(a.out) + (int64_t)blockIdx.y * a.M * a.N;
  const int col = row0 + r;
  bool bad = false;
  if (col < a.N) {
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int row = m * 16 + 4 * g + j;
        if (row < a.M) {
          out[(int64_t)row * a.N + col] = acc[m][j];
          bad |= !__builtin_isfinite(acc[m][j]);
        }
      }
    if (bad) {
#pragma unroll 1
      for (int i = 0; i < 4 * MT; i++) {
        const int row = (i >> 2) * 16 + 4 * g + (i & 3);
        float y;
        if (row < a.M && nonfinite_sum<F>(a, a.w0, row, col, u0 * 256, u1 * 256, y)) out[(int64_t)row * a.N + col] = y;
      }
    }
  }
}

// ---- host side ------------------------------------------------------------------------------

namespace {

template <class K>
int allow_lds(K *kern, std::atomic<bool> (&done)[64], int lds) {
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (dev >= 0 && dev < 64 && done[dev].load(std::memory_order_acquire)) return HQ_OK;
  if (int rc = check(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds),
                     "hipFuncSetAttribute"))
    return rc;
  if (dev >= 0 && dev < 64) done[dev].store(true, std::memory_order_release);
  return HQ_OK;
}

template <class F, int KW, bool GATED, int XM, int XR, int XDT, int ODT>
int run_skinny(SkinnyArgs a, hipStream_t s) {
  constexpr int lds = SkinnyLds<F, XM>::BYTES;
  auto *kern = &skinny_kernel<F, KW, GATED, XM, XR, XDT, ODT>;
  static std::atomic<bool> done[64];  // per device; idempotent
  if (int rc = allow_lds(kern, done, lds)) return rc;
  a.pr = (int)(a.row_bytes / 16);
  a.tsets = (int)cdiv(a.tiles, 16 / KW);
  const int cus = device_cus();
  kern<<<(unsigned)(a.tsets < cus ? a.tsets : cus), 1024, lds, s>>>(a);
  return check_launch("skinny");
}

// One group of 256 k per wave.
template <class F, bool GATED, int XM, int XR, int XDT, int ODT>
int run_resident_k(const SkinnyArgs &a, hipStream_t s) {
  const int nkg = (int)cdiv(a.K, 256);
  if (nkg <= 1) return run_skinny<F, 1, GATED, XM, XR, XDT, ODT>(a, s);
  if (nkg <= 2) return run_skinny<F, 2, GATED, XM, XR, XDT, ODT>(a, s);
  if (nkg <= 4) return run_skinny<F, 4, GATED, XM, XR, XDT, ODT>(a, s);
  if (nkg <= 8) return run_skinny<F, 8, GATED, XM, XR, XDT, ODT>(a, s);
  return run_skinny<F, 16, GATED, XM, XR, XDT, ODT>(a, s);
}

template <class F, bool GATED, int XM, int XDT, int ODT>
int run_resident(const SkinnyArgs &a, hipStream_t s) {
  if constexpr (XM == kX16) {
    return run_resident_k<F, GATED, XM, 16, XDT, ODT>(a, s);
  } else {
    return a.M <= 4 ? run_resident_k<F, GATED, XM, 4, XDT, ODT>(a, s) : run_resident_k<F, GATED, XM, 8, XDT, ODT>(a, s);
  }
}

// Tiles per workgroup of skinny_long_kernel: 1, 2 or 4, or where that leaves CUs idle (rounds of
// workgroups, one per CU, times their tiles and one for a round's start) 3, 5 or 6.  With four, 16896 x
// 8192 (1056 tiles, M = 4) was 264 workgroups, two rounds: 35.3 us, 26.7 with five; 8704 x 8192 half the
// CUs: 19.2, 17.0 with three.  Gains of less than an eighth are none (45056 x 5632: 41.2 us with four, 43.1
// with six).  (Gated: at most two of each weight, four spill.  Q5_K's six spill eight registers and are
// still the faster ones: 21504 x 7680 41.1 us with four, 34.2.)
int long_rt(int64_t tiles, bool gated) {
  const int64_t cus = device_cus();
  auto cost = [&](int c) { return cdiv(cdiv(tiles, c), cus) * (c + 1); };
  int rt = tiles <= cus ? 1 : tiles <= 2 * cus ? 2 : 4;
  if (gated) return std::min(rt, 2);
  if (rt == 4)
    for (int c : {3, 5, 6})
      if (8 * cost(c) <= 7 * cost(4) && cost(c) < cost(rt)) rt = c;
  return rt;
}

// At most six tiles a CU, or the workgroups' rounds seven eighths full.
bool long_few_or_full(int64_t tiles) {
  const int64_t cus = device_cus(), rt = long_rt(tiles, false);
  return tiles <= 6 * cus || 8 * tiles >= 7 * cdiv(cdiv(tiles, rt), cus) * cus * rt;
}

template <class F, int RT, bool GATED, int XM, int ODT>
int run_skinny_long(const SkinnyArgs &a, hipStream_t s) {
  constexpr int lds = SkinnyLongLds<F>::BYTES;
  auto *kern = &skinny_long_kernel<F, RT, GATED, XM, ODT>;
  static std::atomic<bool> done[64];
  if (int rc = allow_lds(kern, done, lds)) return rc;
  kern<<<(unsigned)cdiv(a.tiles, RT), 1024, lds, s>>>(a);
  return check_launch("skinny_long");
}

template <class F, bool GATED, int XM, int XDT, int ODT>
int run_long(SkinnyArgs a, void *ws, hipStream_t s) {
  using T = SkinnyLongLds<F>;
  auto *xf = static_cast<uint8_t *>(ws);
  const int nkg = (int)cdiv(a.K, 256), waves = nkg * a.M;
  skinny_x_kernel<F, XM, XDT><<<(unsigned)cdiv(waves, 4), 256, 0, s>>>(a, xf);
  if (int rc = check_launch("skinny_x")) return rc;
  a.xf = xf;
  a.nch = (int)cdiv(nkg, T::CG);
  a.cg = (int)cdiv(nkg, a.nch);
  a.pr = a.cg * (T::GB / 16);
  const int rt = long_rt(a.tiles, GATED);
  if constexpr (!GATED) {
    if (rt == 3) return run_skinny_long<F, 3, GATED, XM, ODT>(a, s);
    if (rt == 4) return run_skinny_long<F, 4, GATED, XM, ODT>(a, s);
    if (rt == 5) return run_skinny_long<F, 5, GATED, XM, ODT>(a, s);
    if (rt == 6) return run_skinny_long<F, 6, GATED, XM, ODT>(a, s);
  }
  return rt == 1 ? run_skinny_long<F, 1, GATED, XM, ODT>(a, s) : run_skinny_long<F, 2, GATED, XM, ODT>(a, s);
}

constexpr int64_t kSkinnyResMaxK = 4096;  // longer rows: x prepared in the workspace

template <class F, bool GATED, int XM, int XDT, int ODT>
int run_xm(const SkinnyArgs &a, void *ws, hipStream_t s) {
  return a.K > kSkinnyResMaxK ? run_long<F, GATED, XM, XDT, ODT>(a, ws, s) : run_resident<F, GATED, XM, XDT, ODT>(a, s);
}

template <class F, bool GATED, int XDT>
int run_gguf(const SkinnyArgs &a, bool pair, void *ws, hipStream_t s) {
  if constexpr (XDT >= 0)
    if (a.M > 8) return run_xm<F, GATED, kX16, XDT, F32>(a, ws, s);
  return pair ? run_xm<F, GATED, kXPair, XDT, F32>(a, ws, s) : run_xm<F, GATED, kXDup, XDT, F32>(a, ws, s);
}

// (16-bit x is exact in one f16 under its unit's scale, down to 2^-24 of the unit's largest element.)
template <int XDT>
int run_int4(const SkinnyArgs &a, void *ws, hipStream_t s) {
  if (a.M > 8) return run_xm<SkI4, false, kX16, XDT, XDT>(a, ws, s);
  return run_xm<SkI4, false, XDT == F32 ? kXPair : kXDup, XDT, XDT>(a, ws, s);
}

}  // namespace

// Where this file's kernels are the faster ones (us per call, the int8 GEMV or the GEMMs against
// them; layers of more than 600 MB replayed from a graph, a path that the rule does not take and shapes of
// more than 100M weights: of fewer layers; Q4_K unless named):
//  * M = 2: the GEMV reads the weights once for both rows (14336 x 4096: 10.2 / 13.2).
//  * 3 <= M <= 8: from 10M weights (2560 x 4096, M = 3: 9.6 / 6.6; M = 8: 13.3 / 8.3; 2048 x 4096,
//    M = 3: 6.2 / 7.5).  Below, the GEMV's one pass of two row groups per CU beats the conversion
//    of x (2048 x 2048, M = 3: 6.1 / 9.2).  Rows past 4096 prepare x in a launch of its own and
//    need 96 tiles (1536 x 14336, M = 3: 14.9 / 14.3; 1024 x 16384: 10.1 / 16.2).
//  * Gated at M <= 4: rows of (2048, 4096] only (the MLP of 2048 x 8192 at M = 3: 21.0 / 25.1 with
//    both halves here; 4096 x 14336: 52.0 / 37.1).
//    At M <= 4, one pass of the GEMV, past six tiles a CU only where the rounds of workgroups are nearly full
//    (28672 x 8192 39.6 / 36.7; 25600 x 16384 54.0 / 58.1; 50426 x 4864 42.7 / 50.4), or Q4_K past 16384,
//    where its GEMV slows (24576 x 18944: 146.5 / 70.2).
//  * M > 8: always, against the GEMM's conversion, product and split-K launches (14336 x 4096,
//    M = 12: 29.3 / 19.4; 1024 x 4096, M = 9: 14.9 / 12.7), few columns of long rows too, where this does
//    not split K and the GEMM does: 32 to 1536 rows of 2048 to 28672, Q4_K and Q5_K, M = 9 and 16, all
//    faster but Q5_K, 32 x 28672 at M = 16 (20.1 / 21.4; 128 x 28672 28.7 / 22.1).
bool skinny_ok(int64_t M, int64_t N, int64_t K, int dt, const void *w, const void *x) {
  if ((dt != Q4_K && dt != Q5_K) || M < 3 || M > kSkinnyMaxRows || K <= 0 || K % 256 || K > kSkinnyMaxK || N < 1 ||
      (N + 64) * (K / 256) * block_info(dt).bytes > UINT32_MAX || ((uintptr_t)w & 15) || ((uintptr_t)x & 15))
    return false;
  if (M > 8) return true;
  if (N * K < 10000000) return false;
  if (K <= kSkinnyResMaxK) return true;
  return N >= 1536 && (M > 4 || (dt == Q4_K && K > 16384) || long_few_or_full(cdiv(N, 16)));
}

bool skinny_gated_ok(int64_t M, int64_t N, int64_t K, int dt, const void *wg, const void *wu, const void *x) {
  return skinny_ok(M, N, K, dt, wg, x) && ((uintptr_t)wu & 15) == 0 && (M > 4 || (K > 2048 && K <= kSkinnyResMaxK));
}

// int4: 3 <= M <= 8 from 8.3M weights with 16-bit x (2048 x 4096, M = 4: 9.0 / 7.8; 2048 x 2048: 7.4 /
// 7.3), 12M with F32 x, whose two f16 parts cost twice the conversion (2048 x 4096, M = 4: 9.0 /
// 9.9; 3072 x 4096: 14.8 / 10.2), 16M for rows past 4096 (2048 x 8192, M = 4: 18.1 / 14.5; 1024 x
// 8192: 10.4 / 14.3).  At M <= 4, one pass of the GEMV, it stays the faster one for some rows of 8192 to 17408,
// where it slows (BF16 x): below 160 tiles from 10240 on (2048 x 14336: 13.9 / 14.9; 2048 x 17152 15.6 / 17.4;
// x 17408 30.0 / 17.4), from 14336 to 16384 up to three tiles a CU (4608 x 16384: 19.4 / 22.2; 12288 x
// 15360 32.0 / 29.3), up to 16384 from six on, where a workgroup's tiles take rounds (25600 x 10240: 40.1 / 46.3;
// 24576 x 10240 35.6 / 34.6).
// M > 8 replaces one or two launches more of work that grows with N.  F32 x from 30M (8192 x 4096: 19.5 /
// 18.4), 16M past 4096 (2048 x 8192: 16.0 / 15.0).  BF16 x from 45M (11008 x 4096, M = 12: 24.2 / 20.7; 14336 x
// 3072, M = 9: 17.8 / 18.9; 8192 x 4096: 16.5 / 18.3); past 4096 30M (4096 x 8192: 17.8 / 16.2), from 18944 on
// with 192 tiles (3072 x 18944 25.3 / 18.7; 2048 x 18944, G = 256, 19.1 / 20.0).  F16 x past 4096 only, 16M
// (2048 x 8192: 16.7 / 14.9; 18944 x 3584: 18.5 / 24.0), from 16640 on with 128 tiles (1024 x 18944, G = 256,
// 17.8 / 19.8), from 22528 on with 192 (2048 x 22528, G = 256, 20.2 / 22.4; 3072 x 28672, 24.5 / 24.1).
bool skinny_int4_ok(int64_t M, int64_t N, int64_t K, int G, int x_dtype, const void *codes, const void *x) {
  if (M < 3 || M > kSkinnyMaxRows || K <= 0 || K % 128 || K > kSkinnyMaxK || G <= 0 || G % 128 || K % G || N < 1 ||
      (N + 64) * (K / 2) > UINT32_MAX || ((uintptr_t)codes & 15) || ((uintptr_t)x & 15))
    return false;
  const bool lng = K > kSkinnyResMaxK;
  const int64_t W = N * K, mega = 1000000, tiles = cdiv(N, 16);
  if (M <= 8) {
    const int64_t cus = device_cus();
    const bool gemv = M <= 4 && ((K >= 10240 && K < 17408 && tiles < 160) || (K > 14336 && K <= 16384 && tiles <= 3 * cus) ||
                                 (K > 8192 && K <= 16384 && tiles > 6 * cus));
    return W >= (lng ? 16 * mega : x_dtype == F32 ? 12 * mega : 8300000) && !gemv;
  }
  if (x_dtype == F32) return W >= (lng ? 16 : 30) * mega;
  if (x_dtype == BF16) return lng ? W >= 30 * mega && (K < 18944 || tiles >= 192) : W >= 45 * mega;
  return lng && W >= 16 * mega && tiles >= (K < 16640 ? 0 : K < 22528 ? 128 : 192);
}

// Two f16 parts of x where the int8 GEMVs keep two levels: rows below 4096 (kX1MinK), and the long
// rows that gemv_q4kx_kernel's LDS does not take.
static bool skinny_pair(int64_t K) { return K < 4096 || K > 16384; }

size_t skinny_ws_bytes(int64_t M, int64_t K, bool int4) {
  if (M < 3 || M > kSkinnyMaxRows || K <= kSkinnyResMaxK || K > kSkinnyMaxK) return 0;
  const int P = M <= 8 && (int4 || skinny_pair(K)) ? 2 * (int)M : (int)M;  // (int4: as for F32 x)
  const int64_t rec = int4 ? 2 * XRec<SkI4, kX16>::bytes(P) : XRec<SkQk<false>, kX16>::bytes(P);
  return (size_t)((cdiv(K, 256) * rec + 255) & ~(int64_t)255);
}

static SkinnyArgs skinny_args(const void *x, const void *w, float *out, int64_t M, int64_t N, int64_t K, int dt) {
  SkinnyArgs a = {};
  a.x = x;
  a.w0 = static_cast<const uint8_t *>(w);
  a.out = out;
  a.M = (int)M;
  a.N = (int)N;
  a.K = (int)K;
  a.nun = (int)(K / 256);
  a.tiles = (int)cdiv(N, 16);
  a.row_bytes = (uint32_t)(K / 256 * block_info(dt).bytes);
  a.last = (uint32_t)(N * a.row_bytes - 16);
  a.in_q2 = act_q2_off(M, K);
  a.in_d = act_d_off(M, K);
  return a;
}

int launch_skinny(const float *x, const void *w0, const void *w1, float *out, int64_t M, int64_t N, int64_t K, int act,
                  int dt, void *ws, hipStream_t s) {
  SkinnyArgs a = skinny_args(x, w0, out, M, N, K, dt);
  a.w1 = static_cast<const uint8_t *>(w1);
  a.act = act;
  a.xdt = F32;
  const bool pair = skinny_pair(K);
  if (dt == Q5_K)
    return w1 ? run_gguf<SkQk<true>, true, F32>(a, pair, ws, s) : run_gguf<SkQk<true>, false, F32>(a, pair, ws, s);
  return w1 ? run_gguf<SkQk<false>, true, F32>(a, pair, ws, s) : run_gguf<SkQk<false>, false, F32>(a, pair, ws, s);
}

int launch_skinny_act(const void *x, const void *w, float *out, int64_t M, int64_t N, int64_t K, int dt, void *ws,
                      hipStream_t s) {
  SkinnyArgs a = skinny_args(x, w, out, M, N, K, dt);
  a.xdt = kXAct;
  const bool pair = skinny_pair(K);
  return dt == Q5_K ? run_gguf<SkQk<true>, false, kXAct>(a, pair, ws, s) : run_gguf<SkQk<false>, false, kXAct>(a, pair, ws, s);
}

// ---- 17 <= M <= 64, Q4_K / Q5_K (skinny_mid_kernel) ----
// K parts: the fewest rounds of workgroups (one per CU) times units per part, a part's start and its
// share of the reduce counted as three units.
static int mid_splits(int64_t N, int64_t K) {
  const int64_t groups = cdiv(N, 128), nun = K / 256, cus = device_cus();
  int64_t best = INT64_MAX, s = 1;
  for (int64_t c = 1; c <= 16 && (c == 1 || c * 2 <= nun); c++) {
    const int64_t cost = cdiv(groups * c, cus) * (cdiv(nun, c) + (c > 1 ? 3 : 2));
    if (cost < best) best = cost, s = c;
  }
  return (int)s;
}

// Every such call (us, the bf16 GEMM with its conversion and reduce / this; layers of more than 600 MB
// replayed from a graph, Q4_K): 14336 x 4096 M = 17 29.6 / 18.9, M = 24 30.0 / 19.5, M = 40 31.1 / 22.1, M = 64
// 32.6 / 26.0; 4096 x 14336 M = 64 39.8 / 26.5; 512 x 1024 M = 20 13.5 / 8.6; 28672 x 8192 M = 40 96.5 / 62.4.
// Q5_K, which the GEMM first expands to bf16 in memory: 14336 x 4096 M = 40 78.9 / 24.1.  32 to 1536 rows of
// 2048 to 28672 at M = 17, 33 and 64: all faster but Q5_K, 32 x 28672 at M = 64 (23.0 / 23.3).
bool skinny_mid_ok(int64_t M, int64_t N, int64_t K, int dt, const void *w, const void *x) {
  return (dt == Q4_K || dt == Q5_K) && M > kSkinnyMaxRows && M <= 64 && K > 0 && K % 256 == 0 && K <= kSkinnyMaxK && N >= 1 &&
         N * (K / 256) * block_info(dt).bytes <= UINT32_MAX && ((uintptr_t)w & 15) == 0 && ((uintptr_t)x & 15) == 0;
}

static size_t mid_rec_bytes(int64_t M, int64_t K) {
  return (size_t)((K / 256 * XRec<SkQk<false>, kX64>::bytes((int)M) + 255) & ~(int64_t)255);
}

size_t skinny_mid_ws_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= kSkinnyMaxRows || M > 64 || N < 1 || K % 256 || K > kSkinnyMaxK) return 0;
  const int s = mid_splits(N, K);
  return mid_rec_bytes(M, K) + (s > 1 ? (size_t)s * M * N * 4 : 0);
}

int launch_splitk_reduce(const float *part, void *out, int out_dtype, int64_t n, int splits, hipStream_t s);

template <class F, int MT>
static int run_mid(SkinnyArgs a, float *out, void *ws, hipStream_t s) {
  constexpr int lds = SkinnyMidLds<F>::BYTES;
  auto *kern = &skinny_mid_kernel<F, MT>;
  static std::atomic<bool> done[64];
  if (int rc = allow_lds(kern, done, lds)) return rc;
  auto *xf = static_cast<uint8_t *>(ws);
  auto *part = reinterpret_cast<float *>(xf + mid_rec_bytes(a.M, a.K));
  skinny_x_kernel<F, kX64, F32><<<(unsigned)cdiv((int64_t)a.nun * a.M, 4), 256, 0, s>>>(a, xf);
  if (int rc = check_launch("skinny_x")) return rc;
  const int S = mid_splits(a.N, a.K);
  a.xf = xf;
  a.out = S > 1 ? part : out;
  kern<<<dim3((unsigned)cdiv(a.N, 128), (unsigned)S), 512, lds, s>>>(a);
  if (int rc = check_launch("skinny_mid")) return rc;
  return S > 1 ? launch_splitk_reduce(part, out, F32, (int64_t)a.M * a.N, S, s) : HQ_OK;
}

template <class F>
static int run_mid_m(const SkinnyArgs &a, float *out, void *ws, hipStream_t s) {
  if (a.M <= 32) return run_mid<F, 2>(a, out, ws, s);
  if (a.M <= 48) return run_mid<F, 3>(a, out, ws, s);
  return run_mid<F, 4>(a, out, ws, s);
}

int launch_skinny_mid(const float *x, const void *w, float *out, int64_t M, int64_t N, int64_t K, int dt, void *ws,
                      hipStream_t s) {
  SkinnyArgs a = skinny_args(x, w, out, M, N, K, dt);
  a.xdt = F32;
  return dt == Q5_K ? run_mid_m<SkQk<true>>(a, out, ws, s) : run_mid_m<SkQk<false>>(a, out, ws, s);
}

int launch_skinny_int4(const void *x, int x_dtype, const uint32_t *codes, const float *sc, const float *zr, void *y,
                       int64_t M, int64_t N, int64_t K, int G, void *ws, hipStream_t s) {
  SkinnyArgs a = {};
  a.x = x;
  a.xdt = x_dtype;
  a.w0 = reinterpret_cast<const uint8_t *>(codes);
  a.s = sc;
  a.z = zr;
  a.out = y;
  a.M = (int)M;
  a.N = (int)N;
  a.K = (int)K;
  a.gpr = (int)(K / G);
  a.gunits = G / 128;
  a.nun = (int)(K / 128);
  a.tiles = (int)cdiv(N, 16);
  a.row_bytes = (uint32_t)(K / 2);
  a.last = (uint32_t)(N * a.row_bytes - 16);
  switch (x_dtype) {
    case F32: return run_int4<F32>(a, ws, s);
    case BF16: return run_int4<BF16>(a, ws, s);
    case F16: return run_int4<F16>(a, ws, s);
    default: return fail(HQ_EUNSUPPORTED, "int4_matmul", "x dtype %d", x_dtype);
  }
}

}  // namespace hq
