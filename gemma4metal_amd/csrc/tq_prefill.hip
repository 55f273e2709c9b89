// Multi-query (prefill) attention over the int4 cache with K/V tiles shared
// by a workgroup's (query, head) rows -- the engine's prefill fallback
// (engine/gemma4_multilayer.cpp:343-364: dequantize, then masked
// scaled_dot_product_attention), for head_dim 128 / 256 / 512 and 16-bit
// queries (fp32 ones: tq_prefill_f32.hip).
//
// A workgroup takes RS sets of 16 consecutive (query, head) rows of one kv
// head and streams the union of their key ranges in tiles of 32 KH keys; wave
// (rs, kh) runs set rs against keys 32 kh .. 32 kh + 31 of every tile.  Tiles
// are staged in LDS, double-buffered with one barrier a tile, as centred
// nibbles n - 8 in fp16 (one AND-OR into 1024 + n and one packed add per two
// values; exact), in the order of the matrix-core operands, so an A operand is
// one 16-byte read.  They are never dequantized: the group scales go where
// they are cheap, and with b' = b + 8 s
//
//   S^T[key][row] = sum_g s_k[key][g] ((n - 8) . q)_g + b'_k[key][g] (sum q)_g
//     (. . q)_g: v_mfma_f32_16x16x32_f16 over the group's 64 dims, A = nibbles
//     of 16 keys, B = q of 16 rows, scaled by a power of two per row (exact);
//     one fma per (key, row, group) applies s_k.  The bias term is one more
//     product a 16-key half: A = biases and scales, B = the group sums of q in
//     three fp16 parts.
//   O^T[dim][row] = sum_key (n - 8) (p s_v) + sum_key p b'_v
//     A = nibbles of 16 dims (one group) x 32 keys, B = p s_v as fp16 high part
//     and remainder: 22 bits, down to the fp16 step of 2^-24.  p's reference
//     holds p s_v to fp16's range (see m_ref below) in tiles whose V scales are
//     alike; any other tile takes a power of two per row and group of its own,
//     so that a row's precision does not depend on the V scales of other keys
//     and groups.  The bias term is summed in fp32.
// Centred nibbles keep the sums small: the matrix cores' accumulation error
// grows with the running sum, and with n in place of n - 8 the results were
// three times as far from 64 bits.
//
// Lane l = 16 c + m.  S^T leaves it keys 16 h + 4 c + i (h = 0, 1; i = 0 .. 3) of
// row m, and the same keys are slots 4 h + i of lane group c in the P.V
// products: no exchange between the two.  Row r of a P.V product x of group g
// is dim 64 g + 8 (r % 8) + 2 x + r / 8, the odd ones scaled by 16 (bits 4-7 of
// a byte are masked in place).
#include "tq_sdpa_common.h"

#include <type_traits>

namespace tq {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// A running reference moves only when a score passes it by this much (log2).
constexpr float kPfLazy = 8.0f;
// With 2^e0 above every V scale of a workgroup's first tile: p s_v is below
// 2^kPfHead for the row's largest weight and a scale of 2^e0, and below 2^15 (fp16
// overflows at 2^16) for scales up to 2^(e0 + kPfUp).  Scales down to
// 2^(e0 - kPfDown) leave such a weight 19 bits above fp16's step (3 more than bf16
// parts would).  A tile outside these bounds costs half as much again: with every
// tile so (one group of 64 dims at 2^-12), 512 queries after 3,584 keys, 85
// instead of 63 us (Hq 32 Hkv 16 D 256, window 1,024) and 578 instead of 387
// (Hq 32 Hkv 4 D 512).
constexpr int kPfHead = 4, kPfUp = 3, kPfDown = 9;

template <int D, bool F32, int RS>
struct PfGeom {
  using SB = typename std::conditional<F32, float, _Float16>::type;
  static constexpr int W = D / 8;        // packed words per row
  static constexpr int NG = D / 64;      // quant groups per row
  static constexpr int DH = D == 512 ? 2 : 1;  // waves that share a row set's dims
  static constexpr int KH = 2 / DH;            // 32-key parts of a tile
  static constexpr int NW_ = NG / DH;          // groups of a wave
  static constexpr int OW = D / DH;            // dims of a wave
  static constexpr int TK = 32 * KH, NW = RS * KH * DH, NT = 64 * NW;
  // 16-byte units of a 16-key slice of K (8 NG operands) and of V^T per 32 keys
  // (4 NG operands).  An operand is 64 units [c][m]; unit m sits at m ^ swizzle(g),
  // so that the 16 lanes of a store (of several groups) reach distinct banks, as
  // those of a read do.
  static constexpr int KU = 64 * 2 * NG, VU = 64 * 4 * NG;
  static __device__ __forceinline__ constexpr int kswz(int g) { return (16 / NG) * g; }
  static __device__ __forceinline__ constexpr int vswz(int g) { return 8 * (g & 1); }
  static constexpr int UNITS = TK * W / 8;                      // 8-word staging units of K; as many of V
  static constexpr int NU = (2 * UNITS + NT - 1) / NT;
  static constexpr int SDW = TK * NG * static_cast<int>(sizeof(SB)) / 4;  // dwords of one scale tensor a tile
  static constexpr int NSD = (4 * SDW + NT - 1) / NT;
  static constexpr int NSW = SDW / 64;   // waves that stage one of them
  static constexpr int OSTR = OW + 2;    // partial output rows (floats): conflict-free 4-byte stores
  struct Stage {
    u32x4 k[2][2 * KH * KU];             // [16-key slice][g][s][c][key]: word 8 g + 2 c + s
    u32x4 v[2][KH * VU];                 // [kh][g][x][c][dim row]: slots 0-7 of lane group c
    SB sb[2][4][TK * NG];                // k scale, k bias, v scale, v bias
    v4f xch[DH == 2 ? NW : 1][2][64];    // score parts of a row set's waves
  };
  union Lds {
    Stage st;
    float o[NW][16 * OSTR];
  };
  static_assert(SDW % 64 == 0 && UNITS % 64 == 0, "wave-uniform staging roles");
};

// One tile's words and scales, in this thread's registers: a unit is 8 words
// of a key (K), or one word of the 8 keys of a lane group's slots (V).
template <class Gm>
struct PfRaw {
  uint32_t w[Gm::NU][8];
  uint32_t s[Gm::NSD];
};

template <class Gm>
__device__ __forceinline__ void pf_load(PfRaw<Gm>& R, const SdpaParams& p, int64_t row0, int t0, int last) {
  typedef uint32_t u32_a2 __attribute__((aligned(2)));  // scale tensors may start at any element
  // rows past the last key repeat it (the mask drops them); the tile's first
  // row is uniform, so every address is a scalar base and a 32-bit offset
  auto row = [&](int r) { return static_cast<uint32_t>(min(r, last - t0)); };
  const int64_t base = row0 + t0;
#pragma unroll
  for (int i = 0; i < Gm::NU; ++i) {
    const int e = threadIdx.x + i * Gm::NT;
    const int role = __builtin_amdgcn_readfirstlane(e / Gm::UNITS);
    const int u = e % Gm::UNITS;
    if (role == 0) {
      const u32x4* src = reinterpret_cast<const u32x4*>(p.kq + base * Gm::W) + (row(u / Gm::NG) * (Gm::W / 4) + 2 * (u % Gm::NG));
      const u32x4 a = src[0], b = src[1];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        R.w[i][k] = a[k];
        R.w[i][4 + k] = b[k];
      }
    } else {  // (D 128: threads past the units load one again and do not store it)
      const int w = u % Gm::W, kc = u / Gm::W;  // kc = 4 kh + c
      const int r0 = 32 * (kc >> 2) + 4 * (kc & 3);
      const uint32_t* src = p.vq + base * Gm::W;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int r = 16 * (j >> 2) + (j & 3);
        R.w[i][j] = src[row(r0 + r) * Gm::W + w];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < Gm::NSD; ++i) {
    const int e = threadIdx.x + i * Gm::NT;
    // (threads past the tensors load one again and do not store it)
    const int t = min(__builtin_amdgcn_readfirstlane(e / Gm::SDW), 3), d = e % Gm::SDW;
    constexpr int DPR = Gm::SDW / Gm::TK;  // dwords a row
    const void* src = t == 0 ? p.ks : t == 1 ? p.kb : t == 2 ? p.vs : p.vb;
    R.s[i] = (reinterpret_cast<const u32_a2*>(src) + base * DPR)[row(d / DPR) * DPR + d % DPR];
  }
}

// Nibbles in bits 0-3 (HI: 4-7) of both halves of t as fp16 n - 8 (16 (n - 8)).
// mask: 0x000F000F (0x00F000F0) in a vector register -- as a literal beside the
// other one, the AND and the OR are two instructions.
template <bool HI>
__device__ __forceinline__ uint32_t pf_centre(uint32_t t, uint32_t mask) {
  uint32_t b;  // 1024 + n, 1024 + 16 n
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(b) : "v"(t), "v"(mask), "s"(0x64006400u));
  const _Float16 off = static_cast<_Float16>(HI ? -1152.0f : -1032.0f);
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, b) + v2h{off, off});
}

// Whether this thread's V scales are all within [2^(e0 - kPfDown), 2^(e0 + kPfUp)),
// per wave that stages some, into ok[NSW].
template <class Gm>
__device__ __forceinline__ void pf_alike(const PfRaw<Gm>& R, int e0, int* ok) {
  constexpr bool kHalf = sizeof(typename Gm::SB) == 2;
  // the bounds' bit patterns: magnitudes order as these do
  const auto bits = [](float x) -> uint32_t {
    if constexpr (kHalf) return __builtin_bit_cast(uint16_t, static_cast<_Float16>(x));
    else return __float_as_uint(x);
  };
  const uint32_t lo = bits(ldexpf(1.0f, e0 - kPfDown)), n = bits(ldexpf(1.0f, e0 + kPfUp)) - lo;
#pragma unroll
  for (int i = 0; i < Gm::NSD; ++i) {
    const int e = threadIdx.x + i * Gm::NT;
    if (__builtin_amdgcn_readfirstlane(e / Gm::SDW) != 2) continue;
    const uint32_t a = R.s[i];
    bool in;
    if constexpr (kHalf) in = (a & 0x7FFFu) - lo < n && (a >> 16 & 0x7FFFu) - lo < n;
    else in = (a & 0x7FFFFFFFu) - lo < n;
    ok[e % Gm::SDW / 64] = __all(in);  // (one value from every lane)
  }
}

// Into LDS buffer b.
template <class Gm>
__device__ __forceinline__ void pf_store(typename Gm::Stage& S, const PfRaw<Gm>& R, int b) {
  const uint32_t mlo = 0x000F000Fu, mhi = 0x00F000F0u;
#pragma unroll
  for (int i = 0; i < Gm::NU; ++i) {
    const int e = threadIdx.x + i * Gm::NT;
    const int role = __builtin_amdgcn_readfirstlane(e / Gm::UNITS);
    const int u = e % Gm::UNITS;
    if (role == 0) {
      // word 8 g + 2 c + s: nibbles 0, 4, 1, 5, 2, 6, 3, 7
      const int r = u / Gm::NG, g = u % Gm::NG;
      u32x4* d = &S.k[b][(r >> 4) * Gm::KU + 128 * g + ((r & 15) ^ Gm::kswz(g))];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t w = R.w[i][k], h = w >> 8;
        d[64 * (k & 1) + 16 * (k >> 1)] =
            u32x4{pf_centre<false>(w, mlo), pf_centre<true>(w, mhi), pf_centre<false>(h, mlo), pf_centre<true>(h, mhi)};
      }
    } else if (role == 1) {
      const int w = u % Gm::W, kc = u / Gm::W;
      const int g = w >> 3;
      u32x4* d = &S.v[b][(kc >> 2) * Gm::VU + 256 * g + (kc & 3) * 16 + (w & 7)];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        u32x4 lo, hi;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          // byte x of two keys' words into the low bytes of the halves
          const uint32_t t = __builtin_amdgcn_perm(R.w[i][2 * q + 1], R.w[i][2 * q], 0x0C040C00u + 0x00010001u * x);
          lo[q] = pf_centre<false>(t, mlo);
          hi[q] = pf_centre<true>(t, mhi);
        }
        d[64 * x + Gm::vswz(g)] = lo;
        d[64 * x + (8 ^ Gm::vswz(g))] = hi;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < Gm::NSD; ++i) {
    const int e = threadIdx.x + i * Gm::NT;
    const int t = __builtin_amdgcn_readfirstlane(e / Gm::SDW);
    if ((4 * Gm::SDW) % Gm::NT != 0 && t >= 4) continue;
    reinterpret_cast<uint32_t*>(S.sb[b][0])[e] = R.s[i];
  }
}

// The largest |V scale| of the wave's part of a tile, 0 where it has none.
template <class Gm>
__device__ __forceinline__ float pf_vmax(const PfRaw<Gm>& R) {
  float mx = 0.0f;
#pragma unroll
  for (int i = 0; i < Gm::NSD; ++i) {
    const int e = threadIdx.x + i * Gm::NT;
    if (__builtin_amdgcn_readfirstlane(e / Gm::SDW) != 2) continue;
    if constexpr (sizeof(typename Gm::SB) == 2) {
      const v2h h = __builtin_bit_cast(v2h, R.s[i]);
      mx = fmaxf(mx, fmaxf(fabsf(static_cast<float>(h[0])), fabsf(static_cast<float>(h[1]))));
    } else {
      mx = fmaxf(mx, fabsf(__uint_as_float(R.s[i])));
    }
  }
  return wave_max_dpp(mx);
}

// The fp16 remainders x0 - h0, x1 - h1 of a pair whose fp16 high parts are
// packed in hp, as a packed fp16 pair: one mixed-precision fma each.  The
// difference is exact in fp32 and rounded once, to fp16.
__device__ __forceinline__ uint32_t pf_rem_pair(uint32_t hp, float x0, float x1) {
  uint32_t r;
  asm("v_fma_mixlo_f16 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %0, %1, -1.0, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
      : "=&v"(r)
      : "v"(hp), "v"(x0), "v"(x1));
  return r;
}

template <int D, bool F32, int RS>
__device__ __forceinline__ void prefill_rows(const SdpaParams& p) {
  using Gm = PfGeom<D, F32, RS>;
  using SB = typename Gm::SB;
  constexpr int NG = Gm::NG, NWG = Gm::NW_, TK = Gm::TK, KH = Gm::KH, DH = Gm::DH;
  __shared__ __attribute__((aligned(16))) typename Gm::Lds L;
  __shared__ uint32_t vmx;                  // bits of the first tile's largest |V scale|
  __shared__ int alike[2][Gm::NSW];         // a buffer's V scales are alike (all of them set)
  __shared__ float ml[Gm::NW][16], ll[Gm::NW][16];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int rs = wave % RS, kh = wave / RS % KH, dh = wave / (RS * KH);
  const int m = lane & 15, c = lane >> 4;
  // heads vary fastest: with Hkv a multiple or a divisor of 8, an XCD's
  // workgroups (every eighth) stay on a few heads, whose caches its L2 holds;
  // the longest key ranges (last queries) start first
  const int nblk = gridDim.x / p.Hkv;
  const int kvh = blockIdx.x % p.Hkv, blk = nblk - 1 - static_cast<int>(blockIdx.x / p.Hkv);
  const int total = p.nq * p.gqa;           // rows of this kv head
  const int r0 = blk * 16 * RS;             // first row of this workgroup
  const int W_ = p.window;
  const int lo = W_ > 0 ? max(0, p.n + r0 / p.gqa + 1 - W_) : 0;
  const int last = p.n + (min(r0 + 16 * RS, total) - 1) / p.gqa;  // last key of the last row
  const int ntile = (last - lo) / TK + 1;
  const int64_t row0 = static_cast<int64_t>(kvh) * p.cap;

  PfRaw<Gm> raw;
  pf_load<Gm>(raw, p, row0, lo, last);

  const int rw = r0 + 16 * rs;              // the wave's first row
  const int pos_lo = p.n + min(rw, total - 1) / p.gqa, pos_hi = p.n + min(rw + 15, total - 1) / p.gqa;
  const int R = min(rw + m, total - 1);     // this lane's row (column m)
  const int qi = R / p.gqa;
  const int pos = p.n + qi;                 // its absolute position

  // ---- q: B operands of k-step s of group g are dims 64 g + 16 c + 8 s + {0, 4,
  // 1, 5, 2, 6, 3, 7}, times 2^(15 - ex) (the row's largest below 2^15), the odd
  // ones over 16.  The sign of a negative scale goes into q.
  v8h qf[2 * NWG], qb;
  const int64_t qrow = static_cast<int64_t>(qi) * p.Hq + kvh * p.gqa + (R - qi * p.gqa);
  float f[2 * NWG][8];
  float mx = 0.0f;
#pragma unroll
  for (int j = 0; j < 2 * NWG; ++j) {
    const int64_t e0 = qrow * D + Gm::OW * dh + 64 * (j >> 1) + 16 * c + 8 * (j & 1);
    const uint4 u = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p.q) + e0);
    const uint32_t wd[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (p.q_dtype == TQ_F16) {
        const v2h h = __builtin_bit_cast(v2h, wd[i]);
        f[j][2 * i] = static_cast<float>(h[0]);
        f[j][2 * i + 1] = static_cast<float>(h[1]);
      } else {
        f[j][2 * i] = __uint_as_float(wd[i] << 16);
        f[j][2 * i + 1] = __uint_as_float(wd[i] & 0xFFFF0000u);
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) mx = fmaxf(mx, fabsf(f[j][i]));
  }
  mx = xor32_max(xor16_max(mx));
  const int ex = __builtin_amdgcn_frexp_expf(mx);
  const float rf = ldexpf(fabsf(p.scale_log2), ex - 15);  // score = rf * products
  const bool neg = p.scale_log2 < 0.0f;
  float qs[NWG];
#pragma unroll
  for (int g = 0; g < NWG; ++g) qs[g] = 0.0f;
#pragma unroll
  for (int j = 0; j < 2 * NWG; ++j) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float x = ldexpf(f[j][i], 15 - ex);
      x = neg ? -x : x;
      qs[j >> 1] += x;
      const int slot = (i & 2) ? 4 + 2 * (i & 1) + (i >> 2) : 2 * (i & 1) + (i >> 2);
      const float y = (i & 1) ? x * 0.0625f : x;
      qf[j][slot] = static_cast<_Float16>(y);
    }
  }
  // group sums over 512 (|.| < 2^12) in fp16 parts.  fp16 scale/bias: part c
  // in lane group c (parts 0-2) for the biases, 8 times it for the scales;
  // fp32: b' = high + low half, high half times parts 0, 1 in lane groups
  // 0, 1 and low half in 2, 3.
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    _Float16 pt = static_cast<_Float16>(0.0f);
    if (g < NWG) {
      float x = xor32_sum(xor16_sum(qs[g < NWG ? g : 0])) * 0x1p-9f;
      const _Float16 h0 = static_cast<_Float16>(x);
      x -= static_cast<float>(h0);
      const _Float16 h1 = static_cast<_Float16>(x);
      x -= static_cast<float>(h1);
      const _Float16 h2 = static_cast<_Float16>(x);
      if constexpr (F32) pt = (c & 1) ? h1 : h0;
      else pt = c == 0 ? h0 : c == 1 ? h1 : c == 2 ? h2 : pt;
    }
    qb[g] = pt;
    qb[4 + g] = F32 ? static_cast<_Float16>(0.0f) : pt * static_cast<_Float16>(8.0f);
  }

  if (threadIdx.x == 0) vmx = 0;
  __syncthreads();
  const float wm = pf_vmax<Gm>(raw);
  if (lane == 0) atomicMax(&vmx, __float_as_uint(wm));
  pf_store<Gm>(L.st, raw, 0);
  __syncthreads();
  // (a first tile outside these bounds, like an infinity, is not alike)
  const int e0 = min(max(__builtin_amdgcn_frexp_expf(__uint_as_float(__builtin_amdgcn_readfirstlane(vmx))), -20), 24);
  pf_alike<Gm>(raw, e0, alike[0]);
  __syncthreads();

  // p = 2^(x - m_ref), m_ref = a score of the row + e0 - kPfHead, the largest so
  // far up to kPfLazy.  A reference that follows the largest V scale staged so far
  // leaves a row 28 - k bits once a key that it does not attend has 2^k times
  // the scales of those that it does.
  float m_ref = -INFINITY, l_run = 0.0f, bsum[NWG];
  v4f o[4 * NWG];
#pragma unroll
  for (int b = 0; b < 4 * NWG; ++b) o[b] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int g = 0; g < NWG; ++g) bsum[g] = 0.0f;
  const v4f z = v4f{0.0f, 0.0f, 0.0f, 0.0f};

#pragma unroll 1
  for (int it = 0; it < ntile; ++it) {
    const int buf = it & 1;
    if (it + 1 < ntile) pf_load<Gm>(raw, p, row0, lo + (it + 1) * TK, last);
    const int t0 = lo + it * TK + 32 * kh;  // this wave's keys t0 .. t0 + 31
    const bool any = t0 <= pos_hi && (W_ == 0 || pos_lo - (t0 + 31) < W_);  // wave-uniform
    // this wave's groups
    const u32x4* ku = L.st.k[buf] + 2 * kh * Gm::KU + 128 * NWG * dh + 16 * c;
    const u32x4* vu = L.st.v[buf] + kh * Gm::VU + 256 * NWG * dh + 16 * c;
    const SB* sks = L.st.sb[buf][0] + 32 * kh * NG + NWG * dh;
    const SB* skb = L.st.sb[buf][1] + 32 * kh * NG + NWG * dh;
    const SB* svs = L.st.sb[buf][2] + 32 * kh * NG + NWG * dh;
    const SB* svb = L.st.sb[buf][3] + 32 * kh * NG + NWG * dh;

    float sc[8];
    if (any) {
      // ---- S^T: two 16-key halves ------------------------------------------
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        v8h kb;
        {
          const SB* br = skb + (16 * h + m) * NG;
          const SB* sr = sks + (16 * h + m) * NG;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const _Float16 zero = static_cast<_Float16>(0.0f);
            if constexpr (F32) {
              const float bv = g < NWG ? fmaf(8.0f, sr[g < NWG ? g : 0], br[g < NWG ? g : 0]) : 0.0f;
              const _Float16 bh = static_cast<_Float16>(bv);
              kb[g] = c < 2 ? bh : static_cast<_Float16>(bv - static_cast<float>(bh));
              kb[4 + g] = zero;
            } else {
              kb[g] = g < NWG ? br[g < NWG ? g : 0] : zero;
              kb[4 + g] = g < NWG ? sr[g < NWG ? g : 0] : zero;
            }
          }
        }
        const v4f bt = __builtin_amdgcn_mfma_f32_16x16x32_f16(kb, qb, z, 0, 0, 0);
        v4f acc[NWG];
#pragma unroll
        for (int g = 0; g < NWG; ++g) {
          const u32x4* kr = ku + h * Gm::KU + 128 * g + (m ^ Gm::kswz(NWG * dh + g));
          const v8h a0 = __builtin_bit_cast(v8h, kr[0]), a1 = __builtin_bit_cast(v8h, kr[64]);
          v4f a = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, qf[2 * g], z, 0, 0, 0);
          a = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, qf[2 * g + 1], a, 0, 0, 0);
          acc[g] = a;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float s = bt[i] * 512.0f;
#pragma unroll
          for (int g = 0; g < NWG; ++g)
            s = fmaf(static_cast<float>(sks[(16 * h + 4 * c + i) * NG + g]), acc[g][i], s);
          sc[4 * h + i] = s * rf;
        }
      }
    }
    if constexpr (DH == 2) {
      // the other wave's groups: its parts of the same scores
      if (any) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
          L.st.xch[wave][h][lane] = v4f{sc[4 * h], sc[4 * h + 1], sc[4 * h + 2], sc[4 * h + 3]};
      }
      __syncthreads();
      if (any) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const v4f x = L.st.xch[wave ^ RS][h][lane];
#pragma unroll
          for (int i = 0; i < 4; ++i) sc[4 * h + i] += x[i];
        }
      }
    }
    if (any) {
      const bool inside = t0 + 31 <= pos_lo && (W_ == 0 || pos_hi - t0 < W_);  // wave-uniform
      if (!inside) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int t = t0 + 16 * (j >> 2) + 4 * c + (j & 3);
          sc[j] = t <= pos && (W_ == 0 || pos - t < W_) ? sc[j] : -INFINITY;
        }
      }

      // ---- online softmax (log2 domain) of rows m ------------------------------
      const float up = static_cast<float>(e0 - kPfHead);
      float mt = sc[0];
#pragma unroll
      for (int j = 1; j < 8; ++j) mt = fmaxf(mt, sc[j]);
      const float need = xor32_max(xor16_max(mt)) + up;
      // (a row with nothing attended yet and nothing here keeps -inf)
      if (__any(need > m_ref + kPfLazy)) {
        const float m_new = need > m_ref ? need : m_ref;
        const float f = m_new == m_ref ? 1.0f : merge_factor(m_ref, m_new);
        l_run *= f;
#pragma unroll
        for (int b = 0; b < 4 * NWG; ++b) o[b] *= f;
#pragma unroll
        for (int g = 0; g < NWG; ++g) bsum[g] *= f;
        m_ref = m_new;
      }
      float pw[8];
      // (with nothing attended so far, -inf - -inf would be NaN)
      const float ms = m_ref == -INFINITY ? 0.0f : m_ref;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        pw[j] = fast_exp2(sc[j] - ms);
        l_run += pw[j];
      }

      // ---- O^T += V^T P^T ----------------------------------------------------
      // B operands of eight weights, and O^T's 16 dims x of group g
      const auto split = [&](const float (&y)[8], v8h& bh, v8h& bl) {
        u32x4 hi, lw;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          hi[q] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(y[2 * q], y[2 * q + 1]));
          lw[q] = pf_rem_pair(hi[q], y[2 * q], y[2 * q + 1]);
        }
        bh = __builtin_bit_cast(v8h, hi);
        bl = __builtin_bit_cast(v8h, lw);
      };
      float pz[8];  // the weights of the common products
#pragma unroll
      for (int j = 0; j < 8; ++j) pz[j] = pw[j];
      int al = 1;
#pragma unroll
      for (int i = 0; i < Gm::NSW; ++i) al &= alike[buf][i];
      if (!__builtin_amdgcn_readfirstlane(al)) {
        // V scales apart: the largest weight of every row and group to 2^13 .. 2^14
        // (an infinity, of exponent 0, stays one), the products on their own, added
        // in fp32
#pragma unroll
        for (int g = 0; g < NWG; ++g) {
          float y[8], mx = 0.0f;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            y[j] = static_cast<float>(svs[(16 * (j >> 2) + 4 * c + (j & 3)) * NG + g]) * pw[j];
            mx = fmaxf(mx, fabsf(y[j]));
          }
          const int k = min(14 - __builtin_amdgcn_frexp_expf(xor32_max(xor16_max(mx))), 120);
          const float un = ldexpf(1.0f, -k);
#pragma unroll
          for (int j = 0; j < 8; ++j) y[j] = ldexpf(y[j], k);
          v8h bh, bl;
          split(y, bh, bl);
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const v8h a = __builtin_bit_cast(v8h, vu[(4 * g + x) * 64 + (m ^ Gm::vswz(g))]);
            v4f t = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bh, z, 0, 0, 0);
            t = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bl, t, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) o[4 * g + x][i] = fmaf(t[i], un, o[4 * g + x][i]);
          }
        }
        // (nothing is left for the products below: a branch around them cost 50 registers)
#pragma unroll
        for (int j = 0; j < 8; ++j) pz[j] = 0.0f;
      }
      SB s[8][NWG], bb[8][NWG];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = 16 * (j >> 2) + 4 * c + (j & 3);
#pragma unroll
        for (int g = 0; g < NWG; ++g) {
          s[j][g] = svs[key * NG + g];
          bb[j][g] = svb[key * NG + g];
        }
      }
#pragma unroll
      for (int g = 0; g < NWG; ++g) {
        v8h bh, bl;
        float y[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          y[j] = fmaf(static_cast<float>(s[j][g]), pz[j], 0.0f);
          // b' = b + 8 s
          bsum[g] = fmaf(fmaf(static_cast<float>(s[j][g]), 8.0f, static_cast<float>(bb[j][g])), pw[j], bsum[g]);
        }
        split(y, bh, bl);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const v8h a = __builtin_bit_cast(v8h, vu[(4 * g + x) * 64 + (m ^ Gm::vswz(g))]);
          v4f& acc = o[4 * g + x];
          acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bh, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bl, acc, 0, 0, 0);
        }
      }
    }
    if (it + 1 < ntile) {
      pf_store<Gm>(L.st, raw, buf ^ 1);
      pf_alike<Gm>(raw, e0, alike[buf ^ 1]);
    }
    __syncthreads();
  }

  // ---- merge of the KH partials of every row, and the output ------------------
  const float un = c < 2 ? 1.0f : 0.0625f;  // odd nibbles (rows 8-15) were 16 times as large
  const float lt = xor32_sum(xor16_sum(l_run));
  if (c == 0) {
    ml[wave][m] = m_ref;
    ll[wave][m] = lt;
  }
  float* orow = L.o[wave] + m * Gm::OSTR;
#pragma unroll
  for (int g = 0; g < NWG; ++g) {
    const float bg = xor32_sum(xor16_sum(bsum[g]));
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        orow[64 * g + 8 * (4 * (c & 1) + i) + 2 * x + (c >> 1)] = fmaf(o[4 * g + x][i], un, bg);
  }
  __syncthreads();
  for (int u = threadIdx.x; u < 16 * RS * (D / 2); u += Gm::NT) {
    // a wave's 64 units lie in one row and in one wave's dims
    const int r = __builtin_amdgcn_readfirstlane(u / (D / 2)), d = 2 * (u % (D / 2));
    const int Ro = r0 + r;
    if (Ro >= total) break;
    const int rm = r % 16, w0 = r / 16 + RS * KH * (d / Gm::OW);
    float M = -INFINITY;
#pragma unroll
    for (int k = 0; k < KH; ++k) M = fmaxf(M, ml[w0 + RS * k][rm]);
    float l = 0.0f, x0 = 0.0f, x1 = 0.0f;
#pragma unroll
    for (int k = 0; k < KH; ++k) {
      const int wv = w0 + RS * k;
      const float f = merge_factor(ml[wv][rm], M);
      const float2 v = *reinterpret_cast<const float2*>(&L.o[wv][rm * Gm::OSTR + d % Gm::OW]);
      l = fmaf(ll[wv][rm], f, l);
      x0 = fmaf(v.x, f, x0);
      x1 = fmaf(v.y, f, x1);
    }
    const int qo = Ro / p.gqa;
    float* out = p.out + (static_cast<int64_t>(qo) * p.Hq + kvh * p.gqa + (Ro - qo * p.gqa)) * D + d;
    *reinterpret_cast<float2*>(out) = make_float2(normalise(x0, l, 0.0f), normalise(x1, l, 0.0f));
  }
}

// Tiles of 64 keys and two waves a row set, one per 32 keys (D 128 / 256), or
// of 32 keys and two waves a row set, one per half of the dims (D 512; a tile's
// two buffers fill the LDS): eight waves, two per SIMD.
//
// What bounds it: the VALU (about 420 instructions a wave and 32 keys -- weights
// times scales and their split 80, exponentials and masks 90, staging 80, bias
// terms 64, score scales 40 -- against 50 products), busy 60% of the time, the
// rest being phases of the two waves that do not overlap.  Measured (512 queries
// after 3,584 keys; before: loader waves that dequantized every tile into hi / lo
// images, whose LDS reads, three products each, bound it):
//   Hq 32 Hkv 16 D 256, window 1,024: 94.9 -> 61 us; without window 275 -> 183
//   Hq 32 Hkv 4 D 512: 678 -> 386 us;  Hq 16 Hkv 8 D 128: 148 -> 110 us
// A power of two per row and group for every tile, with a check and a branch per
// group, in place of the two kinds of tile: 77 us, 229, 464, 122.
// Slower: nibbles expanded by every wave (no operand images; 70 us before they
// were centred, which would add 128 instructions), two row sets a wave at one
// wave per SIMD (97 us), operand reads half a tile ahead (68), the two waves of
// a SIMD staging at opposite ends of a tile (69).
//
// One body under two names, by which the plan and traces tell D 512 from the
// rest; no wave has a role of its own in either.
template <int D, bool F32, int RS>
__global__ __launch_bounds__(128 * RS) __attribute__((amdgpu_waves_per_eu(RS == 4 ? 2 : 1, RS == 4 ? 2 : 1)))
void prefill_int4_ws_kernel(SdpaParams p) {
  pin_args(p);
  prefill_rows<D, F32, RS>(p);
}

template <int D, bool F32, int RS>
__global__ __launch_bounds__(128 * RS) __attribute__((amdgpu_waves_per_eu(RS == 4 ? 2 : 1, RS == 4 ? 2 : 1)))
void prefill_int4_kernel(SdpaParams p) {
  pin_args(p);
  prefill_rows<D, F32, RS>(p);
}

template <int D, bool F32, int RS>
void launch_sets(const SdpaParams& p, unsigned grid, hipStream_t s) {
  if constexpr (D == 512) prefill_int4_kernel<D, F32, RS><<<grid, 128 * RS, 0, s>>>(p);
  else prefill_int4_ws_kernel<D, F32, RS><<<grid, 128 * RS, 0, s>>>(p);
}

// 32 rows per workgroup of four waves while that gives every CU at most one
// (twice the workgroups: 128 queries of Hq 32 Hkv 16 D 256 60 against 65 us, 100 of
// Hq 32 Hkv 8 D 128 24.7 against 26.6; 16 rows on two waves, which then stage a
// whole tile, 78 and 29), else 64.
template <int D, bool F32>
void launch_rows(const SdpaParams& p, hipStream_t s) {
  const int64_t rows = static_cast<int64_t>(p.nq) * p.gqa;
  const auto grid = [&](int rs) { return static_cast<unsigned>((rows + 16 * rs - 1) / (16 * rs) * p.Hkv); };
  if (grid(2) <= static_cast<unsigned>(target_wgs())) launch_sets<D, F32, 2>(p, grid(2), s);
  else launch_sets<D, F32, 4>(p, grid(4), s);
}

template <bool F32>
void launch_dim(const SdpaParams& p, int D, hipStream_t s) {
  if (D == 128) launch_rows<128, F32>(p, s);
  else if (D == 256) launch_rows<256, F32>(p, s);
  else launch_rows<512, F32>(p, s);
}

}  // namespace

// Returns false when the tile kernels do not serve the shape (the caller then
// runs the split-K decode kernels in prefill mode).
bool prefill_tiles_serve(int D, int sb_dtype, int gqa) {
  if ((sb_dtype != TQ_F16 && sb_dtype != TQ_F32) || (D != 128 && D != 256 && D != 512)) return false;
  return gqa >= 1 && gqa <= 64 && 64 % gqa == 0;
}

int launch_prefill_tiles(const SdpaParams& p, int D, int sb_dtype, hipStream_t s) {
  if (!prefill_tiles_serve(D, sb_dtype, p.gqa)) return -1;
  if (p.q_dtype == TQ_F32) return launch_prefill_tiles_f32(p, D, sb_dtype, s);
  if (sb_dtype == TQ_F32) launch_dim<true>(p, D, s);
  else launch_dim<false>(p, D, s);
  TQ_CHECK_LAUNCH("prefill_int4_kernel");
  return TQ_OK;
}

}  // namespace tq
