// gemm_x3.hip -- fp32 and W4 matrix products on the bf16 matrix cores.
//
// Every fp32 operand is split into three bf16 parts, x = h + m + l exactly (8 +
// 8 + 8 significant bits: h = bf16(x), m = bf16(x - h), l = x - h - m), whose
// products are exact in fp32 (the splitting of G. Henry, P. Tang and A. Heinecke,
// "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", ARITH 2019).  A product of two fp32 values keeps the six parts
// hh, hm, mh, hl, lh and mm; each of the three dropped ones is below 2^-25 of it,
// together they reach 2^-24, half a unit of fp32, at most.  A W4 weight is one
// exact bf16, so there the three products are all of them.
// v_mfma_f32_16x16x32_bf16 runs at 16 times the rate of v_mfma_f32_16x16x4_f32 and
// rounds its accumulator once per 32 products instead of once per 4: six of them
// take less time than the fp32 MFMA, and from four products a sum on come closer to
// 64 bits than the fp32 kernels (K = 4 / 32 / 128 / 512, closed every step 3.3e-8 /
// 3.7e-8 / 5.5e-8 / 7.0e-8 off in the 2-norm, carried 3.2e-8 / 3.8e-8 / 1.5e-7 /
// 3.4e-7, fp32 MFMA or FMA 4.0e-8 / 1.0e-7 / 2.0e-7 / 4.1e-7).  What they do
// not have is a mean error of zero: up to one step, where no sign has turned
// yet, it is 0.16 to 0.35 of the root mean square one, towards smaller values.
#include <algorithm>
#include <type_traits>

#include "rt_device.h"
#include "rt_internal.h"

namespace simp {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
// 16-byte loads and stores of floats that are only 4-byte aligned (odd leading
// dimensions): the type says so, and the compiler picks the instruction.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

enum { kBKN = 0, kBNK = 1, kBW4 = 2 };  // B[K,N], B_T[N,K], W4 rows [N, K/2]

__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  typedef float f2 __attribute__((ext_vector_type(2)));
  const f2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, b2));
}

struct Planes {
  b8 h, m, l;
};

// The matrix cores flush bf16 subnormals, which the low parts of an x below
// 2^-102 would be.  So x is scaled by 2^24 first (exact; the sums are scaled
// back at the end): every fp32 value down to the subnormals keeps its 24 bits,
// and one above 2^103 overflows into the non-finite sums that are formed again
// in fp32.
constexpr float kUp = 16777216.f;

// The three bf16 parts of eight floats, scaled by `up`.
__device__ __forceinline__ Planes split8(const float (&x)[8], float up = kUp) {
  uint32_t h[4], m[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float x0 = up * x[2 * i], x1 = up * x[2 * i + 1];
    h[i] = pk_bf16(x0, x1);
    const float r0 = x0 - __uint_as_float(h[i] << 16), r1 = x1 - __uint_as_float(h[i] & 0xFFFF0000u);
    m[i] = pk_bf16(r0, r1);
    l[i] = pk_bf16(r0 - __uint_as_float(m[i] << 16), r1 - __uint_as_float(m[i] & 0xFFFF0000u));
  }
  Planes p;
  p.h = __builtin_bit_cast(b8, make_uint4(h[0], h[1], h[2], h[3]));
  p.m = __builtin_bit_cast(b8, make_uint4(m[0], m[1], m[2], m[3]));
  p.l = __builtin_bit_cast(b8, make_uint4(l[0], l[1], l[2], l[3]));
  return p;
}

// Eight signed nibbles (low nibble first) as bf16 sixteenths: v_cvt_off_f32_i4
// gives q / 16, exact in the upper half of its fp32 form.  The caller's scale
// carries the 16.
__device__ __forceinline__ b8 nib8_bf16(uint32_t w) {
  const uint32_t v = w >> 4;
  uint32_t p[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float lo = __builtin_amdgcn_cvt_off_f32_i4(w >> (8 * i));
    const float hi = __builtin_amdgcn_cvt_off_f32_i4(v >> (8 * i));
    p[i] = __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
  }
  return __builtin_bit_cast(b8, make_uint4(p[0], p[1], p[2], p[3]));
}

__device__ __forceinline__ v4f mfma_bf16(b8 a, b8 b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// One of up to three matrices B whose columns stand side by side in C.
struct X3Part {
  const void *B;
  const float *S;    // W4 scales [n, lds], one per `cpg` groups of 32
  int n;             // columns
  int c0, t0;        // first column of C, first column tile
};
struct X3Args {
  const float *A;
  int64_t lda;
  X3Part part[3];
  int parts;
  int64_t ldb;       // floats; bytes for W4
  int64_t lds;
  int cpg, cpg_shift;
  float *C;
  int64_t ldc;
  float *P;          // partial products [split][M][N]; null: straight to C
  int M, N, K;       // N: the columns of all parts
  int span;          // K steps of 32 per split
  int tiles_m, tiles_n, splits;
  float beta;
};

// C = beta C + A B.  One workgroup of NW waves: 16 MT rows of C by 16 NT NW
// columns, K in steps of 32.
//   * A is shared by all waves: its fp32 elements come through registers, are
//     split once and go to LDS as fragments in lane order (lane l = 16 g + r
//     of a 16-row block holds row r, k = 8g .. 8g+7: 16 bytes per part), so
//     every LDS write and read is 1 KB in lane order, free of conflicts.  Two
//     buffers, one barrier per step.
//   * B's columns belong to one wave each, so B goes straight from global
//     memory to the registers of the lane that feeds it to the MFMA (lane (n =
//     l % 16, g): k = 8g .. 8g+7), PD steps ahead, and is split there: no LDS
//     traffic and no barrier for the operand that is streamed.  B[K,N]: eight
//     4-byte loads, 16 lanes side by side; B_T: 32 bytes of a row; W4: 4 bytes
//     of a row and its scale.
//   * fp32 B: the MFMA takes B first, so a lane ends with 4 consecutive columns
//     of a row of C.  W4: A first, so a lane's column and scale are one each;
//     a step is one group of 32 or part of a longer one.
//   * The bf16 MFMA rounds its sums down (measured: the mean error is half the
//     root mean square one and negative), so a sum carried through it gathers a
//     bias that averages over rows do not take out.  So each step is summed
//     from zero and added to the accumulator by the VALU, which rounds to
//     nearest, and A's sign turns with every step: 512x4096x4096 is 2e-7 off
//     64-bit sums (the fp32 MFMA kernel 1.2e-6).  CARRY leaves the sums in the
//     MFMA accumulator and turns its sign and A's every four steps (1e-6 off;
//     1024x4096x4096 188 us against 219, 4096^3 690 against 830).
//   * Nothing depends on the alignment of any operand beyond its type's
//     (W4: rows of 4-byte aligned bytes).  Rows past M and columns past N read
//     the last one and are not stored; only the last step reads under a mask.
//   * What bounds it: large products the MFMA rate the chip sustains (4096^3: 580
//     to 690 us from card to card against 1020 for the fp32 MFMA kernel; the MFMA pipe
//     is busy 65% of the cycles at 1.75 GHz, 1.2 PFLOP/s of bf16, where a bf16
//     library GEMM reaches 1.1 to 1.4); mid sizes the splitting next to it
//     (128x2048x8192 32.8 us against 43.0, 301x1537x2003 with B_T 23.1 against 227
//     for the SIMT kernel that odd sizes took; a copy without the operand loads
//     runs as long).  W4:
//     the nibble conversion and the scaling (200x3200x8640: 58 us; one thread
//     per output took 131 ms).
//   * A part that overflows or an infinite or NaN operand makes its products
//     NaN where fp32 arithmetic may give an infinity: 16x16 tiles with a
//     non-finite sum are formed again with v_mfma_f32_16x16x4_f32 from the fp32
//     operands, without LDS.  Both operands are scaled by 2^24, so that happens to
//     finite products too, where a sum on its way reaches 2^80 (W4: 2^104 before
//     its scale) or an operand 2^104.  It costs: 4096^3 0.58 ms, with one infinity
//     in A 1.46 and in B 0.81 (6.0 and 4.9 when whole tiles of a wave were formed
//     again), with all sums beyond 8.0, where the fp32 MFMA kernel takes 1.02
//     whatever the values.
template <int MT, int NT, int NW, int KIND, int PD, bool CARRY = false, int PA = 2>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2)))
    gemm_x3(const X3Args a) {
  constexpr int CH = (MT + NW - 1) / NW;  // 16-row blocks of A a wave stages
  constexpr bool W4 = KIND == kBW4;
  __shared__ uint4 As[2][MT * 3 * 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, g = lane >> 4;

  // XCD-contiguous order over (split, tile): the tiles of one XCD share their
  // columns of B, or their rows of A, in its L2
  const int tiles = a.tiles_m * a.tiles_n, nb = tiles * a.splits;
  int tm, tn, split;
  {
    const int q = nb >> 3, r = nb & 7, xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
    const int t = xcd * q + min(xcd, r) + local;
    split = t / tiles;
    constexpr int G = 8;
    const int w = t - split * tiles, gsz = G * a.tiles_n, gi = w / gsz, first = gi * G;
    const int gm = min(a.tiles_m - first, G), v = w - gi * gsz;
    tm = first + v % gm;
    tn = v / gm;
  }
  const X3Part b = a.part[(a.parts > 1 && tn >= a.part[1].t0) + (a.parts > 2 && tn >= a.part[2].t0)];
  const int m0 = tm * 16 * MT, n0 = ((tn - b.t0) * NW + wave) * 16 * NT;
  const int s0 = split * a.span, s1 = min(s0 + a.span, (a.K + 31) >> 5);
  const int kend = min(a.K, 32 * s1);

  // ---- operand loads
  const float *arow[CH];
#pragma unroll
  for (int i = 0; i < CH; i++) {
    const int mt = wave + i * NW;
    arow[i] = a.A + (int64_t)min(m0 + 16 * mt + r16, a.M - 1) * a.lda + 8 * g;
  }
  // a lane's eight floats of a row at step k0 (p is at 8g); `full`: all below K
  auto load8 = [&](const float *p, int k0, float (&v)[8], auto full) {
    if constexpr (decltype(full)::value) {
      const f4u u0 = *(const f4u *)(p + k0), u1 = *(const f4u *)(p + k0 + 4);
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = u0[e], v[4 + e] = u1[e];
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++) v[e] = k0 + 8 * g + e < a.K ? p[k0 + e] : 0.f;
    }
  };
  struct RawF { float v[NT][8]; };
  struct RawW { uint32_t w[NT]; float s[NT]; };
  using Raw = std::conditional_t<W4, RawW, RawF>;
  const float *brow[NT];    // B_T rows, or the W4 scales
  const uint8_t *wrow[NT];  // W4 rows
  uint32_t boff[NT];        // B[K,N]: byte offset of (8g, n)
#pragma unroll
  for (int j = 0; j < NT; j++) {
    const int n = min(n0 + 16 * j + r16, b.n - 1);
    if constexpr (KIND == kBKN) boff[j] = 4u * (uint32_t)(8 * g * (uint32_t)a.ldb + (uint32_t)n);
    if constexpr (KIND == kBNK) brow[j] = (const float *)b.B + (int64_t)n * a.ldb + 8 * g;
    if constexpr (W4) {
      wrow[j] = (const uint8_t *)b.B + (int64_t)n * a.ldb + 4 * g;
      brow[j] = b.S + (int64_t)n * a.lds;
    }
  }
  const uint32_t ldb4 = 4u * (uint32_t)a.ldb;
  auto loadb = [&](int s, Raw &r, auto full) {
    const int k0 = 32 * s;
    if constexpr (KIND == kBKN) {
      const char *base = (const char *)b.B + (int64_t)k0 * a.ldb * 4;
      if constexpr (decltype(full)::value) {
        // buffer loads: the step's base and the k-row's offset in SGPRs, the
        // lane's offset fixed, so a load costs no address arithmetic
        const __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, 31u * ldb4 + 4u * b.n, 0x00020000);
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
          for (int e = 0; e < 8; e++)
            r.v[j][e] = __uint_as_float(
                __builtin_amdgcn_raw_buffer_load_b32(rs, (int)boff[j], (int)(e * ldb4), 0));
      } else {
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
          for (int e = 0; e < 8; e++)
            r.v[j][e] = k0 + 8 * g + e < a.K
                            ? *(const float *)(base + (boff[j] + e * ldb4)) : 0.f;
      }
    } else if constexpr (KIND == kBNK) {
#pragma unroll
      for (int j = 0; j < NT; j++) load8(brow[j], k0, r.v[j], full);
    } else {
      const int gr = chunk_group(s, a.cpg, a.cpg_shift);
#pragma unroll
      for (int j = 0; j < NT; j++) {
        r.w[j] = *(const uint32_t *)(wrow[j] + 16 * s);
        r.s[j] = brow[j][gr];
      }
    }
  };
  struct RawA { float v[CH][8]; };
  auto loada = [&](int s, RawA &r, auto full) {
#pragma unroll
    for (int i = 0; i < CH; i++)
      if (MT % NW == 0 || wave + i * NW < MT) load8(arow[i], 32 * s, r.v[i], full);
  };
  auto storea = [&](int buf, const RawA &r, float sg) {
#pragma unroll
    for (int i = 0; i < CH; i++) {
      const int mt = wave + i * NW;
      if (MT % NW == 0 || mt < MT) {
        const Planes p = split8(r.v[i], sg * kUp);
        As[buf][(mt * 3 + 0) * 64 + lane] = __builtin_bit_cast(uint4, p.h);
        As[buf][(mt * 3 + 1) * 64 + lane] = __builtin_bit_cast(uint4, p.m);
        As[buf][(mt * 3 + 2) * 64 + lane] = __builtin_bit_cast(uint4, p.l);
      }
    }
  };
  // B's fragments of a step: the three parts, or the W4 integers and scales
  struct FragF { Planes b[NT]; };
  struct FragW { b8 w[NT]; float s[NT]; };
  using Frag = std::conditional_t<W4, FragW, FragF>;
  auto convert = [&](const Raw &r, Frag &f) {
#pragma unroll
    for (int j = 0; j < NT; j++) {
      if constexpr (W4) {
        f.w[j] = nib8_bf16(r.w[j]);
        f.s[j] = 16.f * r.s[j];
      } else {
        f.b[j] = split8(r.v[j]);
      }
    }
  };

  v4f acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  auto frag = [&](int buf, int i) {  // the parts of A's 16-row block i
    Planes p;
    p.h = __builtin_bit_cast(b8, As[buf][(i * 3 + 0) * 64 + lane]);
    p.m = __builtin_bit_cast(b8, As[buf][(i * 3 + 1) * 64 + lane]);
    p.l = __builtin_bit_cast(b8, As[buf][(i * 3 + 2) * 64 + lane]);
    return p;
  };
  // the sign of A in step s and of the carried sums
  auto sign = [&](int s) { return CARRY && ((s - s0) >> 2) & 1 ? -1.f : 1.f; };
  auto compute = [&](int buf, const Frag &f, float sg) {
    // two row blocks at a time: the MFMAs of one sum are 2 NT apart
    constexpr int R = MT % 2 == 0 ? 2 : 1;
    if constexpr (W4) {
#pragma unroll
      for (int i = 0; i < MT; i += R) {
        Planes p[R];
        v4f d[R][NT];
#pragma unroll
        for (int q = 0; q < R; q++) p[q] = frag(buf, i + q);
        auto mul = [&](b8 Planes::*y, auto zero) {
#pragma unroll
          for (int q = 0; q < R; q++)
#pragma unroll
            for (int j = 0; j < NT; j++)
              d[q][j] = mfma_bf16(p[q].*y, f.w[j],
                                  decltype(zero)::value ? v4f{0.f, 0.f, 0.f, 0.f} : d[q][j]);
        };
        mul(&Planes::l, std::true_type{});
        mul(&Planes::m, std::false_type{});
        mul(&Planes::h, std::false_type{});
#pragma unroll
        for (int q = 0; q < R; q++)
#pragma unroll
          for (int j = 0; j < NT; j++)
#pragma unroll
            for (int e = 0; e < 4; e++)
              acc[i + q][j][e] = fmaf(sg < 0.f ? -f.s[j] : f.s[j], d[q][j][e], acc[i + q][j][e]);
      }
    } else {
      // small parts first
#pragma unroll
      for (int i = 0; i < MT; i += R) {
        Planes p[R];
#pragma unroll
        for (int q = 0; q < R; q++) p[q] = frag(buf, i + q);
        v4f d[R][NT];
        auto mul = [&](b8 Planes::*x, b8 Planes::*y, auto zero) {
#pragma unroll
          for (int q = 0; q < R; q++)
#pragma unroll
            for (int j = 0; j < NT; j++) {
              v4f &c = CARRY ? acc[i + q][j] : d[q][j];
              c = mfma_bf16(f.b[j].*x, p[q].*y,
                            decltype(zero)::value ? v4f{0.f, 0.f, 0.f, 0.f} : c);
            }
        };
        mul(&Planes::h, &Planes::l, std::bool_constant<!CARRY>{});
        mul(&Planes::l, &Planes::h, std::false_type{});
        mul(&Planes::m, &Planes::m, std::false_type{});
        mul(&Planes::h, &Planes::m, std::false_type{});
        mul(&Planes::m, &Planes::h, std::false_type{});
        mul(&Planes::h, &Planes::h, std::false_type{});
        if constexpr (!CARRY) {
#pragma unroll
          for (int q = 0; q < R; q++)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
              for (int e = 0; e < 4; e++)
                acc[i + q][j][e] = sg < 0.f ? acc[i + q][j][e] - d[q][j][e]
                                            : acc[i + q][j][e] + d[q][j][e];
        }
      }
    }
  };
  auto negate = [&] {
    if constexpr (CARRY) {
#pragma unroll
      for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
          for (int e = 0; e < 4; e++) acc[i][j][e] = -acc[i][j][e];
    }
  };

  // Whole steps s0 .. sf-1, software-pipelined: step s's MFMAs run while step
  // s+1's operands are split (A into the other LDS buffer, B into registers)
  // and the loads of the steps up to s+1+PA (A) and s+1+PD (B) are in flight.
  // Loads return in order, so each step requests its A before its B: waiting
  // for A then leaves the younger loads of B outstanding.  Loads past the last
  // whole step repeat it: in bounds, never used.
  using Full = std::true_type;
  using Part = std::false_type;
  const int sf = min(s1, a.K >> 5), last = sf - 1;
  const int sg0 = s0 + max(sf - s0, 0) / 4 * 4;  // end of the whole runs of four
  if (s0 < sf) {
    RawA ra[PA];
    Raw rb[PD];
    Frag fr[2];
    loada(s0, ra[0], Full{});
    loadb(s0, rb[0], Full{});
    storea(0, ra[0], 1.f);
    convert(rb[0], fr[0]);
#pragma unroll
    for (int p = 0; p < PA || p < PD; p++) {
      if (p < PA) loada(min(s0 + 1 + p, last), ra[p], Full{});
      if (p < PD) loadb(min(s0 + 1 + p, last), rb[p], Full{});
    }
    lds_barrier();
    static_assert(4 % PD == 0 && 4 % PA == 0, "unroll");
    auto step = [&](int s, auto pp) {
      constexpr int p = decltype(pp)::value;
      // the sign of A in this step and in the next
      const float sg = CARRY ? sign(s) : p & 1 ? -1.f : 1.f, sn = CARRY ? sign(s + 1) : -sg;
      storea((p & 1) ^ 1, ra[p % PA], sn);
      loada(min(s + 1 + PA, last), ra[p % PA], Full{});
      convert(rb[p % PD], fr[(p + 1) & 1]);
      loadb(min(s + 1 + PD, last), rb[p % PD], Full{});
      compute(p & 1, fr[p & 1], sg);
      lds_barrier();
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    // (a test before each step keeps the compiler from merging the four: merged,
    // W4 ran 16% longer and fp32 10%)
    for (int s = s0; s < sf; s += 4) {
      step(s, I0{});
      if (s + 1 < sf) step(s + 1, I1{});
      if (s + 2 < sf) step(s + 2, I2{});
      if (s + 3 < sf) {
        step(s + 3, I3{});
        negate();
      }
    }
  }
  if (sf < s1) {  // the last K % 32 (never for W4)
    RawA ra;
    Raw r;
    Frag f;
    loada(sf, ra, Part{});
    loadb(sf, r, Part{});
    convert(r, f);
    storea(0, ra, sign(sg0));  // the pipeline's last step ended in a barrier
    lds_barrier();
    compute(0, f, sign(sg0));
  }

  // ---- scale back; sums that are not finite, again in fp32
  const float down = (W4 ? 1.f / kUp : 1.f / kUp / kUp) * (CARRY ? sign(sg0) : 1.f);
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) acc[i][j][e] *= down;
  bool bad = false;
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) bad |= !(fabsf(acc[i][j][e]) <= 3.4028235e38f);
  if (__builtin_expect(__any(bad), 0)) {
    uint32_t which = 0;  // 16x16 tiles of this wave
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int j = 0; j < NT; j++) {
        bool b16 = false;
#pragma unroll
        for (int e = 0; e < 4; e++) b16 |= !(fabsf(acc[i][j][e]) <= 3.4028235e38f);
        if (__any(b16)) which |= 1u << (i * NT + j);
      }
#pragma unroll 1
    for (int t = 0; t < MT * NT; t++) {
      if (!(which >> t & 1)) continue;
      const int ti = t / NT, tj = t - ti * NT;
      const float *ap = a.A + (int64_t)min(m0 + 16 * ti + r16, a.M - 1) * a.lda;
      const int n = min(n0 + 16 * tj + r16, b.n - 1);
      auto bat = [&](int kk) {
        if constexpr (KIND == kBKN) return ((const float *)b.B)[(int64_t)kk * a.ldb + n];
        if constexpr (KIND == kBNK) return ((const float *)b.B)[(int64_t)n * a.ldb + kk];
        if constexpr (W4) {
          const uint8_t w = ((const uint8_t *)b.B)[(int64_t)n * a.ldb + (kk >> 1)];
          const int q = (int)((uint32_t)w << (kk & 1 ? 24 : 28)) >> 28;
          return (float)q * b.S[(int64_t)n * a.lds + chunk_group(kk >> 5, a.cpg, a.cpg_shift)];
        }
      };
      v4f c = {0.f, 0.f, 0.f, 0.f};
      auto mul = [&](float av, float bv) {
        c = W4 ? __builtin_amdgcn_mfma_f32_16x16x4f32(av, bv, c, 0, 0, 0)
               : __builtin_amdgcn_mfma_f32_16x16x4f32(bv, av, c, 0, 0, 0);
      };
      int k = 32 * s0;
      for (; k + 32 <= kend; k += 32) {  // eight loads of each operand in flight
        float av[8], bv[8];
#pragma unroll
        for (int u = 0; u < 8; u++) av[u] = ap[k + 4 * u + g], bv[u] = bat(k + 4 * u + g);
#pragma unroll
        for (int u = 0; u < 8; u++) mul(av[u], bv[u]);
      }
      for (; k < kend; k += 4) {
        const bool in = k + g < kend;
        mul(in ? ap[k + g] : 0.f, in ? bat(k + g) : 0.f);
      }
#pragma unroll
      for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
          if (i * NT + j == t) acc[i][j] = c;
    }
  }

  // ---- store
  float *out = (a.P ? a.P + (int64_t)split * a.M * a.N : a.C) + b.c0;
  const int64_t ldo = a.P ? a.N : a.ldc;
  const bool add = !a.P && a.beta != 0.f;
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) {
      if constexpr (W4) {
        // rows 4g .. 4g+3 of column r16
        const int n = n0 + 16 * j + r16;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int m = m0 + 16 * i + 4 * g + e;
          if (m < a.M && n < b.n) {
            float *o = out + (int64_t)m * ldo + n;
            *o = add ? *o + acc[i][j][e] : acc[i][j][e];
          }
        }
      } else {
        // columns 4g .. 4g+3 of row r16
        const int m = m0 + 16 * i + r16, n = n0 + 16 * j + 4 * g;
        if (m < a.M) {
          float *o = out + (int64_t)m * ldo + n;
          if (n + 3 < b.n) {
            f4u v = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
            if (add) v += *(const f4u *)o;
            *(f4u *)o = v;
          } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
              if (n + e < b.n) o[e] = add ? o[e] + acc[i][j][e] : acc[i][j][e];
          }
        }
      }
    }
}

// out[m][n] = beta out + sum over parts p (in order: deterministic) of
// P[p][m][n]; the loads of B parts are issued together.
template <int B>
__global__ void __launch_bounds__(256)
    x3_sum_parts(const float *__restrict__ P, int parts, float *__restrict__ C, int64_t ldc, int M,
                 int N, float beta) {
  const int64_t mn = (int64_t)M * N, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= mn) return;
  float v = 0.f;
  for (int s = 0; s < parts; s += B) {
    float t[B];
#pragma unroll
    for (int u = 0; u < B; u++) t[u] = s + u < parts ? P[(int64_t)(s + u) * mn + i] : 0.f;
#pragma unroll
    for (int u = 0; u < B; u++)
      if (s + u < parts) v += t[u];
  }
  const int64_t m = i / N;
  float *o = C + m * ldc + (i - m * N);
  *o = beta != 0.f ? *o + v : v;
}

// K splits for `tiles` tiles of `steps` K steps: a round of workgroups over the
// CUs costs its steps and about four more to fill and drain its pipeline; the
// partial sums cost a launch (about three steps' time) and their traffic (a
// step is about 1 us, in which 4 MB go by).  Measured (W4, 200 x 3200 -> 8640,
// 68 tiles: 3 / 6 / 7 splits 61 / 72 / 71 us).  More than 16 splits only within
// one round (64x256x8640, 2 tiles: 16 / 30 splits 19.7 / 14.8 us).
int pick_splits(int64_t tiles, int steps, int64_t mn, int64_t cus) {
  int best = 1;
  double cost = 0;
  for (int s = 1; s <= 32 && s * 4 <= std::max(steps, 4); s++) {
    const int span = (int)cdiv(steps, s);
    if (cdiv(steps, span) != s) continue;
    if (s > 16 && tiles * s > cus) break;
    if (s > 1 && s * mn > (int64_t(1) << 28)) break;  // 1 GiB of partials
    const double c = (double)cdiv(tiles * s, cus) * (span + 4) +
                     (s > 1 ? 3.0 + 1e-6 * (double)(s + 1) * (double)mn : 0.0);
    if (s == 1 || c < cost) best = s, cost = c;
  }
  return best;
}

// 128x256 tiles from two per CU on (4096^3: 686 us against 790 with 64x128)
bool large_tiles(int64_t cus, int M, int64_t N, bool carry) {
  return M > 32 && carry && cdiv(M, 128) * cdiv(N, 256) >= 2 * cus;
}

template <int MT, int NT, int NW, int KIND, int PD, bool CARRY = false>
int go_x3(X3Args a, bool must, hipStream_t st) {
  const int64_t cus = num_cus(), tm = cdiv(a.M, 16 * MT);
  int64_t tn = 0;
  a.N = 0;
  for (int i = 0; i < a.parts; i++) {
    a.part[i].c0 = a.N;
    a.part[i].t0 = (int)tn;
    a.N += a.part[i].n;
    tn += cdiv(a.part[i].n, 16 * NT * NW);
  }
  const int steps = (int)cdiv(a.K, 32);
  int splits = pick_splits(tm * tn, steps, (int64_t)a.M * a.N, cus);
  a.P = nullptr;
  Workspace ws;
  if (splits > 1 && !ws.try_get(st, sizeof(float) * (size_t)splits * a.M * a.N, (void **)&a.P, 3)) {
    if (!must) return 1;
    splits = 1;
    a.P = nullptr;
  }
  a.span = (int)cdiv(steps, splits);
  a.splits = (int)cdiv(steps, a.span);
  if (tm * tn * a.splits > INT32_MAX) return 1;
  a.tiles_m = (int)tm;
  a.tiles_n = (int)tn;
  KernelTimer kt(st, "gemm_x3");
  hipLaunchKernelGGL((gemm_x3<MT, NT, NW, KIND, PD, CARRY>), dim3((unsigned)(tm * tn * a.splits)),
                     dim3(64 * NW), 0, st, a);
  SIMP_HIP(hipGetLastError());
  if (a.P) {
    const dim3 g((unsigned)cdiv((int64_t)a.M * a.N, 256));
    if (a.splits <= 4)
      hipLaunchKernelGGL(x3_sum_parts<4>, g, dim3(256), 0, st, a.P, a.splits, a.C, a.ldc, a.M, a.N, a.beta);
    else if (a.splits <= 8)
      hipLaunchKernelGGL(x3_sum_parts<8>, g, dim3(256), 0, st, a.P, a.splits, a.C, a.ldc, a.M, a.N, a.beta);
    else
      hipLaunchKernelGGL(x3_sum_parts<16>, g, dim3(256), 0, st, a.P, a.splits, a.C, a.ldc, a.M, a.N, a.beta);
    SIMP_HIP(hipGetLastError());
  }
  return SIMP_RT_OK;
}

}  // namespace

// The model behind pick_splits with the constants of each tile in us, fitted
// together with mfma_f32_us (f32.hip), which tells the sizes and what choosing by
// it costs: fixed and per K split, per K step and round of tiles, and per million
// partial sums and outputs.
double split_f32_us(int64_t cus, bool bt, int M, int N, int K, bool carry) {
  struct Cost { double fixed, split, step, round, part, out; };
  static const Cost k32[2] = {{3.25, 2.0, 0.70, 0, 2.2, 0.5}, {3.8, 2.2, 0.60, 0, 2.5, 2.6}},
                    k64[2] = {{1.3, 2.0, 0.78, 2.75, 1.75, 0.77}, {2.8, 2.0, 0.71, 1.8, 2.1, 1.0}},
                    kCarry[2] = {{4.1, 4.4, 0.69, 0, 0.73, 0.92}, {2.8, 4.0, 0.72, 2.4, 0.9, 0.76}},
                    kLarge[2] = {{3.0, 4.4, 2.27, 0, 0.8, 1.0}, {3.0, 4.4, 2.19, 0, 0.8, 1.1}};
  const bool large = large_tiles(cus, M, N, carry);
  const Cost &c = (M <= 32 ? k32 : large ? kLarge : carry ? kCarry : k64)[bt];
  const int64_t mn = (int64_t)M * N;
  const int64_t tiles = M <= 32 ? cdiv(M, 32) * cdiv(N, 128)
                        : large ? cdiv(M, 128) * cdiv(N, 256) : cdiv(M, 64) * cdiv(N, 128);
  const int steps = (int)cdiv(K, 32);
  const int span = (int)cdiv(steps, pick_splits(tiles, steps, mn, cus)), s = (int)cdiv(steps, span);
  const double us = c.fixed + 1e-6 * c.out * mn + (double)cdiv(tiles * s, cus) * (c.step * span + c.round) +
                    (s > 1 ? c.split + 1e-6 * c.part * (s + 1) * mn : 0.) + 0.1 * std::min(K % 32, 8);
  // rows of B_T that are whole 128 bytes apart meet in the same memory channels; a
  // remainder of K is dearer yet to the fp32 MFMA kernels once they run many steps
  return us * (K % 32 ? K < 256 && !bt ? 1.05 : 0.93 : bt ? 1.06 : 1.);
}

int launch_x3(const X3Mat *mats, int nmat, int64_t ldb, X3Fmt fmt, int64_t lds, int gs,
              const float *A, int64_t lda, float *C, int64_t ldc, int M, int K, float beta,
              bool must, bool carry, hipStream_t st) {
  int64_t N = 0;
  for (int i = 0; i < nmat; i++) N += mats[i].n;
  if (M <= 0 || N <= 0 || K <= 0 || nmat > 3 || !indexes_fit(M, N, K)) return 1;
  // lane and row offsets of B[K,N] are 32-bit: 32 rows within 2 GiB
  if (fmt == X3Fmt::kN && ldb >= (int64_t(1) << 24)) return 1;
  X3Args a{};
  if (fmt == X3Fmt::kW4) {
    if (K % 32 != 0 || gs % 32 != 0 || K % gs != 0 || ldb % 4 != 0) return 1;
    a.cpg = gs / 32;
    a.cpg_shift = (a.cpg & (a.cpg - 1)) == 0 ? __builtin_ctz((unsigned)a.cpg) : -1;
  }
  for (int i = 0; i < nmat; i++) {
    if (fmt == X3Fmt::kW4 && ((uintptr_t)mats[i].B & 3) != 0) return 1;
    a.part[i] = X3Part{mats[i].B, mats[i].S, mats[i].n, 0, 0};
  }
  a.parts = nmat;
  a.A = A;
  a.lda = lda;
  a.ldb = ldb;
  a.lds = lds;
  a.C = C;
  a.ldc = ldc;
  a.M = M;
  a.K = K;
  a.beta = beta;
#define X3_GO(MT, NT, NW, ...)                                                         \
  (fmt == X3Fmt::kN ? go_x3<MT, NT, NW, kBKN, __VA_ARGS__>(a, must, st)                 \
                    : go_x3<MT, NT, NW, kBNK, __VA_ARGS__>(a, must, st))
  if (fmt == X3Fmt::kW4) {
    // 256 columns on 8 waves, which split A half as often, from 24 tiles on (200x
    // 3200x8640 61 us against 77, 64x3200x32000 60 against 65); fewer leave too
    // few workgroups to a split of K (64x8640x3200 28.8 against 26.8, 64x2048x2048
    // 19 against 15)
#define X3_W4(MT)                                                          \
  (cdiv(M, 16 * MT) * cdiv(N, 256) >= 24 ? go_x3<MT, 2, 8, kBW4, 4>(a, must, st) \
                                         : go_x3<MT, 2, 4, kBW4, 4>(a, must, st))
    return M <= 16 ? X3_W4(1) : M <= 32 ? X3_W4(2) : M <= 64 ? X3_W4(4) : X3_W4(8);
#undef X3_W4
  }
  // 16- and 32-row tiles for few rows (24x2048x8192: 16 us on 32x128 tiles of 8
  // waves, 22 on 32x64 of 4, 20 on 64x128)
  if (M <= 16) return X3_GO(1, 1, 4, 4);
  if (M <= 32) return X3_GO(2, 1, 8, 4);
  if (carry && large_tiles(num_cus(), M, N, carry)) return X3_GO(8, 2, 8, 2, true);
  if (carry) return X3_GO(4, 1, 8, 4, true);
  return X3_GO(4, 1, 8, 4);
#undef X3_GO
}

}  // namespace simp
