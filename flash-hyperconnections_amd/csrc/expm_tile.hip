// P in {16, 32} kernel (n = 9..32): one 64-lane wavefront per matrix, every
// product on the matrix cores: P = 16 on v_mfma_f32_16x16x4_f32, P = 32 on
// v_mfma_f32_32x32x16_bf16 with each FP32 value as the sum of three bf16 ones
// (and late squarings of very large operands on v_mfma_f32_32x32x2_f32; the
// section on bf16 below).
//
// Layout: a P x P matrix occupies R = P*P/64 VGPRs per lane in the MFMA
// accumulator ("D") layout: lane l, VGPR r holds M[row(l, r)][l % P] with
//   P = 16: row = 4*(l/16) + r
//   P = 32: row = 8*(r/4) + 4*(l/32) + r%4,
// i.e. row(l, r) = row0(l) + step(r).  Step r of a product feeds the A
// operand from VGPR r of X^T and the B operand from VGPR r of Y; lane group g
// then contributes k = row(g, r), so the R steps together cover k = 0..P-1 and
//   X.Y = sum_r mfma(a = (X^T).v[r], b = Y.v[r])
// needs no data movement for Y.  Left operands are transposed through a
// padded LDS tile (P x (P+1) floats); the workgroup is the one wavefront,
// whose LDS accesses complete in issue order, so the transposes need
// compiler ordering only, no barrier and no wait.
//
// On gfx950 the MFMA pipe and the VALU barely overlap (about 15% when
// different wavefronts of a SIMD feed them; not at all within one), so every
// VALU instruction adds to the MFMA time.  The kernel therefore keeps VALU
// work to the combines:
// * loads and stores go through buffer resources: one per-lane offset fixed
//   for the whole kernel, the per-VGPR row offsets in scalar registers and
//   the matrix base in the descriptor, so addressing costs no VALU;
// * no prefetch of a next matrix, on a grid of one wavefront per matrix
//   (P = 32) or four times the resident workgroups (P = 16): against a
//   persistent grid that prefetched the next matrix's storage bits, the
//   forward at config 5 ran 151.3 -> 143.7 us, and without the prefetch's
//   registers no Frechet variant spills and the P = 16 one runs six
//   wavefronts per SIMD instead of five;
// * s comes from an FP32 estimate of the norm (a few adds and a cross-lane
//   maximum) whenever that estimate decides it exactly; the FP64 sequential
//   column sums of the reference run only near a squaring boundary or for
//   non-finite input;
// * the Frechet half D1.U2 + U1.D2 is one accumulation chain, fed step by
//   step together with the D chain (two independent MFMA chains, and each
//   operand register dies after its step).
// Each FP32 MFMA step equals an fmaf chain over its k terms in ascending
// order, so at P = 16 results differ from the reference's sequential FMA chains
// only through the order of the k terms within a product and that one U chain;
// at P = 32 the bf16 sums round less often (parity is by tolerance; s is
// bit-identical).
#include "fh_kernels.h"

namespace fh {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

template <int P>
struct TileCfg;

template <>
struct TileCfg<16> {
  static constexpr int R = 4;
  using acc_t = v4f;
  __device__ static constexpr int step(int r) { return r; }
  __device__ static __forceinline__ int row0(int lane) { return 4 * (lane >> 4); }
  __device__ static __forceinline__ int col(int lane) { return lane & 15; }
  // VGPR holding this lane's diagonal entry, -1 when it holds none.
  __device__ static __forceinline__ int diag_reg(int lane) { return (lane >> 4) == ((lane & 15) >> 2) ? (lane & 3) : -1; }
  __device__ static __forceinline__ acc_t mfma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

template <>
struct TileCfg<32> {
  static constexpr int R = 16;
  using acc_t = v16f;
  __device__ static constexpr int step(int r) { return 8 * (r >> 2) + (r & 3); }
  __device__ static __forceinline__ int row0(int lane) { return 4 * (lane >> 5); }
  __device__ static __forceinline__ int col(int lane) { return lane & 31; }
  __device__ static __forceinline__ int diag_reg(int lane) {
    const int c = lane & 31;
    return ((c >> 2) & 1) == (lane >> 5) ? 4 * (c >> 3) + (c & 3) : -1;
  }
  __device__ static __forceinline__ acc_t mfma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
  }
};

template <int P>
using Acc = typename TileCfg<P>::acc_t;

// The lane's number, formed anew at each call so that nothing derived from an
// earlier one is kept live: the P = 32 kernels have no registers to spare.
__device__ __forceinline__ int fresh_lane() {
  int lane;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
  return lane;
}

template <int P>
struct Tm {
  float v[TileCfg<P>::R];
};

template <int P, bool Pair>
struct PTm {
  Tm<P> d;
  Tm<P> u;
};

template <int P>
__device__ __forceinline__ Tm<P> from_acc(const Acc<P>& a) {
  Tm<P> m;
#pragma unroll
  for (int r = 0; r < TileCfg<P>::R; ++r) m.v[r] = a[r];
  return m;
}

// (D1, U1).(D2, U2) = (D1.D2, D1.U2 + U1.D2).  Step r feeds all three
// products, so each operand register dies after its step and the D and U
// accumulations alternate as two independent MFMA chains.  WantD = false
// skips the D chain (a last squaring, whose D block nothing reads); the D
// block is then left as x's.
template <int P, bool Pair, bool WantD = true>
__device__ __forceinline__ PTm<P, Pair> pmm(const PTm<P, Pair>& xt, const PTm<P, Pair>& y) {
  Acc<P> d = {}, u = {};
#pragma unroll
  for (int r = 0; r < TileCfg<P>::R; ++r) {
    if constexpr (WantD) d = TileCfg<P>::mfma(xt.d.v[r], y.d.v[r], d);
    if constexpr (Pair) {
      u = TileCfg<P>::mfma(xt.d.v[r], y.u.v[r], u);
      u = TileCfg<P>::mfma(xt.u.v[r], y.d.v[r], u);
    }
  }
  PTm<P, Pair> out;
  if constexpr (WantD) {
    out.d = from_acc<P>(d);
  } else {
    out.d = y.d;
  }
  if constexpr (Pair) out.u = from_acc<P>(u);
  return out;
}

// Compiler ordering of the wavefront's LDS accesses (the hardware already
// performs one wavefront's LDS operations in issue order).
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

template <int P>
__device__ __forceinline__ void tile_write(const Tm<P>& m, float* buf, int lane) {
  using C = TileCfg<P>;
  constexpr int LD = P + 1;
  const int c = C::col(lane);
  const int r0 = C::row0(lane);
#pragma unroll
  for (int r = 0; r < C::R; ++r) buf[(r0 + C::step(r)) * LD + c] = m.v[r];
}
template <int P>
__device__ __forceinline__ Tm<P> tile_read_transposed(const float* buf, int lane) {
  using C = TileCfg<P>;
  constexpr int LD = P + 1;
  const int c = C::col(lane);
  const int r0 = C::row0(lane);
  Tm<P> t;
#pragma unroll
  for (int r = 0; r < C::R; ++r) t.v[r] = buf[c * LD + r0 + C::step(r)];
  return t;
}

// D layout of M -> D layout of M^T.
template <int P>
__device__ __forceinline__ Tm<P> transpose(const Tm<P>& a, float* buf, int lane) {
  tile_write<P>(a, buf, lane);
  lds_order();
  const Tm<P> t = tile_read_transposed<P>(buf, lane);
  lds_order();
  return t;
}
// The same of both halves of a pair in one round.
template <int P, bool Pair>
__device__ __forceinline__ PTm<P, Pair> ptranspose(const PTm<P, Pair>& a, float* buf, int lane) {
  constexpr int T = P * (P + 1);
  tile_write<P>(a.d, buf, lane);
  if constexpr (Pair) tile_write<P>(a.u, buf + T, lane);
  lds_order();
  PTm<P, Pair> t;
  t.d = tile_read_transposed<P>(buf, lane);
  if constexpr (Pair) t.u = tile_read_transposed<P>(buf + T, lane);
  lds_order();
  return t;
}

// ---- P = 32: products on the bf16 matrix instructions ---------------------------
//
// An FP32 value is the exact sum of three bf16 values, v = h + m + l with
// |m| <= 2^-8 |v| and |l| <= 2^-16 |v|, and X.Y is the six products
//   xh.yh + (xm.yh + xh.ym) + (xl.yh + xm.ym + xh.yl)
// (Henry, Tang, Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype
// for Higher-Precision Computations", ARITH 2019; the three left out add up to at
// most 2^-24 |x||y|), summed smallest first in FP32.  Products of bf16 values are
// exact and an instruction sums 16 of them before it rounds, so results of long
// sums are closer to the exact product than the FP32 instructions' chain: over 512
// products of N(0, 1) matrices 3.8e-8 against 1.03e-7 relative error in the 2-norm
// (cutting values instead of rounding them to their parts gave that advantage away
// over a whole exponential); short sums are as close (split_pmm).
//
// Six bf16 instructions take 3/8 of the FP32 ones' cycles; splitting a matrix
// costs 16 conversions, shifts or masks and subtractions a lane and part, so that
// a matrix takes 1412 and 3224 VALU instructions (forward, Frechet) for 593 and 1104
// before, and the matrix pipe is busy 38 and 48% of the time for 75 and 82%.
// 32768 32 x 32 FP16 matrices N(0, 1) / sqrt(32), forward + Frechet: 143 + 478 ->
// 111 + 333 us (328 + 1113 -> 223 + 672 thousand cycles, the chip at 2.0 GHz for
// 2.3, on another box at 1.8); a step over norms of 1.8 decades 581 -> 420 us.  P = 16 keeps the FP32
// instructions: its products are shorter against the splits (a trial: 150 -> 170 us
// over 65536 matrices).
//
// The k index is permuted as for the FP32 instructions: the B operand of Y
// comes from the lane's own D-layout values, eight to a 32x32x16 instruction.
// The A operand is the transposed X: its parts go to LDS column by column (8
// bytes, four rows, to a write) and come back through the transposing read
// ds_read_b64_tr_b16, which hands lane i of a row of 16 element i of each of four
// columns.  So a matrix is split once for both sides.

typedef __bf16 Bf16x8 __attribute__((ext_vector_type(8)));
typedef short Short4 __attribute__((ext_vector_type(4)));
typedef uint32_t U32x2 __attribute__((ext_vector_type(2)));

// Parts of a matrix: w[k][s] holds part k of VGPRs 8s..8s+7, two to a word.  N of
// the three parts are non-zero: BF16 inputs have one, FP16 inputs (11 bits) two.
template <int N>
struct Parts {
  U32x4 w[N][2];
};
template <bool Pair, int N = 3>
struct PParts {
  Parts<N> d, u;
};
template <typename T>
constexpr int kInputParts = T::code == F32::code ? 3 : T::code == F16::code ? 2 : 1;

// (bf16(lo), bf16(hi)) in one word, round to nearest even.
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  typedef float Float2 __attribute__((ext_vector_type(2)));
  typedef __bf16 Bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((Float2{lo, hi}), Bf16x2));
}

template <int N>
__device__ __forceinline__ Parts<N> split(const Tm<32>& m) {
  // The mask in a VGPR: an SGPR operand costs a full-rate instruction 1.5x.
  uint32_t mask;
  asm("v_mov_b32 %0, 0xffff0000" : "=v"(mask));
  Parts<N> p;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float a = m.v[2 * i], b = m.v[2 * i + 1];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const uint32_t w = pack_bf16(a, b);
      p.w[k][i / 4][i % 4] = w;
      a -= __uint_as_float(w << 16);
      b -= __uint_as_float(w & mask);
    }
  }
  return p;
}
template <int N, bool Pair>
__device__ __forceinline__ PParts<Pair, N> psplit(const PTm<32, Pair>& m) {
  PParts<Pair, N> p;
  p.d = split<N>(m.d);
  if constexpr (Pair) p.u = split<N>(m.u);
  return p;
}

// LDS image of one part: column by column, its rows in chunks of four (8 bytes);
// lane group g's VGPRs 4q..4q+3 are chunk 2q + g of its column.  A lane writes the
// chunks of its own column and reads back, per q, the lane's row of four columns.
// Columns are 72 bytes apart: writes are free of bank conflicts, reads all but.
constexpr int kPartPitch = 72;
constexpr int kPartBytes = 32 * kPartPitch;
struct PartLds {
  char *wr, *rd;  // q = 0; 16 and 8 * kPartPitch bytes on per q
  __device__ __forceinline__ PartLds(char* buf, int lane) {
    const int g = lane >> 5, i = lane & 15;
    wr = buf + (lane & 31) * kPartPitch + 8 * g;
    rd = buf + (4 * g + (i >> 2)) * kPartPitch + 8 * ((i & 3) + ((lane & 16) >> 2));
  }
};

// Transposed parts of a left operand, laid out as Parts are.
template <int N>
struct Left {
  Parts<N> p;
  __device__ __forceinline__ void through_lds(const Parts<N>& m, const PartLds& at, int slot) {
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<U32x2*>(at.wr + (3 * slot + k) * kPartBytes + 16 * q) =
            U32x2{m.w[k][q / 2][2 * (q % 2)], m.w[k][q / 2][2 * (q % 2) + 1]};
    lds_order();
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        using LdsShort4 = __attribute__((address_space(3))) Short4;
        const U32x2 t = __builtin_bit_cast(
            U32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                       (LdsShort4*)(at.rd + (3 * slot + k) * kPartBytes + 8 * kPartPitch * q)));
        p.w[k][q / 2][2 * (q % 2)] = t[0];
        p.w[k][q / 2][2 * (q % 2) + 1] = t[1];
      }
  }
};
template <bool Pair, int N>
struct PLeft {
  Left<N> d, u;
};

// Splits m into right operands y and, through LDS, the left ones; the second
// half's split covers the first one's way through LDS.
template <int N, bool Pair>
__device__ __forceinline__ PLeft<Pair, N> to_left(const PTm<32, Pair>& m, PParts<Pair, N>& y, const PartLds& at) {
  PLeft<Pair, N> x;
  y.d = split<N>(m.d);
  x.d.through_lds(y.d, at, 0);
  if constexpr (Pair) {
    y.u = split<N>(m.u);
    x.u.through_lds(y.u, at, 1);
  }
  lds_order();
  return x;
}

// acc + the products of parts i of x and j of y with Lo <= i + j <= Hi, smallest
// first.
template <int Hi, int Lo, int NX, int NY>
__device__ __forceinline__ v16f madd(const Left<NX>& x, const Parts<NY>& y, v16f acc) {
#pragma unroll
  for (int t = Hi; t >= Lo; --t)
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int j = t - i;
      if (j < 0 || j >= NY) continue;
#pragma unroll
      for (int s = 0; s < 2; ++s)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(Bf16x8, x.p.w[i][s]),
                                                      __builtin_bit_cast(Bf16x8, y.w[j][s]), acc, 0, 0, 0);
    }
  return acc;
}

// pmm on the bf16 instructions.  Every chain takes its small products first, so
// that only the last few instructions round at the result's magnitude.
//
// Apart: the leading products h.h and the small ones have an accumulator each.  An
// instruction cuts the smaller of accumulator and products off near the larger
// one's last bit: one product onto an accumulator of its sign errs by up to 1 ulp
// and by -0.17 ulp on average, onto zero by half an ulp at most (measured).  Apart,
// short sums gain that and long ones pay for a third rounding.  So the powers of A
// and the squarings, whose errors add up or double, are formed apart in FP32, and
// the polynomial's last two products, to which a sum is added, are not.  Mean error
// against FP64 relative to the FP32 instructions' chains, 2048 matrices, n = 32,
// entries N(0, 100) on the diagonal / in 2 x 2 blocks / N(0, 100 / n) everywhere:
// 1.25 / 1.13 / 0.64 with no product apart, 1.02 / 0.99 / 0.65 so, 1.01 / 0.97 / 0.68
// with all.  With the operands' scale, 32768 matrices forward + Frechet 135 + 370 ->
// 141 + 384 us.  Results in 16 bits, rounded 2^13 times coarser, go without.
template <bool Pair, bool Apart, bool WantD = true, int NX, int NY>
__device__ __forceinline__ PTm<32, Pair> split_pmm(const PLeft<Pair, NX>& x, const PParts<Pair, NY>& y) {
  v16f d = {}, u = {};
  if constexpr (WantD) d = madd<2, 1>(x.d, y.d, d);
  if constexpr (Pair) {
    u = madd<2, 1>(x.d, y.u, u);
    u = madd<2, 1>(x.u, y.d, u);
  }
  v16f dh = {}, uh = {};
  if constexpr (WantD) dh = madd<0, 0>(x.d, y.d, Apart ? dh : d);
  if constexpr (Pair) {
    uh = madd<0, 0>(x.d, y.u, Apart ? uh : u);
    uh = madd<0, 0>(x.u, y.d, uh);
  }
  if constexpr (Apart) {
    if constexpr (WantD) dh += d;
    if constexpr (Pair) uh += u;
  }
  PTm<32, Pair> out;
  out.d = from_acc<32>(dh);
  if constexpr (Pair) out.u = from_acc<32>(uh);
  return out;
}
template <typename T>
constexpr bool kApart = T::code == F32::code;

// bf16 MFMAs read subnormal operands as zero, and the low part of a value below
// 2^-103 may be one.  So every operand of a product is 2^24 times its matrix or
// more: its parts are multiples of 2^24 * 2^-149, all normal, and the products
// and sums of values that FP32 holds at all are normal as well.  The scales are
// powers of two: they go into the factor 2^-s of the input and into the
// polynomial's coefficients and cost a multiply per entry only of A^3 and of a
// result.  kScale[k] are the exponents of I, A, A^2, A^3 and A^6, kOperandScale
// those of the operands B1, B5 and exp.
constexpr int kOperandScale = 24;
constexpr int kScale[5] = {0, kOperandScale, 2 * kOperandScale, 32, 64};

__device__ constexpr float pow2(int e) { return e < 0 ? 0.5f * pow2(e + 1) : e > 0 ? 2.f * pow2(e - 1) : 1.f; }

// m * 2^e, of a pair U alone when nothing reads D.
template <bool Pair, bool WantD = true>
__device__ __forceinline__ void rescale(PTm<32, Pair>& m, int e) {
  float factor = __builtin_ldexpf(1.f, e);
  asm("" : "+v"(factor));  // a VGPR: an SGPR operand costs a full-rate instruction 1.5x
#pragma unroll
  for (int r = 0; r < TileCfg<32>::R; ++r) {
    if constexpr (WantD) m.d.v[r] *= factor;
    if constexpr (Pair) m.u.v[r] *= factor;
  }
}

// Whether squaring the scaled `m` keeps every partial product and sum finite (64
// terms below 2^120); otherwise a low part's product could overflow to the
// opposite infinity and make NaN of a result that is infinite.
template <bool Pair>
__device__ __forceinline__ bool squares_in_range(const PTm<32, Pair>& m) {
  float top = 0.f;
#pragma unroll
  for (int r = 0; r < TileCfg<32>::R; ++r) {
    top = __builtin_fmaxf(top, __builtin_fabsf(m.d.v[r]));
    if constexpr (Pair) top = __builtin_fmaxf(top, __builtin_fabsf(m.u.v[r]));
  }
  return __builtin_amdgcn_ballot_w64(!(top < 0x1p60f)) == 0;
}

// The polynomial has norm at most exp(theta18) = e^3.01 and i squarings raise
// that to exp(theta18 2^i): four rounds (operands to e^24, results to e^48, 2^118
// with the scale of both sides) need no check.
constexpr int kUncheckedSquarings = 4;

// c0*I in the D layout for the two combines with an identity term (B3 and B4,
// reference csrc/MatrixExpSmall.cuh:268-281), from `dreg`, the VGPR of this
// lane's diagonal entry (-1 for none).  P = 16 keeps these 2R values in
// registers for the whole kernel (it has registers to spare); P = 32 selects
// them where they are used.
struct Ident16 {
  Tm<16> b3, b4;
  __device__ __forceinline__ explicit Ident16(int dreg) {
#pragma unroll
    for (int r = 0; r < TileCfg<16>::R; ++r) {
      b3.v[r] = dreg == r ? kCoef[2][0] : 0.f;
      b4.v[r] = dreg == r ? kCoef[3][0] : 0.f;
    }
  }
  __device__ __forceinline__ float value(int k, int r) const { return k == 2 ? b3.v[r] : b4.v[r]; }
};
// The same scaled by 2^Out.
template <int Out>
struct Ident32 {
  static constexpr float kB3 = kCoef[2][0] * pow2(Out), kB4 = kCoef[3][0] * pow2(Out);
  int dreg;
  __device__ __forceinline__ float value(int k, int r) const { return dreg == r ? (k == 2 ? kB3 : kB4) : 0.f; }
};

// B(K+1) = c0*I + c1*A + c2*A^2 + c3*A^3 + c6*A^6 (reference
// csrc/MatrixExpSmall.cuh:268-281), the contracted chain with zero
// coefficients skipped; the identity term (D only) comes from `id`.  At P = 32
// the powers are scaled by 2^kScale and B by 2^Out.
template <int K, int Out = 0, int P, bool Pair, typename Id>
__device__ __forceinline__ PTm<P, Pair> combine(const PTm<P, Pair>& a, const PTm<P, Pair>& a2,
                                                const PTm<P, Pair>& a3, const PTm<P, Pair>& a6, const Id& id) {
  using C = TileCfg<P>;
  const auto scale = [](int k) constexpr { return P == 32 ? pow2(Out - kScale[k]) : 1.f; };
  constexpr float c0 = kCoef[K][0], c1 = kCoef[K][1] * scale(1), c2 = kCoef[K][2] * scale(2),
                  c3 = kCoef[K][3] * scale(3), c6 = kCoef[K][4] * scale(4);
  static_assert(c0 == 0.f || K == 2 || K == 3, "identity terms are B3 and B4");
  PTm<P, Pair> b;
#pragma unroll
  for (int r = 0; r < C::R; ++r) {
    float t = 0.f;
    if constexpr (c0 != 0.f) t = id.value(K, r);
    if constexpr (c1 != 0.f) t = __builtin_fmaf(c1, a.d.v[r], t);
    t = __builtin_fmaf(c2, a2.d.v[r], t);
    t = __builtin_fmaf(c3, a3.d.v[r], t);
    if constexpr (c6 != 0.f) t = __builtin_fmaf(c6, a6.d.v[r], t);
    b.d.v[r] = t;
    if constexpr (Pair) {
      float w = 0.f;
      if constexpr (c1 != 0.f) w = __builtin_fmaf(c1, a.u.v[r], w);
      w = __builtin_fmaf(c2, a2.u.v[r], w);
      w = __builtin_fmaf(c3, a3.u.v[r], w);
      if constexpr (c6 != 0.f) w = __builtin_fmaf(c6, a6.u.v[r], w);
      b.u.v[r] = w;
    }
  }
  return b;
}

template <int P, bool Pair>
__device__ __forceinline__ PTm<P, Pair> padd(const PTm<P, Pair>& x, const PTm<P, Pair>& y) {
  PTm<P, Pair> z;
#pragma unroll
  for (int r = 0; r < TileCfg<P>::R; ++r) {
    z.d.v[r] = x.d.v[r] + y.d.v[r];
    if constexpr (Pair) z.u.v[r] = x.u.v[r] + y.u.v[r];
  }
  return z;
}

// Layout classes for loading: rows contiguous (kLoadRows) loads the D layout
// of the matrix itself; columns contiguous (kLoadCols) loads the D layout of
// its transpose.  Either works for any strides; the class only decides which
// of the two layouts comes from memory and which from the LDS transpose.
constexpr int kLoadRows = 0;
constexpr int kLoadCols = 1;

// Byte addressing of one operand in the D layout of the loaded matrix: the
// matrix base goes into the descriptor, `lane_off` is this lane's offset for
// VGPR 0 and step(r) * `major` the uniform offset of VGPR r; `major` is the
// elements per D-layout row step, given by the caller (op.sc or op.sr).
struct TileSrc {
  const char* data;
  int64_t sb;        // bytes per batch step
  int32_t major;     // bytes per D-layout row step
  int32_t lane_off;  // bytes, VGPR 0 of this lane
  uint32_t records;  // footprint of one matrix in bytes
};

template <typename T, int P>
__device__ __forceinline__ TileSrc make_src(const Operand& op, int layout, int64_t major, int n, int lane) {
  using C = TileCfg<P>;
  constexpr int es = ElemIO<T>::bytes;
  const int64_t minor = layout == kLoadCols ? op.sr : op.sc;
  TileSrc s;
  s.data = static_cast<const char*>(op.data);
  s.sb = op.sb * es;
  s.major = static_cast<int32_t>(major * es);
  s.lane_off = static_cast<int32_t>((C::row0(lane) * major + C::col(lane) * minor) * es);
  s.records = static_cast<uint32_t>(((n - 1) * (op.sr + op.sc) + 1) * es);
  return s;
}

template <typename T, int P>
struct RawTile {
  typename ElemIO<T>::raw_t v[TileCfg<P>::R];
};

// Storage bits of matrix b; entries outside the n x n block read as +0.
template <typename T, int P, bool Full>
__device__ __forceinline__ RawTile<T, P> load_raw(const TileSrc& s, int64_t b, int n, int lane) {
  using C = TileCfg<P>;
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(s.data + b * s.sb, s.records);
  RawTile<T, P> t;
  if constexpr (Full) {
#pragma unroll
    for (int r = 0; r < C::R; ++r) t.v[r] = ElemIO<T>::load(rs, s.lane_off, C::step(r) * s.major);
  } else {
    const bool col_ok = C::col(lane) < n;
#pragma unroll
    for (int r = 0; r < C::R; ++r) {
      const bool ok = col_ok && C::row0(lane) + C::step(r) < n;
      t.v[r] = ElemIO<T>::load(rs, ok ? s.lane_off + C::step(r) * s.major : kOutOfRange, 0);
    }
  }
  return t;
}

template <typename T, int P>
__device__ __forceinline__ Tm<P> to_tile(const RawTile<T, P>& raw) {
  Tm<P> m;
#pragma unroll
  for (int r = 0; r < TileCfg<P>::R; ++r) m.v[r] = ElemIO<T>::value(raw.v[r]);
  return m;
}

// Contiguous [batch, n, n] output in the input dtype.
template <typename T, int P, bool Full>
__device__ __forceinline__ void store_tile(void* out, int64_t b, int n, int lane, const Tm<P>& m) {
  using C = TileCfg<P>;
  constexpr int es = ElemIO<T>::bytes;
  const int64_t nn = static_cast<int64_t>(n) * n;
  const __amdgpu_buffer_rsrc_t rs =
      make_rsrc(static_cast<char*>(out) + b * nn * es, static_cast<uint32_t>(nn * es));
  const int32_t lane_off = (C::row0(lane) * n + C::col(lane)) * es;
  if constexpr (Full) {
#pragma unroll
    for (int r = 0; r < C::R; ++r) ElemIO<T>::template store<kNontemporal>(m.v[r], rs, lane_off, C::step(r) * P * es);
  } else {
    const bool col_ok = C::col(lane) < n;
#pragma unroll
    for (int r = 0; r < C::R; ++r) {
      const bool ok = col_ok && C::row0(lane) + C::step(r) < n;
      ElemIO<T>::template store<kNontemporal>(m.v[r], rs, ok ? lane_off + C::step(r) * n * es : kOutOfRange, 0);
    }
  }
}

// Maximum over the lanes of a row of 16 (every lane of the row gets it).
__device__ __forceinline__ uint32_t row_max_u32(uint32_t v) {
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0xB1, 0xF, 0xF, false)));
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x4E, 0xF, 0xF, false)));
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x141, 0xF, 0xF, false)));
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x140, 0xF, 0xF, false)));
  return v;
}

// FP32 estimate of the 1-norm max_j sum_i |A[i][j]| (+ |G[i][j]|) from the D
// layout of A (and G): each lane sums its column entries, the lanes sharing a
// column add up, and the column maximum is taken on the bit patterns (equal
// order for non-negative floats; NaN and inf compare above every finite
// value).  Relative error at most (2R + 2) * 2^-24 < 2^-18.
template <int P, bool Pair>
__device__ __forceinline__ float norm_estimate(const PTm<P, Pair>& a) {
  float p = 0.f;
#pragma unroll
  for (int r = 0; r < TileCfg<P>::R; ++r) {
    p += __builtin_fabsf(a.d.v[r]);
    if constexpr (Pair) p += __builtin_fabsf(a.u.v[r]);
  }
  // Rows of 16 (P = 16) and halves of 32 exchanged in registers.
  const uint32_t w = __float_as_uint(p);
  if constexpr (P == 16) {
    const auto rows = __builtin_amdgcn_permlane16_swap(w, w, false, false);
    p = __uint_as_float(rows[0]) + __uint_as_float(rows[1]);
  }
  const uint32_t v = __float_as_uint(p);
  const auto halves = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  p = __uint_as_float(halves[0]) + __uint_as_float(halves[1]);
  uint32_t m = row_max_u32(__float_as_uint(p) & 0x7FFFFFFFu);
  uint32_t top = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(m), 0));
  if constexpr (P == 32) top = max(top, static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(m), 16)));
  return __uint_as_float(top);
}

// The reference's FP64 norm (csrc/MatrixExpSmall.cuh:343-357): per column the
// rows summed sequentially, |A| then |G| per row, then the column maximum; the
// total of the column sums is finite exactly when every entry is (non-finite
// rule, :318-331), i.e. when every column sum is.  Returns false for
// non-finite input.  This path is rare, so it is written for few live
// registers: the row loop is not unrolled, and the maximum over columns reads
// each lane's sum into scalar registers (the order of a maximum is free).
template <int P, bool Pair>
__device__ __forceinline__ bool exact_squarings(const PTm<P, Pair>& a, float* buf, int lane, int& s) {
  constexpr int LD = P + 1;
  tile_write<P>(a.d, buf, lane);
  if constexpr (Pair) tile_write<P>(a.u, buf + P * LD, lane);
  lds_order();
  double v = 0.;
  if (lane < P) {
#pragma unroll 1
    for (int row = 0; row < P; ++row) {
      v += fabs(static_cast<double>(buf[row * LD + lane]));
      if constexpr (Pair) v += fabs(static_cast<double>(buf[P * LD + row * LD + lane]));
    }
  }
  lds_order();
  if (__builtin_amdgcn_ballot_w64(!__builtin_isfinite(v)) != 0) return false;
  double norm = 0.;
  const uint64_t bits = __builtin_bit_cast(uint64_t, v);
  const int vlo = static_cast<int>(bits), vhi = static_cast<int>(bits >> 32);
#pragma unroll 1
  for (int j = 0; j < P; ++j) {
    const uint64_t w = static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(vlo, j))) |
                       (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(vhi, j))) << 32);
    norm = fmax(norm, __builtin_bit_cast(double, w));
  }
  s = squarings_from_norm(norm);
  return true;
}

// Occupancy target (wavefronts per SIMD) the register allocation must meet.
template <int P, bool Pair>
constexpr int kTileWaves() {
  return P == 16 ? 4 : (Pair ? 2 : 3);
}

// LDS of a workgroup; P = 32 uses it for the FP32 transposes and the bf16 parts in
// turn.
template <int P, bool Pair>
constexpr int kTileLds = (Pair ? 2 : 1) * (P == 32 ? 3 * kPartBytes : 4 * P * (P + 1));
static_assert(3 * kPartBytes >= 4 * 32 * 33);

// Degree-18 polynomial (csrc/MatrixExpSmall.cuh:83-106): A^2 = A.A,
// A^3 = A.A^2, A^6 = A^3.A^3, A9 = B1.B5 + B4, T = B2 + (B3 + A9).A9.
// The sums B1.B5 + B4, B3 + A9 and B2 + (..).A9 are formed after their
// products, as in the reference: starting the MFMA accumulations from B4
// and B2 instead raised the FP32 error 1.4-fold on average (measured over
// 32768 32 x 32 matrices against the FP64 result and the reference's own
// arithmetic).
//
// P = 16, on the FP32 instructions; `at` is a's transpose.
template <bool Pair>
__device__ __forceinline__ PTm<16, Pair> polynomial(const PTm<16, Pair>& a, const PTm<16, Pair>& at, const Ident16& id,
                                                    float* buf, int lane) {
  const PTm<16, Pair> a2 = pmm<16, Pair>(at, a);
  const PTm<16, Pair> a3 = pmm<16, Pair>(at, a2);
  const PTm<16, Pair> a6 = pmm<16, Pair>(ptranspose<16, Pair>(a3, buf, lane), a3);
  const PTm<16, Pair> b1t = ptranspose<16, Pair>(combine<0>(a, a2, a3, a6, id), buf, lane);
  const PTm<16, Pair> b5 = combine<4>(a, a2, a3, a6, id);
  const PTm<16, Pair> b1b5 = pmm<16, Pair>(b1t, b5);
  const PTm<16, Pair> a9 = padd<16, Pair>(b1b5, combine<3>(a, a2, a3, a6, id));
  const PTm<16, Pair> lhst = ptranspose<16, Pair>(padd<16, Pair>(combine<2>(a, a2, a3, a6, id), a9), buf, lane);
  const PTm<16, Pair> b2 = combine<1>(a, a2, a3, a6, id);
  return padd<16, Pair>(b2, pmm<16, Pair>(lhst, a9));
}

// P = 32, on the bf16 instructions, for inputs of N parts: from 2^24 A to 2^96 T.
constexpr int kPolynomialScale = 4 * kOperandScale;
template <int N, bool Apart, bool Pair>
__device__ __forceinline__ PTm<32, Pair> split_polynomial(const PTm<32, Pair>& a, int dreg, const PartLds& at) {
  constexpr int kB = kOperandScale;  // B1 and B5; twice that B1.B5, B3 and B4
  const Ident32<2 * kB> id{dreg};
  PParts<Pair, N> ya;
  const PLeft<Pair, N> xa = to_left<N, Pair>(a, ya, at);
  const PTm<32, Pair> a2 = split_pmm<Pair, Apart>(xa, ya);
  PTm<32, Pair> a3 = split_pmm<Pair, Apart>(xa, psplit<3, Pair>(a2));
  rescale<Pair>(a3, kScale[3] - kScale[1] - kScale[2]);
  PParts<Pair> y3, unused;
  const PLeft<Pair, 3> x3 = to_left<3, Pair>(a3, y3, at);
  const PTm<32, Pair> a6 = split_pmm<Pair, Apart>(x3, y3);
  const PLeft<Pair, 3> x1 = to_left<3, Pair>(combine<0, kB>(a, a2, a3, a6, id), unused, at);
  const PParts<Pair> y5 = psplit<3, Pair>(combine<4, kB>(a, a2, a3, a6, id));
  const PTm<32, Pair> b4 = combine<3, 2 * kB>(a, a2, a3, a6, id);
  const PTm<32, Pair> b3 = combine<2, 2 * kB>(a, a2, a3, a6, id);
  const PTm<32, Pair> b2 = combine<1, kPolynomialScale>(a, a2, a3, a6, id);
  const PTm<32, Pair> a9 = padd<32, Pair>(split_pmm<Pair, false>(x1, y5), b4);
  const PLeft<Pair, 3> x9 = to_left<3, Pair>(padd<32, Pair>(b3, a9), unused, at);
  return padd<32, Pair>(b2, split_pmm<Pair, false>(x9, psplit<3, Pair>(a9)));
}

template <typename T, int P, bool Pair, int XL, int GL, bool Full>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kTileWaves<P, Pair>(), 8))) void expm_tile_kernel(
    ExpmArgs args) {
  using C = TileCfg<P>;
  constexpr int R = C::R;
  __shared__ __attribute__((aligned(16))) char lds[kTileLds<P, Pair>];
  float* const buf = reinterpret_cast<float*>(lds);
  const int thread = threadIdx.x;
  const int n = Full ? P : args.n;

  int64_t b = blockIdx.x;
  Ident16 id(P == 16 ? C::diag_reg(thread) : -1);
  if constexpr (P == 16) {
#pragma unroll
    for (int r = 0; r < R; ++r) asm volatile("" : "+v"(id.b3.v[r]), "+v"(id.b4.v[r]));
  }
  for (; b < args.batch; b += gridDim.x) {
    // P = 32 derives everything that depends on the lane or the strides afresh
    // for each matrix and for its store, so that offsets, bounds predicates and
    // identity terms are not kept live across the products: registers these
    // kernels do not have, on a grid where a wavefront seldom sees a second
    // matrix.  P = 16 keeps them.
    int lane = P == 32 ? fresh_lane() : thread;
    int64_t major_x = XL == kLoadCols ? args.x.sc : args.x.sr, major_g = GL == kLoadCols ? args.g.sc : args.g.sr;
    if constexpr (P == 32) asm volatile("" : "+s"(major_x), "+s"(major_g));
    const TileSrc sx = make_src<T, P>(args.x, XL, major_x, n, lane);
    const TileSrc sg = make_src<T, P>(args.g, GL, major_g, n, lane);
    const Tm<P> lx = to_tile<T, P>(load_raw<T, P, Full>(sx, b, n, lane));
    Tm<P> lg;
    if constexpr (Pair) lg = to_tile<T, P>(load_raw<T, P, Full>(sg, b, n, lane));

    // The D layout of X and G and, for P = 16, of their transposes: the loaded
    // one and its LDS transpose.
    PTm<P, Pair> a, at;
    if constexpr (P == 16) {
      PTm<P, Pair> loaded;
      loaded.d = lx;
      if constexpr (Pair) loaded.u = lg;
      const PTm<P, Pair> other = ptranspose<P, Pair>(loaded, buf, lane);
      a.d = XL == kLoadCols ? other.d : lx;
      at.d = XL == kLoadCols ? lx : other.d;
      if constexpr (Pair) {
        a.u = GL == kLoadCols ? other.u : lg;
        at.u = GL == kLoadCols ? lg : other.u;
      }
    } else {
      a.d = XL == kLoadCols ? transpose<P>(lx, buf, lane) : lx;
      if constexpr (Pair) a.u = GL == kLoadCols ? transpose<P>(lg, buf, lane) : lg;
    }

    int s;
    if (!squarings_from_estimate(norm_estimate<P, Pair>(a), s) && !exact_squarings<P, Pair>(a, buf, lane, s)) {
      // Non-finite entry: the whole matrix is NaN (csrc/MatrixExpSmall.cuh:318-331).
      Tm<P> nan;
#pragma unroll
      for (int r = 0; r < R; ++r) nan.v[r] = __builtin_nanf("");
      store_tile<T, P, Full>(args.out, b, n, lane, nan);
      if (lane == 0 && args.s_out) args.s_out[b] = -1;
      continue;
    }
    s = __builtin_amdgcn_readfirstlane(s);

    // Scale by 2^-s (csrc/MatrixExpSmall.cuh:362-367), the views' lazy
    // negation and the scale of P = 32's operands folded into the same exact
    // multiply.
    const float scale = __builtin_ldexpf(1.f, (P == 32 ? kOperandScale : 0) - s);
    const float scale_x = scale * args.x.sign;
    const float scale_g = scale * args.g.sign;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      a.d.v[r] *= scale_x;
      if constexpr (Pair) a.u.v[r] *= scale_g;
      if constexpr (P == 16) {
        at.d.v[r] *= scale_x;
        if constexpr (Pair) at.u.v[r] *= scale_g;
      }
    }

    // The last squaring of a pair forms only the U block (the output).
    PTm<P, Pair> res;
    if constexpr (P == 16) {
      res = polynomial<Pair>(a, at, id, buf, lane);
      for (int i = Pair ? 1 : 0; i < s; ++i) res = pmm<P, Pair>(ptranspose<P, Pair>(res, buf, lane), res);
      if (Pair && s > 0) res = pmm<P, Pair, !Pair>(ptranspose<P, Pair>(res, buf, lane), res);
    } else {
      const PartLds part_lds(lds, lane);
      res = split_polynomial<kInputParts<T>, kApart<T>>(a, C::diag_reg(lane), part_lds);
      int scale = s > 0 ? kOperandScale : 0;  // of res, as a power of two
      rescale<Pair>(res, scale - kPolynomialScale);
      int i = 0;
      for (; i < s; ++i) {
        if (i >= kUncheckedSquarings && !squares_in_range<Pair>(res)) break;
        PParts<Pair> y;
        const PLeft<Pair, 3> x = to_left<3, Pair>(res, y, part_lds);
        const int twice = 2 * scale;
        scale = i == s - 1 ? 0 : kOperandScale;
        if (Pair && i == s - 1) {
          res = split_pmm<Pair, kApart<T>, !Pair>(x, y);
          rescale<Pair, !Pair>(res, -twice);
        } else {
          res = split_pmm<Pair, kApart<T>>(x, y);
          // Two squarings of the polynomial, to e^12, fit without a rescaling between them.
          if (i == 0 && s > 1) {
            scale = twice;
          } else {
            rescale<Pair>(res, scale - twice);
          }
        }
      }
      if (i < s) {
        rescale<Pair>(res, -kOperandScale);
        for (; i < (Pair ? s - 1 : s); ++i) res = pmm<P, Pair>(ptranspose<P, Pair>(res, buf, fresh_lane()), res);
        if (Pair) res = pmm<P, Pair, !Pair>(ptranspose<P, Pair>(res, buf, fresh_lane()), res);
      }
      lane = fresh_lane();
    }

    store_tile<T, P, Full>(args.out, b, n, lane, Pair ? res.u : res.d);
    if (lane == 0 && args.s_out) args.s_out[b] = s;
  }
}

template <typename T, int P, bool Pair, int XL, int GL, bool Full>
hipError_t launch_tile_l(const ExpmArgs& args, hipStream_t stream) {
  // P = 32: one matrix per wavefront (up to 2^24 workgroups, beyond which
  // wavefronts walk the batch with a grid stride), the hardware starting a
  // workgroup as another retires.  P = 16: four times the resident workgroups,
  // each walking two or three matrices, which spreads the per-wavefront setup
  // (C4 step 158.1 -> 155.0 and 159.2 -> 154.9 us against one matrix per
  // wavefront; 2x, 8x and 16x resident measured slower; P = 32 at 2x and 4x
  // slower than one per wavefront).
  static const int64_t resident =
      resident_blocks(reinterpret_cast<const void*>(&expm_tile_kernel<T, P, Pair, XL, GL, Full>), 64);
  const int64_t cap = P == 16 ? 4 * resident : int64_t{1} << 24;
  const int64_t grid = args.batch < cap ? args.batch : cap;
  hipLaunchKernelGGL((expm_tile_kernel<T, P, Pair, XL, GL, Full>), dim3(static_cast<unsigned>(grid)), dim3(64), 0,
                     stream, args);
  return hipGetLastError();
}

int load_class(const Operand& op) { return (op.sr == 1 && op.sc != 1) ? kLoadCols : kLoadRows; }

template <typename T, int P, bool Pair, bool Full>
hipError_t launch_tile_f(const ExpmArgs& args, hipStream_t stream) {
  const int xl = load_class(args.x);
  if constexpr (Pair) {
    const int gl = load_class(args.g);
    if (xl == kLoadRows) {
      return gl == kLoadRows ? launch_tile_l<T, P, Pair, kLoadRows, kLoadRows, Full>(args, stream)
                             : launch_tile_l<T, P, Pair, kLoadRows, kLoadCols, Full>(args, stream);
    }
    return gl == kLoadRows ? launch_tile_l<T, P, Pair, kLoadCols, kLoadRows, Full>(args, stream)
                           : launch_tile_l<T, P, Pair, kLoadCols, kLoadCols, Full>(args, stream);
  } else {
    return xl == kLoadRows ? launch_tile_l<T, P, Pair, kLoadRows, kLoadRows, Full>(args, stream)
                           : launch_tile_l<T, P, Pair, kLoadCols, kLoadRows, Full>(args, stream);
  }
}

template <typename T, int P, bool Pair>
hipError_t launch_tile_tp(const ExpmArgs& args, hipStream_t stream) {
  return args.n == P ? launch_tile_f<T, P, Pair, true>(args, stream) : launch_tile_f<T, P, Pair, false>(args, stream);
}

template <typename T, bool Pair>
hipError_t launch_tile_t(const ExpmArgs& args, int P, hipStream_t stream) {
  return P == 16 ? launch_tile_tp<T, 16, Pair>(args, stream) : launch_tile_tp<T, 32, Pair>(args, stream);
}

// Buffer addressing needs non-negative in-matrix strides and a per-matrix
// footprint below 2^31 bytes.
bool addressable(const Operand& op, int n, int es) {
  if (op.sr < 0 || op.sc < 0) return false;
  const int64_t limit = (int64_t{1} << 31) / es;
  if (op.sr >= limit || op.sc >= limit) return false;
  return (n - 1) * (op.sr + op.sc) + 1 < limit;
}

}  // namespace

hipError_t launch_tile(const ExpmArgs& args, int dtype, int P, bool pair, hipStream_t stream) {
  const int es = dtype == F32::code ? 4 : 2;
  if (!addressable(args.x, args.n, es) || (pair && !addressable(args.g, args.n, es)))
    return launch_generic(args, dtype, P, pair, stream);
  if (dtype == F32::code) return pair ? launch_tile_t<F32, true>(args, P, stream) : launch_tile_t<F32, false>(args, P, stream);
  if (dtype == BF16::code) return pair ? launch_tile_t<BF16, true>(args, P, stream) : launch_tile_t<BF16, false>(args, P, stream);
  return pair ? launch_tile_t<F16, true>(args, P, stream) : launch_tile_t<F16, false>(args, P, stream);
}

}  // namespace fh
