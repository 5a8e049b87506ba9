// Hyper-connection stream mixing with the exponential fused in:
//   forward   Y_b = exp(H_b) X_b                         H [B, n, n], X [B, n, C]
//   backward  dX_b = exp(H_b)^T dY_b,
//             dE_b = dY_b X_b^T,  dH_b = L(H_b^T, dE_b)   (the gradient of exp)
// for n = 2..4 residual streams and any width C.  Nothing of the reference
// fuses this; its matrix_exp (ops/matrix_exp/__init__.py:80-97) returns
// exp(H) to the caller, who multiplies.  Here exp(H_b) never leaves the chip:
//
// * A workgroup of four wavefronts takes a set of T tokens spread over the
//   batch: set k of S = ceil(B / T) holds tokens k, k + S, k + 2S, ..., so
//   workgroups running at the same time stream neighbouring tokens and the rows
//   in flight form one contiguous region of HBM (consecutive tokens per
//   workgroup put every concurrent access T tokens apart, a power-of-two stride
//   that costs about 15% of the bandwidth).  T follows the batch (launch_sets):
//   8 to 64 when there are tokens enough to fill the chip that way, down to one
//   token a workgroup.  One wavefront to 8 tokens, however few there were, left
//   most of the chip idle below 16384 tokens: 64 x 4 x 4096 BF16 forward 61 ->
//   6.3 us, 2048 x 4 x 4096 forward 80 -> 27 us and backward 132 -> 47 us,
//   2048 x 8 x 4096 forward 162 -> 50 us and backward 289 -> 79 us.
// * The wavefronts split each token's columns between them, 64 lanes' chunks in
//   turn (column_parts), so that one token already keeps four wavefronts
//   streaming.  The split depends on C alone, so a token's results do not
//   depend on the batch.
// * Lane l of a wavefront computes exp(H) of its l-th token with the
//   per-lane P == 4 code (p4_lane.h, the same arithmetic as the
//   matrix-exponential kernel, so E is bit-identical to it) and parks it in the
//   wavefront's own LDS.
// * A wavefront then streams its columns of each token: every lane loads 16
//   bytes of each of the n rows per chunk (the whole wavefront covers 1 KB of
//   each row per chunk, coalesced), multiplies by E read back from LDS (one
//   broadcast read per token) and stores 16 bytes of each output row.  Rows
//   are read and written once, with the nontemporal cache hint.  Rows
//   are addressed through a buffer resource rebased per token in SGPRs, so no
//   VALU address arithmetic is needed and offsets never exceed one token.
// * The backward accumulates dE_b = dY_b X_b^T per lane over its columns (in
//   column order), reduces the 16 partial sums across the wavefront with a
//   fixed exchange tree, adds the wavefronts' parts in order through LDS (the
//   result does not depend on anything but the data), and after the set's
//   tokens each lane of one wavefront runs the P == 4 Frechet polynomial on
//   (H^T, dE) of one token -- the same arithmetic as the Frechet kernel.
//
// Both directions are bound by HBM traffic (16 FMAs per 2n elements moved
// forward, 32 per 3n backward); the exponential and Frechet work per token is
// small beside C >= a few hundred columns.
#include <type_traits>

#include "fh_plan.h"
#include "p4_lane.h"

namespace fh {
namespace {

using namespace p4;

constexpr int kWaves = 4;    // wavefronts per workgroup
constexpr int kTokens = 16;  // tokens per wavefront, at most; per workgroup where its wavefronts share them
constexpr int kWideTokens = 8;  // the same at n = 5..8, where a set has no exponential to share

struct HcArgs {
  Operand h;        // [B, n, n]
  const void* x;    // [B, n, C], unit column stride
  int64_t xb, xr;   // element strides of X (token, row)
  const void* gy;   // backward: dY [B, n, C], unit column stride
  int64_t gb, gr;
  void* out;        // forward: Y, backward: dX; contiguous [B, n, C]
  void* dh;         // backward: dH, contiguous [B, n, n]
  float* aux;       // optional FP32 [B, n, n]: exp(H) (forward) or dE (backward)
  int64_t batch;
  int64_t cols;
  int64_t sets;     // workgroups
  int tokens;       // per workgroup
  int parts;        // wavefronts that share a token's columns (column_parts)
  int n;
};

// Buffer resource over `bytes` bytes at `base` + `offset_elems` elements (uniform).
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rebased(const void* base, int64_t offset_elems, int64_t bytes) {
  const char* p = static_cast<const char*>(base) + offset_elems * static_cast<int64_t>(sizeof(typename T::storage));
  return make_rsrc(p, static_cast<uint32_t>(bytes));
}

// 16 bytes of storage as FP32 values (4 for FP32, 8 for FP16/BF16).
template <typename T>
struct Vec {
  static constexpr int V = 16 / static_cast<int>(sizeof(typename T::storage));
  float f[V];
};

template <typename T>
__device__ __forceinline__ Vec<T> unpack(U32x4 w) {
  using S = typename T::storage;
  Vec<T> r;
#pragma unroll
  for (int i = 0; i < Vec<T>::V; ++i) {
    if constexpr (sizeof(S) == 4) {
      r.f[i] = __uint_as_float(w[i]);
    } else {
      const uint16_t h = static_cast<uint16_t>(w[i >> 1] >> (16 * (i & 1)));
      r.f[i] = to_f32<T>(__builtin_bit_cast(S, h));
    }
  }
  return r;
}

template <typename T>
__device__ __forceinline__ U32x4 pack(const Vec<T>& v) {
  using S = typename T::storage;
  U32x4 w;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (sizeof(S) == 4) {
      w[i] = __float_as_uint(v.f[i]);
    } else {
      w[i] = static_cast<uint32_t>(__builtin_bit_cast(uint16_t, from_f32<T>(v.f[2 * i]))) |
             (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, from_f32<T>(v.f[2 * i + 1]))) << 16);
    }
  }
  return w;
}

// Stream rows with the nontemporal hint (cache-policy bit 1: "nt" on gfx950).
constexpr int kStreamPolicy = 2;

// A lane's column in `voff`, the row in `soff`, a scalar register: no VALU work a
// row (forming (row, column) offsets per token cost the backward at n = 8 and 64
// BF16 columns 8%), and neither overflows for lanes past the row's end either (a
// token spans less than 2^31 bytes, in n >= 2 rows).
__device__ __forceinline__ U32x4 load16(__amdgpu_buffer_rsrc_t rs, int32_t voff, int32_t soff) {
  return __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, kStreamPolicy);
}

// The row in the vector offset as well: a wide store needs a scalar offset of 0
// (kStoreSOffset).  A resource a row instead measured 9 to 17% faster at 64 to 256
// BF16 columns, but 2 to 4% slower at 2048 to 8192.
__device__ __forceinline__ void store16(U32x4 w, __amdgpu_buffer_rsrc_t rs, int32_t voff, int32_t row) {
  const uint32_t at = static_cast<uint32_t>(voff) + static_cast<uint32_t>(row);
  __builtin_amdgcn_raw_buffer_store_b128(w, rs, static_cast<int32_t>(at), kStoreSOffset, kStreamPolicy);
}

// One lane's vector of a row of which `left` elements remain.  Ragged: rows in
// whole dwords at any dword (a multi-dword buffer access needs no more), the
// row's last vector by dwords, zero past its end.  The lanes hold the columns
// they hold of a row padded to whole vectors, so the results are the same bits.
// Against padding the operands and unpadding the result (ten launches a step),
// us forward and forward + backward: 4096 x 4 x 1026 BF16 69.8 -> 20.5 and
// 213 -> 57 (host), 4096 x 4 x 4093 FP32 361 -> 117 and 964 -> 299 (4.6 and
// 4.5 TB/s), 16384 x 3 x 1538 FP16 195 -> 64 and 506 -> 171.
template <typename T, bool Ragged>
__device__ __forceinline__ U32x4 load_vec(__amdgpu_buffer_rsrc_t rs, int32_t voff, int32_t soff, int left) {
  constexpr int V = Vec<T>::V;
  if constexpr (!Ragged) return left > 0 ? load16(rs, voff, soff) : U32x4{0, 0, 0, 0};
  U32x4 w{0, 0, 0, 0};
  if (left >= V) {
    w = load16(rs, voff, soff);
  } else {
#pragma unroll
    for (int d = 0; d < 3; ++d)
      if (d * (V / 4) < left) w[d] = __builtin_amdgcn_raw_buffer_load_b32(rs, voff + 4 * d, soff, kStreamPolicy);
  }
  return w;
}

template <typename T, bool Ragged>
__device__ __forceinline__ void store_vec(U32x4 w, __amdgpu_buffer_rsrc_t rs, int32_t voff, int32_t row, int left) {
  constexpr int V = Vec<T>::V;
  if (Ragged ? left >= V : left > 0) {
    store16(w, rs, voff, row);
  } else if constexpr (Ragged) {
#pragma unroll
    for (int d = 0; d < 3; ++d)
      if (d * (V / 4) < left) __builtin_amdgcn_raw_buffer_store_b32(w[d], rs, voff + 4 * d, row, kStreamPolicy);
  }
}

// Wavefronts of a workgroup that share one token's columns, for passes of
// `width` columns: four, or fewer when C has fewer passes, in which case the
// others take other tokens.  By C alone (see above).
int column_parts(int64_t cols, int64_t width) {
  const int64_t passes = cols / width;
  return passes >= 4 ? 4 : passes >= 2 ? 2 : 1;
}

// A workgroup's set of tokens, slots 0 .. slots - 1, and a wavefront's share of
// it.  `parts` wavefronts share a token's columns, in passes of chunks part,
// part + parts, ...; abreast = kWaves / parts tokens run side by side in slots
// first, first + abreast, ....  Slots side by side hold neighbouring tokens,
// slots after one another tokens sets * abreast apart; the set's last slots may
// lie past the batch.
struct Share {
  int64_t base, stride;  // token of slot i: base + i % abreast + i / abreast * stride
  int64_t batch;
  int slots, abreast, shift, parts, first, part;  // abreast = 1 << shift
  __device__ __forceinline__ int64_t token(int i) const { return base + (i & (abreast - 1)) + (i >> shift) * stride; }
  __device__ __forceinline__ bool holds(int i) const { return i < slots && token(i) < batch; }
  __device__ __forceinline__ int column(int chunk, int width) const { return (chunk * parts + part) * width; }
};

template <typename Args>
__device__ __forceinline__ Share share_of(const Args& a, int wave) {
  static_assert(kWaves == 4, "parts is 1, 2 or 4");
  const int shift = a.parts == 4 ? 0 : a.parts == 2 ? 1 : 2;
  return Share{static_cast<int64_t>(blockIdx.x) << shift, a.sets << shift, a.batch, a.tokens, 1 << shift, shift,
               a.parts, wave >> (2 - shift), wave & (a.parts - 1)};
}

// exp(H) of token `b` for this lane (valid lanes), NaN for a non-finite H
// (csrc/MatrixExpSmall.cuh:126-140).
template <typename T, int N>
__device__ __forceinline__ M4 exp_of_token(const Operand& h, int64_t b, bool valid) {
  PM<false> cur;
  if (valid) {
    cur.d = load_elements<T>(h, b, N);
  } else {
#pragma unroll
    for (int e = 0; e < 16; ++e) cur.d.v[e] = 0.f;
  }
  M4 e;
  const int s = expm_lane<false>(cur, h.sign, 1.f, [&](const M4& out) { e = out; });
  if (s < 0) {
#pragma unroll
    for (int i = 0; i < 16; ++i) e.v[i] = __builtin_nanf("");
  }
  return e;
}

// exp(H) of the wavefront's tokens into its `etile` (16 floats per token): lane
// l computes the l-th of them (lanes past the last a zero matrix).  `aux`
// (optional) receives it in FP32 from one of the wavefronts that share a token.
template <typename T, int N>
__device__ __forceinline__ void exp_tokens(const HcArgs& a, const Share& sh, int lane, float* etile, float* aux) {
  const int slot = sh.first + (lane << sh.shift);
  const bool valid = sh.holds(slot);
  const int64_t b = sh.token(slot);
  const M4 e = exp_of_token<T, N>(a.h, b, valid);
  if (valid) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<float4*>(etile + 16 * lane + 4 * q) =
          make_float4(e.v[4 * q], e.v[4 * q + 1], e.v[4 * q + 2], e.v[4 * q + 3]);
    if (aux && sh.part == 0) {
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < N; ++j) aux[b * N * N + i * N + j] = e.v[4 * i + j];
    }
  }
  lds_order();
}

__device__ __forceinline__ M4 read_token(const float* tile, int i) {
  M4 m;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 v = *reinterpret_cast<const float4*>(tile + 16 * i + 4 * q);
    m.v[4 * q] = v.x;
    m.v[4 * q + 1] = v.y;
    m.v[4 * q + 2] = v.z;
    m.v[4 * q + 3] = v.w;
  }
  return m;
}

// 16-byte column chunks per lane in flight per token: the forward keeps four
// (n loads each); the backward, which loads X and dY, two -- so that it fits
// two wavefronts per SIMD beside the Frechet polynomial's registers.
constexpr int kChunks = 4;
constexpr int kChunksBwd = 2;

// Forward: Y_b = E_b X_b, row i of Y = sum_k E[i][k] X[k] (fmaf chain k = 0..n-1 from +0).
template <typename T, int N, bool Ragged>
__global__ __launch_bounds__(64 * kWaves) void hc_mix_fwd_kernel(HcArgs a) {
  __shared__ __attribute__((aligned(16))) float etile_mem[kWaves][kTokens * 16];
  constexpr int es = static_cast<int>(sizeof(typename T::storage));
  constexpr int V = Vec<T>::V;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float* etile = etile_mem[wave];
  const Share sh = share_of(a, wave);
  // One token's offsets stay below 2^31 (the host checks the spans).
  const int cols = static_cast<int>(a.cols);
  const int xr_step = static_cast<int>(a.xr);
  exp_tokens<T, N>(a, sh, lane, etile, a.aux);
  // Passes of Chunks chunks.  Ragged rows cost two branches a vector, so chunks past
  // the row's end are left out: rows of one chunk have passes of one, longer ones
  // compute and store what is there (a branch between the loads as well costs rows
  // of 4 KiB 5%).  100000 x 4 x 34, 130 and 258 BF16: 236 -> 88, 238 -> 98 and 239 ->
  // 106 us (padding the operands instead: 108, 177 and 286).
  const auto stream = [&](auto chunks) {
    constexpr int Chunks = decltype(chunks)::value;
    for (int i = sh.first; sh.holds(i); i += sh.abreast) {
      const M4 e = read_token(etile, i >> sh.shift);
      const __amdgpu_buffer_rsrc_t xs = rebased<T>(a.x, sh.token(i) * a.xb, ((N - 1) * a.xr + a.cols) * es);
      const __amdgpu_buffer_rsrc_t ys = rebased<T>(a.out, sh.token(i) * N * a.cols, N * a.cols * es);
      for (int m = 0; sh.column(m, 64 * V) < cols; m += Chunks) {
        U32x4 raw[Chunks][N];
#pragma unroll
        for (int u = 0; u < Chunks; ++u) {
          const int c = sh.column(m + u, 64 * V) + lane * V;
#pragma unroll
          for (int k = 0; k < N; ++k) raw[u][k] = load_vec<T, Ragged>(xs, c * es, k * xr_step * es, cols - c);
        }
#pragma unroll
        for (int u = 0; u < Chunks; ++u) {
          if (Ragged && sh.column(m + u, 64 * V) >= cols) break;
          const int c = sh.column(m + u, 64 * V) + lane * V;
          Vec<T> xv[N];
#pragma unroll
          for (int k = 0; k < N; ++k) xv[k] = unpack<T>(raw[u][k]);
#pragma unroll
          for (int i2 = 0; i2 < N; ++i2) {
            Vec<T> y;
#pragma unroll
            for (int v = 0; v < V; ++v) {
              float acc = __builtin_fmaf(e.v[4 * i2], xv[0].f[v], 0.f);
#pragma unroll
              for (int k = 1; k < N; ++k) acc = __builtin_fmaf(e.v[4 * i2 + k], xv[k].f[v], acc);
              y.f[v] = acc;
            }
            store_vec<T, Ragged>(pack<T>(y), ys, c * es, i2 * cols * es, cols - c);
          }
        }
      }
    }
  };
  if (Ragged && cols <= 64 * V) {
    stream(std::integral_constant<int, 1>());
  } else {
    stream(std::integral_constant<int, kChunks>());
  }
}

// Value of the lane whose index differs in bit 3 (row_ror:8) or bit 2
// (row_ror:4 for lanes with the bit set, row_ror:12 for the others) or by a
// permutation of the quad.
template <int Quad>
__device__ __forceinline__ float quad_lane(float v) {
  const int w = __float_as_int(v);
  return __int_as_float(__builtin_amdgcn_update_dpp(w, w, Quad, 0xF, 0xF, false));
}
__device__ __forceinline__ float lane_xor8(float v) {
  const int w = __float_as_int(v);
  return __int_as_float(__builtin_amdgcn_update_dpp(w, w, 0x128, 0xF, 0xF, false));
}
__device__ __forceinline__ float lane_xor4(float v) {
  const int w = __float_as_int(v);
  const int t = __builtin_amdgcn_update_dpp(w, w, 0x124, 0xF, 0xA, false);
  return __int_as_float(__builtin_amdgcn_update_dpp(t, w, 0x12C, 0xF, 0x5, false));
}

// Sums of M per-lane values (a power of two up to 64) over the wavefront,
// reduce-scatter style: six exchanges with the lane 32, 16, 8, 4, 2, 1 apart;
// while more than one value is left, each keeps the half this lane's bit
// selects.  Lane l returns the total of entry l / (64 / M), summed in a fixed
// tree.  The first two exchanges are register swaps between halves and between
// rows of the wavefront, the others DPP moves: against exchanges through
// ds_bpermute the backward at 16384 x 2 x 4096 BF16 ran 189 -> 135 us and at 16384 x 4 x 1024 86 -> 79 us.
template <int M>
__device__ __forceinline__ float wave_sum(const float (&v)[M], int lane) {
  float a[M];
#pragma unroll
  for (int e = 0; e < M; ++e) a[e] = v[e];
#pragma unroll
  for (int step = 0; step < 6; ++step) {
    const int half = M >> (step + 1);
    const bool upper = (lane >> (5 - step)) & 1;
#pragma unroll
    for (int j = 0; j < (half > 0 ? half : 1); ++j) {
      const float x = a[j];
      const float y = half > 0 ? a[j + half] : a[j];
      if (step < 2) {
        // Swaps x of the upper lanes with y of the lower ones: the sum of both
        // registers is x's pair sum in the lower lanes, y's in the upper.
        typedef uint32_t U2 __attribute__((ext_vector_type(2)));
        const U2 s = step == 0
                         ? __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false)
                         : __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
        a[j] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
      } else {
        const float keep = upper ? y : x;
        const float send = upper ? x : y;
        a[j] = keep + (step == 2   ? lane_xor8(send)
                       : step == 3 ? lane_xor4(send)
                       : step == 4 ? quad_lane<0x4E>(send)
                                   : quad_lane<0xB1>(send));
      }
    }
  }
  return a[0];
}

// Backward: dX row k = sum_r E[r][k] dY[r] (fmaf chain r = 0..n-1 from +0);
// dE[r][k] = sum_c dY[r][c] X[k][c] (per lane in column order, then
// wave_sum, then the wavefronts' parts in order); dH = L(H^T, dE).
template <typename T, int N, bool Ragged>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 8))) void hc_mix_bwd_kernel(HcArgs a) {
  __shared__ __attribute__((aligned(16))) float etile_mem[kWaves][kTokens * 16];
  __shared__ __attribute__((aligned(16))) float gtile_mem[kWaves][kTokens * 16];  // dE by column part
  constexpr int es = static_cast<int>(sizeof(typename T::storage));
  constexpr int V = Vec<T>::V;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float* etile = etile_mem[wave];
  const Share sh = share_of(a, wave);
  // One token's offsets stay below 2^31 (the host checks the spans).
  const int cols = static_cast<int>(a.cols);
  const int xr_step = static_cast<int>(a.xr);
  const int gr_step = static_cast<int>(a.gr);
  exp_tokens<T, N>(a, sh, lane, etile, nullptr);
  for (int i = sh.first; sh.holds(i); i += sh.abreast) {
    const int64_t b = sh.token(i);
    const M4 e = read_token(etile, i >> sh.shift);
    const __amdgpu_buffer_rsrc_t xs = rebased<T>(a.x, b * a.xb, ((N - 1) * a.xr + a.cols) * es);
    const __amdgpu_buffer_rsrc_t gs = rebased<T>(a.gy, b * a.gb, ((N - 1) * a.gr + a.cols) * es);
    const __amdgpu_buffer_rsrc_t ds = rebased<T>(a.out, b * N * a.cols, N * a.cols * es);
    constexpr int M = N == 2 ? 4 : 16;  // entries r N + k of dE, a power of two
    float acc[M];
#pragma unroll
    for (int q = 0; q < M; ++q) acc[q] = 0.f;
    for (int m = 0; sh.column(m, 64 * V) < cols; m += kChunksBwd) {
      U32x4 xr[kChunksBwd][N], gr[kChunksBwd][N];
#pragma unroll
      for (int u = 0; u < kChunksBwd; ++u) {
        const int c = sh.column(m + u, 64 * V) + lane * V;
#pragma unroll
        for (int k = 0; k < N; ++k) {
          xr[u][k] = load_vec<T, Ragged>(xs, c * es, k * xr_step * es, cols - c);
          gr[u][k] = load_vec<T, Ragged>(gs, c * es, k * gr_step * es, cols - c);
        }
      }
#pragma unroll
      for (int u = 0; u < kChunksBwd; ++u) {
        const int c = sh.column(m + u, 64 * V) + lane * V;
        Vec<T> xv[N], gv[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
          xv[k] = unpack<T>(xr[u][k]);
          gv[k] = unpack<T>(gr[u][k]);
        }
#pragma unroll
        for (int k = 0; k < N; ++k) {
          Vec<T> dx;
#pragma unroll
          for (int v = 0; v < V; ++v) {
            float d = __builtin_fmaf(e.v[k], gv[0].f[v], 0.f);
#pragma unroll
            for (int r = 1; r < N; ++r) d = __builtin_fmaf(e.v[4 * r + k], gv[r].f[v], d);
            dx.f[v] = d;
          }
          store_vec<T, Ragged>(pack<T>(dx), ds, c * es, k * cols * es, cols - c);
        }
#pragma unroll
        for (int r = 0; r < N; ++r)
#pragma unroll
          for (int k = 0; k < N; ++k)
#pragma unroll
            for (int v = 0; v < V; ++v) acc[N * r + k] = __builtin_fmaf(gv[r].f[v], xv[k].f[v], acc[N * r + k]);
      }
    }
    const float total = wave_sum(acc, lane);
    const int entry = lane / (64 / M);
    if (lane % (64 / M) == 0 && entry < N * N) gtile_mem[sh.part][16 * i + 4 * (entry / N) + entry % N] = total;
  }
  __syncthreads();
  if (wave != 0) return;
  // L(H^T, dE) of the set's token `lane`.
  const int64_t b = sh.token(lane);
  const bool valid = sh.holds(lane);
  PM<true> cur;
  if (valid) {
    const M4 h = load_elements<T>(a.h, b, N);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c) cur.d.v[4 * r + c] = h.v[4 * c + r];
    cur.u = read_token(gtile_mem[0], lane);
    for (int p = 1; p < sh.parts; ++p) {
      const M4 more = read_token(gtile_mem[p], lane);
#pragma unroll
      for (int q = 0; q < 16; ++q) cur.u.v[q] += more.v[q];
    }
#pragma unroll
    for (int q = 0; q < 16; ++q)
      if (q / 4 >= N || q % 4 >= N) cur.u.v[q] = 0.f;
    // The debug copy of dE goes out now, so that cur.u is not kept live
    // across the Frechet polynomial (it would spill at the 256-VGPR cap).
    if (a.aux) {
#pragma unroll
      for (int r = 0; r < N; ++r)
#pragma unroll
        for (int k = 0; k < N; ++k) a.aux[b * N * N + r * N + k] = cur.u.v[4 * r + k];
    }
  } else {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      cur.d.v[q] = 0.f;
      cur.u.v[q] = 0.f;
    }
  }
  M4 dh;
  const int s = expm_lane<true>(cur, a.h.sign, 1.f, [&](const M4& out) { dh = out; });
  if (s < 0) {
#pragma unroll
    for (int q = 0; q < 16; ++q) dh.v[q] = __builtin_nanf("");
  }
  if (valid) store_elements<T>(a.dh, b, N, dh);
}

// ---- 5 <= n <= 8 streams: exp(H) supplied in FP32 ----------------------------
//
// For n = 5..8 the exponential runs in its own kernel (P = 8, FP32 output, the
// same bits the fused path would keep on chip); these kernels apply it.  The
// token sets, column shares, row streaming and nontemporal hints are the fused
// kernels'.  E of the set's tokens sits in the workgroup's LDS in rows of 8
// floats (64 per token): E itself for the forward, E^T for the backward, so
// that the row an output row needs is two 16-byte broadcast reads.

struct WideArgs {
  const float* e;   // FP32 [B, n, n], contiguous
  const void* x;    // [B, n, C], unit column stride
  int64_t xb, xr;
  const void* gy;   // backward: dY [B, n, C], unit column stride
  int64_t gb, gr;
  void* out;        // forward: Y, backward: dX; contiguous [B, n, C]
  float* de;        // backward: dE = dY X^T, FP32 [B, n, n], contiguous
  int64_t batch;
  int64_t cols;
  int64_t sets;     // workgroups
  int tokens;       // per workgroup
  int parts;        // wavefronts that share a token's columns (column_parts)
  int n;
};

constexpr int kWideChunks = 2;     // 16-byte column chunks per lane in flight (forward)
constexpr int kWideChunksBwd = 2;  // 8-byte column chunks per lane in flight (backward)

// 8 bytes of storage as FP32 values (2 for FP32, 4 for FP16/BF16).
template <typename T>
struct Vec8 {
  static constexpr int V = 8 / static_cast<int>(sizeof(typename T::storage));
  float f[V];
};

template <typename T>
__device__ __forceinline__ Vec8<T> unpack8(U32x2 w) {
  using S = typename T::storage;
  Vec8<T> r;
#pragma unroll
  for (int i = 0; i < Vec8<T>::V; ++i) {
    if constexpr (sizeof(S) == 4) {
      r.f[i] = __uint_as_float(w[i]);
    } else {
      const uint16_t h = static_cast<uint16_t>(w[i >> 1] >> (16 * (i & 1)));
      r.f[i] = to_f32<T>(__builtin_bit_cast(S, h));
    }
  }
  return r;
}

template <typename T>
__device__ __forceinline__ U32x2 pack8(const Vec8<T>& v) {
  using S = typename T::storage;
  U32x2 w;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if constexpr (sizeof(S) == 4) {
      w[i] = __float_as_uint(v.f[i]);
    } else {
      w[i] = static_cast<uint32_t>(__builtin_bit_cast(uint16_t, from_f32<T>(v.f[2 * i]))) |
             (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, from_f32<T>(v.f[2 * i + 1]))) << 16);
    }
  }
  return w;
}

__device__ __forceinline__ U32x2 load8(__amdgpu_buffer_rsrc_t rs, int32_t voff, int32_t soff) {
  return __builtin_amdgcn_raw_buffer_load_b64(rs, voff, soff, kStreamPolicy);
}

__device__ __forceinline__ void store8(U32x2 w, __amdgpu_buffer_rsrc_t rs, int32_t voff, int32_t soff) {
  __builtin_amdgcn_raw_buffer_store_b64(w, rs, voff, soff, kStreamPolicy);
}

// E of the set's tokens into `etile` (64 floats per token, rows of 8), eight
// threads a token: thread p of them copies row p (transposed: column p).  The
// whole workgroup loads the tokens its wavefronts share; when they share none,
// each wavefront loads its own and waits for no other.
template <int N, bool Transposed>
__device__ __forceinline__ void load_set_e(const WideArgs& a, const Share& sh, int lane, float* etile) {
  const bool shared = sh.parts > 1;
  const int p = threadIdx.x & 7;
  const int step = shared ? 8 * kWaves : 8 * sh.abreast;
  for (int j = shared ? threadIdx.x >> 3 : sh.first + (lane >> 3) * sh.abreast; j < sh.slots; j += step) {
    if (p < N && sh.holds(j)) {
      const float* src = a.e + sh.token(j) * (N * N);
#pragma unroll
      for (int k = 0; k < N; ++k) etile[64 * j + 8 * p + k] = Transposed ? src[k * N + p] : src[p * N + k];
    }
  }
  if (shared) {
    __syncthreads();
  } else {
    lds_order();
  }
}

// Row r of the token's 8-float rows (the first N entries are used).
__device__ __forceinline__ void read_row8(const float* tile, int token, int r, float (&row)[8]) {
  const float4 lo = *reinterpret_cast<const float4*>(tile + 64 * token + 8 * r);
  const float4 hi = *reinterpret_cast<const float4*>(tile + 64 * token + 8 * r + 4);
  row[0] = lo.x; row[1] = lo.y; row[2] = lo.z; row[3] = lo.w;
  row[4] = hi.x; row[5] = hi.y; row[6] = hi.z; row[7] = hi.w;
}

// Forward: row i of Y = sum_k E[i][k] X[k] (fmaf chain k = 0..n-1 from +0).
template <typename T, int N>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 8))) void hc_wide_fwd_kernel(WideArgs a) {
  __shared__ __attribute__((aligned(16))) float etile[kWaves * kWideTokens * 64];
  constexpr int es = static_cast<int>(sizeof(typename T::storage));
  constexpr int V = Vec<T>::V;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Share sh = share_of(a, wave);
  // One token's offsets stay below 2^31 (the host checks the spans).
  const int cols = static_cast<int>(a.cols);
  const int xr_step = static_cast<int>(a.xr);
  load_set_e<N, false>(a, sh, lane, etile);
  for (int i = sh.first; sh.holds(i); i += sh.abreast) {
    const int64_t b = sh.token(i);
    float e[N][8];
#pragma unroll
    for (int r = 0; r < N; ++r) read_row8(etile, i, r, e[r]);
    const __amdgpu_buffer_rsrc_t xs = rebased<T>(a.x, b * a.xb, ((N - 1) * a.xr + a.cols) * es);
    const __amdgpu_buffer_rsrc_t ys = rebased<T>(a.out, b * N * a.cols, N * a.cols * es);
    for (int m = 0; sh.column(m, 64 * V) < cols; m += kWideChunks) {
      U32x4 raw[kWideChunks][N];
#pragma unroll
      for (int u = 0; u < kWideChunks; ++u) {
        const int c = sh.column(m + u, 64 * V) + lane * V;
#pragma unroll
        for (int k = 0; k < N; ++k)
          raw[u][k] = c < cols ? load16(xs, c * es, k * xr_step * es) : U32x4{0, 0, 0, 0};
      }
#pragma unroll
      for (int u = 0; u < kWideChunks; ++u) {
        const int c = sh.column(m + u, 64 * V) + lane * V;
        Vec<T> xv[N];
#pragma unroll
        for (int k = 0; k < N; ++k) xv[k] = unpack<T>(raw[u][k]);
#pragma unroll
        for (int i2 = 0; i2 < N; ++i2) {
          Vec<T> y;
#pragma unroll
          for (int v = 0; v < V; ++v) {
            float acc = __builtin_fmaf(e[i2][0], xv[0].f[v], 0.f);
#pragma unroll
            for (int k = 1; k < N; ++k) acc = __builtin_fmaf(e[i2][k], xv[k].f[v], acc);
            y.f[v] = acc;
          }
          if (c < cols) store16(pack<T>(y), ys, c * es, i2 * cols * es);
        }
      }
    }
  }
}

// Backward: dX row k = sum_r E[r][k] dY[r] (fmaf chain r = 0..n-1 from +0);
// dE[r][k] = sum_c dY[r][c] X[k][c] (per lane in column order, then
// wave_sum, then the wavefronts' parts in order), written to a.de.
template <typename T, int N>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 8))) void hc_wide_bwd_kernel(WideArgs a) {
  // E of the set and, where wavefronts share tokens (a set has kWideTokens then), dE
  // by column part.
  __shared__ __attribute__((aligned(16))) float etile[(1 + kWaves) * kWideTokens * 64];
  float(*const gtile)[kWideTokens * 64] = reinterpret_cast<float(*)[kWideTokens * 64]>(etile + kWideTokens * 64);
  constexpr int es = static_cast<int>(sizeof(typename T::storage));
  constexpr int V = Vec8<T>::V;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Share sh = share_of(a, wave);
  // One token's offsets stay below 2^31 (the host checks the spans).
  const int cols = static_cast<int>(a.cols);
  const int xr_step = static_cast<int>(a.xr);
  const int gr_step = static_cast<int>(a.gr);
  load_set_e<N, true>(a, sh, lane, etile);
  for (int i = sh.first; sh.holds(i); i += sh.abreast) {
    const int64_t b = sh.token(i);
    const __amdgpu_buffer_rsrc_t xs = rebased<T>(a.x, b * a.xb, ((N - 1) * a.xr + a.cols) * es);
    const __amdgpu_buffer_rsrc_t gs = rebased<T>(a.gy, b * a.gb, ((N - 1) * a.gr + a.cols) * es);
    const __amdgpu_buffer_rsrc_t ds = rebased<T>(a.out, b * N * a.cols, N * a.cols * es);
    float acc[64];
#pragma unroll
    for (int q = 0; q < 64; ++q) acc[q] = 0.f;
    for (int m = 0; sh.column(m, 64 * V) < cols; m += kWideChunksBwd) {
      U32x2 xr[kWideChunksBwd][N], gr[kWideChunksBwd][N];
#pragma unroll
      for (int u = 0; u < kWideChunksBwd; ++u) {
        const int c = sh.column(m + u, 64 * V) + lane * V;
#pragma unroll
        for (int k = 0; k < N; ++k) {
          xr[u][k] = c < cols ? load8(xs, c * es, k * xr_step * es) : U32x2{0, 0};
          gr[u][k] = c < cols ? load8(gs, c * es, k * gr_step * es) : U32x2{0, 0};
        }
      }
#pragma unroll
      for (int u = 0; u < kWideChunksBwd; ++u) {
        const int c = sh.column(m + u, 64 * V) + lane * V;
        Vec8<T> xv[N], gv[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
          xv[k] = unpack8<T>(xr[u][k]);
          gv[k] = unpack8<T>(gr[u][k]);
        }
#pragma unroll
        for (int k = 0; k < N; ++k) {
          float col[8];
          read_row8(etile, i, k, col);  // column k of E
          Vec8<T> dx;
#pragma unroll
          for (int v = 0; v < V; ++v) {
            float d = __builtin_fmaf(col[0], gv[0].f[v], 0.f);
#pragma unroll
            for (int r = 1; r < N; ++r) d = __builtin_fmaf(col[r], gv[r].f[v], d);
            dx.f[v] = d;
          }
          if (c < cols) store8(pack8<T>(dx), ds, c * es, k * cols * es);
        }
#pragma unroll
        for (int r = 0; r < N; ++r)
#pragma unroll
          for (int k = 0; k < N; ++k)
#pragma unroll
            for (int v = 0; v < V; ++v) acc[r * N + k] = __builtin_fmaf(gv[r].f[v], xv[k].f[v], acc[r * N + k]);
      }
    }
    const float total = wave_sum(acc, lane);
    if (sh.parts == 1) {
      if (lane < N * N) a.de[b * (N * N) + lane] = total;
    } else {
      gtile[sh.part][64 * i + lane] = total;
    }
  }
  if (sh.parts == 1) return;
  __syncthreads();
  for (int t = threadIdx.x; t < 64 * sh.slots; t += 64 * kWaves) {
    const int entry = t & 63;
    if (entry < N * N && sh.holds(t >> 6)) {
      float total = gtile[0][t];
      for (int p = 1; p < sh.parts; ++p) total += gtile[p][t];
      a.de[sh.token(t >> 6) * (N * N) + entry] = total;
    }
  }
}

// Grid: two workgroups a compute unit, until each has `most` tokens; from there
// on more workgroups, which the hardware starts as others retire (finer sets
// balance the last ones, coarser sets pay for fewer exponentials).
template <typename Args>
hipError_t launch_sets(void (*kernel)(Args), Args a, int most, hipStream_t stream) {
  const int64_t target = 2 * compute_units();
  const int abreast = kWaves / a.parts;
  const int64_t rounds = (a.batch + target * abreast - 1) / (target * abreast);
  a.tokens = rounds * abreast < most ? static_cast<int>(rounds * abreast) : most;
  a.sets = (a.batch + a.tokens - 1) / a.tokens;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(a.sets)), dim3(64 * kWaves), 0, stream, a);
  return hipGetLastError();
}

// Tokens of a wavefront that shares none, at most: as many as have 4 KiB of one row
// together (what a pass takes of a row that wide), but 2 and no more than `most`.
// An exponential pass serves a wavefront's tokens however few they are, so sets
// have to grow as rows shrink: forward 262144 x 4 x C BF16, us, 2 / 4 / 8 / 16
// tokens, C = 64 264 / 213 / 185 / 174, C = 256 301 / 248 / 223 / 222; 131072 x 4
// x 512 196 / 180 / 183, 40000 x 4 x 1024 112 / 116 / 122.
int own_tokens(int64_t row_bytes, int most) {
  const int64_t each = 4096 / row_bytes;
  return each < 2 ? 2 : each > most ? most : static_cast<int>(each);
}

// Where wavefronts share a token, or share the backward's Frechet polynomial a set:
// 8 / 16 / 32 tokens, 40000 x 4 x 1024 and 16384 x 4 x 1024 BF16 backward 195 / 178 /
// 183 and 87 / 81 / 79 us.
template <typename T, int N, bool Backward>
hipError_t launch_one(HcArgs a, hipStream_t stream) {
  // Whole 16-byte vectors everywhere, or rows in whole dwords at any dword.  The
  // line lies at the dword because buffer accesses of a dword or more need that
  // alignment: rows of an odd number of 16-bit values are padded by the caller.
  constexpr int V = Vec<T>::V;
  const bool ragged = ((reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.gy) |
                        reinterpret_cast<uintptr_t>(a.out)) % 16 != 0) ||
                      ((a.cols | a.xb | a.xr | a.gb | a.gr) % V != 0);
  const auto kernel = Backward ? (ragged ? hc_mix_bwd_kernel<T, N, true> : hc_mix_bwd_kernel<T, N, false>)
                               : (ragged ? hc_mix_fwd_kernel<T, N, true> : hc_mix_fwd_kernel<T, N, false>);
  // A ragged row shares its columns as the row padded to whole vectors would.
  a.parts = column_parts((a.cols + V - 1) / V * V, 64 * V * kChunksBwd);
  const int most = Backward        ? kTokens
                   : a.parts > 1 ? kTokens / 2
                                 : kWaves * own_tokens(a.cols * static_cast<int64_t>(sizeof(typename T::storage)), kTokens);
  return launch_sets(kernel, a, most, stream);
}

template <typename T>
hipError_t launch_t(const HcArgs& a, bool backward, hipStream_t stream) {
  switch (a.n) {
    case 2:
      return backward ? launch_one<T, 2, true>(a, stream) : launch_one<T, 2, false>(a, stream);
    case 3:
      return backward ? launch_one<T, 3, true>(a, stream) : launch_one<T, 3, false>(a, stream);
    default:
      return backward ? launch_one<T, 4, true>(a, stream) : launch_one<T, 4, false>(a, stream);
  }
}

// n = 5..8, where sets cost a load of E: 2 / 4 / 8 / 16 tokens a wavefront at 262144 x
// 8 x 64 BF16, us, forward 441 / 423 / 407 / 404 and backward 701 / 677 / 656 / 648,
// but at 100000 x 6 x 128 95 / 92 / 96 / 104 and 181 / 166 / 170 / 188; 8 / 16 tokens
// a workgroup at 16384 x 6 x 1024 forward 68.7 / 70.6 and backward 103 / 108.
template <typename T, int N, bool Backward>
hipError_t launch_wide_one(WideArgs a, hipStream_t stream) {
  const auto kernel = Backward ? hc_wide_bwd_kernel<T, N> : hc_wide_fwd_kernel<T, N>;
  constexpr int pass = 64 * (Backward ? Vec8<T>::V * kWideChunksBwd : Vec<T>::V * kWideChunks);
  // The backward's reduction of 64 sums costs a fifth of a pass: two passes per wavefront at least.
  a.parts = column_parts(a.cols, Backward ? 2 * pass : pass);
  const int64_t row_bytes = a.cols * static_cast<int64_t>(sizeof(typename T::storage));
  return launch_sets(kernel, a, a.parts > 1 ? kWideTokens : kWaves * own_tokens(row_bytes, kWideTokens), stream);
}

template <typename T, bool Backward>
hipError_t launch_wide_t(const WideArgs& a, hipStream_t stream) {
  switch (a.n) {
    case 5:
      return launch_wide_one<T, 5, Backward>(a, stream);
    case 6:
      return launch_wide_one<T, 6, Backward>(a, stream);
    case 7:
      return launch_wide_one<T, 7, Backward>(a, stream);
    default:
      return launch_wide_one<T, 8, Backward>(a, stream);
  }
}

}  // namespace

// A launch takes at most kSlice tokens (a grid holds fewer than 2^24 workgroups
// of 256 threads); a larger batch goes in slices.
constexpr int64_t kSlice = int64_t{1} << 26;

const void* advanced(const void* p, int64_t bytes) { return p ? static_cast<const char*>(p) + bytes : nullptr; }
void* advanced(void* p, int64_t bytes) { return p ? static_cast<char*>(p) + bytes : nullptr; }

hipError_t launch_hc_apply(const float* e, const void* x, const int64_t* xs, const void* gy, const int64_t* gs,
                           void* out, float* de, int dtype, int64_t batch, int n, int64_t cols, hipStream_t stream) {
  return in_slices(batch, kSlice, [&](int64_t first, int64_t count) {
    WideArgs a;
    a.xb = xs[0];
    a.xr = xs[1];
    a.gb = gs ? gs[0] : 0;
    a.gr = gs ? gs[1] : 0;
    const MixBytes at = mix_bytes(first, dtype == F32::code ? 4 : 2, n, cols, 0, a.xb, a.gb);
    a.e = static_cast<const float*>(advanced(e, at.square_f32));
    a.x = advanced(x, at.x);
    a.gy = advanced(gy, at.gy);
    a.out = advanced(out, at.rows);
    a.de = static_cast<float*>(advanced(de, at.square_f32));
    a.batch = count;
    a.cols = cols;
    a.n = n;
    if (gy != nullptr) {
      if (dtype == F32::code) return launch_wide_t<F32, true>(a, stream);
      if (dtype == BF16::code) return launch_wide_t<BF16, true>(a, stream);
      return launch_wide_t<F16, true>(a, stream);
    }
    if (dtype == F32::code) return launch_wide_t<F32, false>(a, stream);
    if (dtype == BF16::code) return launch_wide_t<BF16, false>(a, stream);
    return launch_wide_t<F16, false>(a, stream);
  });
}

hipError_t launch_hc_mix(const Operand& h, const void* x, const int64_t* xs, const void* gy, const int64_t* gs,
                         void* out, void* dh, float* aux, int dtype, int64_t batch, int n, int64_t cols,
                         hipStream_t stream) {
  return in_slices(batch, kSlice, [&](int64_t first, int64_t count) {
    HcArgs a;
    a.h = h;
    a.xb = xs[0];
    a.xr = xs[1];
    a.gb = gs ? gs[0] : 0;
    a.gr = gs ? gs[1] : 0;
    const MixBytes at = mix_bytes(first, dtype == F32::code ? 4 : 2, n, cols, h.sb, a.xb, a.gb);
    a.h.data = advanced(h.data, at.h);
    a.x = advanced(x, at.x);
    a.gy = advanced(gy, at.gy);
    a.out = advanced(out, at.rows);
    a.dh = advanced(dh, at.square);
    a.aux = static_cast<float*>(advanced(aux, at.square_f32));
    a.batch = count;
    a.cols = cols;
    a.n = n;
    const bool backward = gy != nullptr;
    if (dtype == F32::code) return launch_t<F32>(a, backward, stream);
    if (dtype == BF16::code) return launch_t<BF16>(a, backward, stream);
    return launch_t<F16>(a, backward, stream);
  });
}

}  // namespace fh
