// fp32 contractions on the bf16 matrix cores (gfx950), without giving up fp32
// precision.
//
// An fp32 number is the exact sum of three bf16 numbers (Henry, Tang and
// Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for
// higher-precision computations", 2019): x = h + m + l, where h is x rounded to
// bf16, m the difference rounded to bf16 and l what is left (both differences
// are exact in fp32, |m| <= 2^-8 and |l| <= 2^-17 of x's power of two).  A
// product x*y is then nine bf16 products, each exact in fp32, of which the MFMA
// sums the six that reach fp32 precision:
//   x y = h h' + (h m' + m h') + (h l' + l h' + m m')  + [m l' + l m' + l l']
// The three left out are together below 2^-24 (1 + 2^-10) of |x y|, one fp32
// rounding, of either sign (2^-28 on average over normal data).  Rounded to
// nearest, not cut off: the parts of a cut number all have its sign and are up
// to twice as large, and the three left out reach 2^-21 of every product, all
// the same way (x = y = 1 + 2^-7 - 2^-23).  The six products go to two
// accumulators -- h h' to one, the small five to the other -- added once at the
// end: a small product added to a large accumulator inside the MFMA would lose
// its low bits at every step (measured over K = 2048 products of one sign: one
// accumulator 3.5e-6 relative error, two 2.5e-7, the fp32 MFMA 7.0e-7; K = 64
// of either sign 7.8e-8 against 1.4e-7 of the fp32 MFMA).
//
// The upper parts of an infinity leave NaN below them, and so do those of a
// number from FLT_MAX (1 - 2^-9) on, which rounds to infinity; h h' may also
// pass the range where the product does not.  A result that is not finite is
// therefore formed again without the split by each kernel.
//
// Why: v_mfma_f32_32x32x16_bf16 does 32768 flops in 32 cycles, v_mfma_f32_16x16x4
// (fp32) 2048 in 32, so six bf16 products take 0.375 of the fp32 matrix time;
// and a bf16 MFMA leaves the VALU issue slots beside it free (measured: 64 VALU
// operations between 16 32x32x16 MFMAs cost 3%, an fp32 MFMA and a VALU
// operation do not overlap at all).
//
// MFMA operand layout (v_mfma_f32_32x32x16_bf16, wave64, lane group g = l/32):
//   A (32x16): lane l supplies A[m = l%32][k = 8g + j], j = 0..7
//   B (16x32): lane l supplies B[k = 8g + j][n = l%32]
//   D (32x32): lane l holds    D[m = 8(i/4) + 4g + i%4][n = l%32], i = 0..15
// The contraction index k can be mapped to any physical index as long as A and
// B agree.
#pragma once
#include <type_traits>

#include "wha_device.hpp"

namespace wha {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// A pair of floats as bf16, to nearest (ties to even), packed in one register
// (first float in the low half), and what remains of the pair.
__device__ __forceinline__ unsigned bf16_pair(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector((floatx2{a, b}), bf16x2));
}
__device__ __forceinline__ unsigned take_pair(float& a, float& b) {
  const unsigned h = bf16_pair(a, b);
  a -= __uint_as_float(h << 16);
  b -= __uint_as_float(h & 0xffff0000u);
  return h;
}
// The three bf16 parts of a pair of floats.
struct SplitPair {
  unsigned h, m, l;
};
__device__ __forceinline__ SplitPair split_pair(float a, float b) {
  SplitPair s;
  s.h = take_pair(a, b);
  s.m = take_pair(a, b);
  s.l = bf16_pair(a, b);
  return s;
}

// One MFMA operand (8 k values of one row or column) in its three parts.
struct Frag3 {
  bf16x8 h, m, l;
};
__device__ __forceinline__ Frag3 split_frag(const float (&x)[8]) {
  uintx4 h, m, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const SplitPair s = split_pair(x[2 * i], x[2 * i + 1]);
    h[i] = s.h;
    m[i] = s.m;
    l[i] = s.l;
  }
  return Frag3{__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}

__device__ __forceinline__ floatx16 mfma_bf16(bf16x8 a, bf16x8 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// Two k of fp32 as they stand: lane l supplies A[m = l%32][k = l/32] and
// B[k = l/32][n = l%32], D as above.
__device__ __forceinline__ floatx16 mfma_f32(float a, float b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
// The five small products, smallest first.
__device__ __forceinline__ floatx16 mfma_small(const Frag3& a, const Frag3& b, floatx16 c) {
  c = mfma_bf16(a.l, b.h, c);
  c = mfma_bf16(a.h, b.l, c);
  c = mfma_bf16(a.m, b.m, c);
  c = mfma_bf16(a.m, b.h, c);
  return mfma_bf16(a.h, b.m, c);
}
// Product e (0..4) of mfma_small.
__device__ __forceinline__ floatx16 mfma_small_step(int e, const Frag3& a, const Frag3& b, floatx16 c) {
  return e == 0   ? mfma_bf16(a.l, b.h, c)
         : e == 1 ? mfma_bf16(a.h, b.l, c)
         : e == 2 ? mfma_bf16(a.m, b.m, c)
         : e == 3 ? mfma_bf16(a.m, b.h, c)
                  : mfma_bf16(a.h, b.m, c);
}
// Keeps the computation of x where it stands in program order, between the
// fences around it: an empty statement (no instruction) that x passes through.
// The optimizer otherwise moves a pure MFMA or VALU chain to its first use.
template <class T>
__device__ __forceinline__ void pin(T& x) {
  asm volatile("" : "+v"(x));
}

// NM MFMAs, mfma(i), with NP pieces of other work, piece(j), spread evenly
// between them in program order.  A wave issues in order, so only work placed
// right behind an MFMA runs beside it: up to six VALU operations per MFMA are
// free there (36 cycles per MFMA against 36 without, measured), in a block after
// the MFMAs none are -- neither the compiler's order nor a second wave on the
// SIMD overlapped them.
template <int J, int END, class P>
__device__ __forceinline__ void run_pieces(P&& piece) {
  if constexpr (J < END) {
    piece(std::integral_constant<int, J>{});
    run_pieces<J + 1, END>(piece);
  }
}
template <int NM, int NP, int I = 0, class M, class P>
__device__ __forceinline__ void interleave(M&& mfma, P&& piece) {
  if constexpr (I < NM) {
    mfma(std::integral_constant<int, I>{});
    run_pieces<I * NP / NM, (I + 1) * NP / NM>(piece);
    WHA_FENCE();
    interleave<NM, NP, I + 1>(mfma, piece);
  }
}
__device__ __forceinline__ floatx16 zero16() {
  floatx16 z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.f;
  return z;
}

// Row within a 32 x 32 MFMA result of element i of lane group g.
__device__ __forceinline__ int acc_row(int i, int g) { return 8 * (i >> 2) + 4 * g + (i & 3); }

// A 32-row tile of a [T][D] operand in LDS, as three bf16 planes, in one of two
// layouts:
//   rows  [32][16 NKS d]: operand of contractions over the head dimension
//         (k-slot s of k-step ks is d = 16 ks + s).  Row pitch an odd number of
//         quads, so any 16 lanes reading the same quad of rows distinct mod 16
//         (the sets the LDS serves together) meet 16 different quads.
//   cols  [32 NDT d][32 slots]: operand of contractions over the tile's rows.
//         Slot 8g + j of k-step ks is row 16 ks + acc_row(j, g), the order in
//         which a lane holds the elements of a 32 x 32 MFMA result -- which is
//         so the other operand as it stands, without a shuffle.  d = 4q + u is
//         stored at row (8 NDT) u + q, quad c at c ^ ((q >> 2) ^ u) & 3: reads
//         and stores (below) are free of bank conflicts.
// A staging unit is two adjacent rows x 4 d, two 128-bit loads; unit x is
// d-group x % G of row pair x / G, pairs ordered so that four consecutive ones
// fill one quad of cols.
template <int NKS, int NDT>
struct Tile3 {
  static constexpr int RP = 4 * (2 * NKS | 1);  // rows pitch (dwords)
  static constexpr int RPLANE = 32 * RP, CPLANE = 32 * NDT * 16;
  static constexpr int RSIZE = 3 * RPLANE, CSIZE = 3 * CPLANE;

  __device__ __forceinline__ static int pair_row(int jj) {
    return 16 * (jj >> 3) + 8 * ((jj >> 1) & 1) + 4 * ((jj >> 2) & 1) + 2 * (jj & 1);
  }
  // dword offset in a rows plane of d = 4q .. 4q + 3 of row r
  __device__ __forceinline__ static int rows_at(int r, int q) { return r * RP + 2 * q; }
  // dword offset in a cols plane of row pair jj of d = 4q + u
  __device__ __forceinline__ static int cols_at(int q, int u, int jj) {
    const int c = 2 * (jj >> 3) + ((jj >> 2) & 1);
    return (8 * NDT * u + q) * 16 + 4 * (c ^ (((q >> 2) ^ u) & 3)) + (jj & 3);
  }
  __device__ __forceinline__ static Frag3 read(const unsigned* p, int plane) {
    return Frag3{*reinterpret_cast<const bf16x8*>(p), *reinterpret_cast<const bf16x8*>(p + plane),
                 *reinterpret_cast<const bf16x8*>(p + 2 * plane)};
  }
  __device__ __forceinline__ static const unsigned* rows_ptr(const unsigned* t, int ks, int lane) {
    return t + (lane & 31) * RP + 4 * (2 * ks + (lane >> 5));
  }
  __device__ __forceinline__ static Frag3 rows_frag(const unsigned* t, int ks, int lane) {
    return read(rows_ptr(t, ks, lane), RPLANE);
  }
  // d = 32 dt + lane % 32
  __device__ __forceinline__ static const unsigned* cols_ptr(const unsigned* t, int dt, int ks, int lane) {
    const int d = 32 * dt + (lane & 31), q = d >> 2, u = d & 3;
    return t + (8 * NDT * u + q) * 16 + 4 * ((2 * ks + (lane >> 5)) ^ (((q >> 2) ^ u) & 3));
  }
  __device__ __forceinline__ static Frag3 cols_frag(const unsigned* t, int dt, int ks, int lane) {
    return read(cols_ptr(t, dt, ks, lane), CPLANE);
  }
};

// Staging registers of one operand tile for NT threads: G d-groups of 4.
template <int NKS, int NDT, int G, int NT, bool VEC>
struct TileLoad {
  using T3 = Tile3<NKS, NDT>;
  static constexpr int UNITS = 16 * G, PER = (UNITS + NT - 1) / NT;
  float v[PER][2][4];
  uint32_t off[PER];  // VEC: byte offset of the unit's first row at tile row 0

  __device__ __forceinline__ static int unit(int p, int tid) { return (tid + p * NT) % UNITS; }
  __device__ __forceinline__ void init(int64_t st, int D, int tid) {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int x = unit(p, tid), c = 4 * (x % G);
      // past the head dim: an offset past any descriptor's range reads as zero
      off[p] = c < D ? (uint32_t)(T3::pair_row(x / G) * st + c) * 4u : 0x80000000u;
    }
  }
  // Rows row0 .. row0+31 of the head's rows (zero past T and D).  VEC: through
  // the head's descriptor ((T-1)*st + D floats, below 2 GiB).
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rsrc, const float* base, int row0, int T, int D,
                                       int64_t st, int tid) {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      if (VEC) {
        const uint32_t o = off[p] + (uint32_t)(row0 * st) * 4u;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const float4 x = buffer_load_quad(rsrc, (int)(o + (uint32_t)(r * st) * 4u), 0);
          v[p][r][0] = x.x, v[p][r][1] = x.y, v[p][r][2] = x.z, v[p][r][3] = x.w;
        }
      } else {
        const int x = unit(p, tid), c = 4 * (x % G), r0 = row0 + T3::pair_row(x / G);
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v[p][r][e] = (r0 + r < T && c + e < D) ? base[(int64_t)(r0 + r) * st + c + e] : 0.f;
      }
    }
  }
  // Splits the units into the planes of one layout (COLS: cols, else rows), in
  // two pieces of five or six VALU operations per pair of elements (a pair is
  // what a packed register holds: two rows of one d, or two d of one row).
  struct Pending {  // parts of two pairs, not stored yet
    uintx2 h, m, l;
  };
  static constexpr int kPieces = PER * 8;
  template <bool COLS>
  __device__ __forceinline__ void store_piece(int j, Pending& w, unsigned* tile, int tid) {
    const int p = j / 8, k = (j >> 1) & 3;
    const int x = unit(p, tid), q = x % G, jj = x / G;
    float& a = COLS ? v[p][0][k] : v[p][k >> 1][2 * (k & 1)];
    float& b = COLS ? v[p][1][k] : v[p][k >> 1][2 * (k & 1) + 1];
    if ((j & 1) == 0) {
      if constexpr (NDT > 2) {  // not before: the load has until here (costs registers)
        pin(a);
        pin(b);
      }
      w.h[k & 1] = take_pair(a, b);
      return;
    }
    w.m[k & 1] = take_pair(a, b);
    w.l[k & 1] = bf16_pair(a, b);
    if (COLS) {
      unsigned* d = tile + T3::cols_at(q, k, jj);
      d[0] = w.h[k & 1];
      d[T3::CPLANE] = w.m[k & 1];
      d[2 * T3::CPLANE] = w.l[k & 1];
    } else if (k & 1) {
      static_assert(COLS || G == 4 * NKS, "a d-group per quad of a row");
      unsigned* d = tile + T3::rows_at(T3::pair_row(jj) + (k >> 1), q);
      *reinterpret_cast<uintx2*>(d) = w.h;
      *reinterpret_cast<uintx2*>(d + T3::RPLANE) = w.m;
      *reinterpret_cast<uintx2*>(d + 2 * T3::RPLANE) = w.l;
    }
  }
  template <bool COLS>
  __device__ __forceinline__ void store(unsigned* tile, int tid) {
    Pending w;
    run_pieces<0, kPieces>([&](auto j) { store_piece<COLS>(j, w, tile, tid); });
  }
};

// A wave's 32 rows as the other operand of contractions over the head
// dimension: lane l holds d = 16 ks + 8 (l/32) + j of row `row`, split (zero
// past T and D).
template <int NKS, bool VEC>
__device__ __forceinline__ void load_frags(const float* __restrict__ base, int row, int T, int D, int64_t st, int lane,
                                           Frag3 (&f)[NKS]) {
  const float* src = base + (int64_t)min(row, T - 1) * st;
  float x[NKS][8];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    const int c = 16 * ks + 8 * (lane >> 5);
    if (VEC) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row < T && c + 4 * h < D) v = *reinterpret_cast<const float4*>(src + c + 4 * h);
        x[ks][4 * h] = v.x, x[ks][4 * h + 1] = v.y, x[ks][4 * h + 2] = v.z, x[ks][4 * h + 3] = v.w;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[ks][j] = (row < T && c + j < D) ? src[c + j] : 0.f;
    }
  }
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) f[ks] = split_frag(x[ks]);
}

// Writes a lane's part of a result X^T[d][row] (d = 32 dt + acc_row(i, g)) to
// its row of a [T][D] tensor.
template <int NDT, bool VEC>
__device__ __forceinline__ void store_cols(float* __restrict__ dst, int D, int g, const floatx16 (&x)[NDT], float mul) {
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int c = 32 * dt + 8 * u + 4 * g;
      if (VEC) {
        if (c < D)
          *reinterpret_cast<float4*>(dst + c) = make_float4(x[dt][4 * u] * mul, x[dt][4 * u + 1] * mul,
                                                            x[dt][4 * u + 2] * mul, x[dt][4 * u + 3] * mul);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < D) dst[c + e] = x[dt][4 * u + e] * mul;
      }
    }
}

}  // namespace wha
