// Causal attention forward on the bf16 matrix cores at fp32 precision
// (wha_split.hpp): o = softmax(q k^T scale, causal) v and the row log-sum-exp,
// for every problem but the small ones (small_problem).
//
// A block takes NW x 32 consecutive queries of one (b,h) (NW = 4; 2 for short rows
// of wide heads, two_waves), a wave 32 of them: Q
// in registers (split, unscaled), 32-key tiles of K and V split by the whole
// block into two LDS buffers, one barrier per tile -- while a tile is consumed
// the next one is split into the other buffer and the one after it is loaded.
// A wave forms S^T = K Q^T (keys on MFMA rows, its queries on columns): a lane
// holds 16 keys of one query, its running maximum needs one cross-lane step, and
// P^T is the B operand of O^T += V^T P^T as it stands.
//
// S sums its five small products first, then the four (NKS) large ones, in one
// accumulator; scale*log2(e) is applied in the exponent.  Each tile's V^T P^T is
// likewise one accumulator from zero, added to O with its factor in one fused
// multiply-add per element (no branch that keeps a second copy of O).
//
// The low parts of an infinity are NaN, so a row that meets one comes out NaN
// here; rows whose result is not finite are formed again in fp32 at the end
// (again), which is where infinities, NaN and overflow get the values that the
// formula gives them.
//
// Bound by the matrix cores and the VALU beside them: per 32 x 32 tile and wave
// at head dim 64, 48 MFMAs (1536 cycles) and about 300 VALU issue slots (1200);
// the MFMAs are busy 45% of the time at the 2.0 GHz that the power leaves them.
// The softmax of a tile is therefore issued between the MFMAs of the next one's
// scores, the staging between those of O (interleave, wha_split.hpp).
//
// Forward alone, fp32 MFMA kernel (16 queries per wave, 64 per block) -> this
// one, us; and the relative error of O against 64 bits:
//   8 x 12 heads, 1024 x 64       114 -> 77      3.3e-7 -> 1.2e-7
//   16 x 8 heads, 512 x 48        39.3 -> 27.8   2.7e-7 -> 1.1e-7
//   4 x 32 heads, 2048 x 128      1071 -> 790    4.4e-7 -> 1.5e-7
//   3 x 10 heads, 1531 x 56       110 -> 68      3.7e-7 -> 1.3e-7
//   the same at head dim 50       133 -> 88      4.1e-7 -> 1.6e-7
//   4 x 16 heads, 700 x 96        100 -> 52      3.3e-7 -> 1.3e-7
//   8 x 8 heads, 600 x 32         38.1 -> 22.3   2.8e-7 -> 1.0e-7
//   2 x 32 heads, 333 x 100       41.5 -> 30.7   3.0e-7 -> 1.2e-7 (fewer blocks than CUs)
//   1 x 4 heads, 8192 x 64        428 -> 300     6.4e-7 -> 1.7e-7
// and keeping the scores (the figures at `save`).  It was the faster one at every
// head dim and length tried but for short rows of many heads (up to 64
// positions, 192 above head dim 96: the figures at two_waves; 512 heads of 40 x
// 64 9.0 -> 10.1), so the other, with three times the error, is gone.
#include <type_traits>

#include "wha_launch.hpp"
#include "wha_split.hpp"

namespace wha {

// The rows q0 .. q0 + 31 of a head marked in `bad` once more in fp32, straight
// from memory, by one wave: S^T and O^T on the fp32 MFMA in the layout of the
// kernel below, the maximum of each row first (an online one would meet
// -infinity - -infinity), then probabilities and O.  On the last tile some keys
// follow some queries: there a probability of zero must not meet an infinite
// value, so its keys are added one at a time to the queries that they precede.
// All rows NaN or infinite, the whole forward, us: 8 x 12 heads of 1024 x 64 630
// (one row after another on the VALU 24600; finite 90), 16 x 8 of 512 x 48 231
// (4870; 35), 4 x 8 of 2048 x 128 2040 (71000; 209).
template <int NKS, int NDT, bool VEC, bool SAVE>
__device__ __forceinline__ void again(const float* Qb, const float* Kb, const float* Vb, float* Ob, float* lse,
                                      __amdgpu_buffer_rsrc_t rsc, int q0, uint32_t bad, const View& L, float sl2,
                                      int lane) {
  pin(lane);  // addresses formed from it here, not held in registers since the main loop
  const int g = lane >> 5, c = lane & 31, qrow = q0 + c, t = min(qrow, L.T - 1), n_w = q0 / 32 + 1;
  const bool mine = (bad >> c) & 1;
  // d = 8j + 4g + e of a row (zero past the head dim): k-slot g of MFMA (j, e)
  auto quad = [&](const float* row, int j, float (&x)[4]) {
    const int d = 8 * j + 4 * g;
    if (VEC) {
      const float4 y = d < L.D ? *reinterpret_cast<const float4*>(row + d) : make_float4(0.f, 0.f, 0.f, 0.f);
      x[0] = y.x, x[1] = y.y, x[2] = y.z, x[3] = y.w;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = d + e < L.D ? row[d + e] : 0.f;
    }
  };
  float qf[2 * NKS][4];
#pragma unroll
  for (int j = 0; j < 2 * NKS; ++j) {
    quad(Qb + (int64_t)t * L.st, j, qf[j]);
#pragma unroll
    for (int e = 0; e < 4; ++e) qf[j][e] *= sl2;
  }
  // scores of the keys k0 + acc_row(i, g), log2 units
  auto scores = [&](int k0) {
    const float* row = Kb + (int64_t)min(k0 + c, L.T - 1) * L.st;
    floatx16 s = zero16();
#pragma unroll
    for (int j = 0; j < 2 * NKS; ++j) {
      float x[4];
      quad(row, j, x);
#pragma unroll
      for (int e = 0; e < 4; ++e) s = mfma_f32(x[e], qf[j][e], s);
    }
    return s;
  };
  auto masked = [&](int k0, int i) { return k0 + acc_row(i, g) > t; };
  float m = -INFINITY;
  for (int kt = 0; kt < n_w; ++kt) {
    const int k0 = kt * 32;
    const floatx16 s = scores(k0);
    if constexpr (SAVE) {
      const int at = (int)(((ds_block_row(k0 >> 6, L.T) - (k0 & ~63) + qrow) * 64 + (k0 & 63) + 4 * g) * 4);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        floatx4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = s[4 * u + e] / sl2;
        buffer_store_quad(rsc, x, mine ? at + 32 * u : (int)0x80000000, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) m = masked(k0, i) ? m : vmax2(m, s[i]);
  }
  m = pair_max32(m);
  float l = 0.f;
  floatx16 o[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) o[dt] = zero16();
  for (int kt = 0; kt + 1 < n_w; ++kt) {
    floatx16 p = scores(kt * 32);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      p[i] = fast_exp2(p[i] - m);
      l += p[i];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float* v = Vb + (int64_t)(kt * 32 + acc_row(i, g)) * L.st;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) o[dt] = mfma_f32(32 * dt + c < L.D ? v[32 * dt + c] : 0.f, p[i], o[dt]);
    }
  }
  const int k0 = (n_w - 1) * 32;
  floatx16 p = scores(k0);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    p[i] = fast_exp2(p[i] - m);
    l += masked(k0, i) ? 0.f : p[i];
  }
#pragma unroll 1
  for (int x = 0; x < 32 && k0 + x < L.T; ++x) {  // key x = acc_row(i, h)
    const int i = 4 * (x >> 3) + (x & 3), h = (x >> 2) & 1;
    float px = p[0];
#pragma unroll
    for (int j = 1; j < 16; ++j) px = j == i ? p[j] : px;
    px = __shfl(px, c + 32 * h, 64);
    const float* v = Vb + (int64_t)(k0 + x) * L.st;
    if (k0 + x <= t) {
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int y = 0; y < 16; ++y) {
          const int d = 32 * dt + acc_row(y, g);
          if (d < L.D) o[dt][y] = fmaf(px, v[d], o[dt][y]);
        }
    }
  }
  l = pair_sum32(l);
  if (mine) {
    store_cols<NDT, VEC>(Ob + (int64_t)qrow * L.st, L.D, g, o, 1.f / l);
    if (lse != nullptr && g == 0) lse[qrow] = fmaf(m, kLn2, logf(l));
  }
}

// SAVE: also keeps the raw scores q.k of every tile it computes in SC (the
// layout of the backward's dS workspace, ds_block_row; entries after the
// diagonal hold whatever the tile gave, the backward masks them).
template <int NKS, int NDT, int NW, bool VEC, bool SAVE>
__global__ __launch_bounds__(NW * 64, NDT <= 2 ? 2 : 1) void attn_fwd_split_kernel(
    const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V, float* __restrict__ O,
    float* __restrict__ LSE, float* __restrict__ SC, View L, float sl2) {
  using T3 = Tile3<NKS, NDT>;
  constexpr int NT = NW * 64, BM = NW * 32;
  // two waves at the widest head dim: one buffer of V, so that two blocks fit a CU
  constexpr bool V_TWO = !(NW == 2 && NDT == 4);
  __shared__ __align__(16) unsigned K0[T3::RSIZE], K1[T3::RSIZE], V0[T3::CSIZE], V1[V_TWO ? T3::CSIZE : 4];

  const int BH = L.B * L.H;
  const int n_qt = (L.T + BM - 1) / BM;
  const int bh = blockIdx.x % BH;  // B*H a multiple of 8: a head's blocks share an XCD's L2
  // The longest rows of tiles first.  Where every block is resident at once, two
  // to a CU, the later ones from the shortest up: a CU's pair then has about the
  // same work everywhere (16 x 8 heads of 512 x 48: 30.2 -> 29.2 us, kept
  // 36.5 -> 35.4).
  const int j = (int)(blockIdx.x / BH), j0 = (256 + BH - 1) / BH;
  const int qt = NDT <= 2 && n_qt * BH <= 512 && j >= j0 ? j - j0 : n_qt - 1 - j;
  const int b = bh / L.H, h = bh % L.H;
  const int64_t base = (int64_t)b * L.sb + (int64_t)h * L.sh;
  const float* Kb = K + base;
  const float* Vb = V + base;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q0 = qt * BM + wave * 32, qrow = q0 + (lane & 31);

  const uint32_t bytes = VEC ? (uint32_t)(((int64_t)(L.T - 1) * L.st + L.D) * 4) : 0u;
  const __amdgpu_buffer_rsrc_t rk = buffer_rsrc(Kb, bytes), rv = buffer_rsrc(Vb, bytes);
  const int64_t sc_rows = ds_rows(L.T);
  const __amdgpu_buffer_rsrc_t rsc = buffer_rsrc(SAVE ? SC + (int64_t)bh * sc_rows * 64 : Q,
                                                 SAVE ? (uint32_t)(sc_rows * 256) : 0u);
  const int Tp = (L.T + 63) / 64 * 64;

  const int n_kt = (min(L.T, (qt + 1) * BM) + 31) / 32;  // tiles the block sweeps
  const int n_w = min(n_kt, q0 / 32 + 1);                // tiles with a key before some query of the wave
  TileLoad<NKS, NDT, 4 * NKS, NT, VEC> kl;
  TileLoad<NKS, NDT, 8 * NDT, NT, VEC> vl;
  if (VEC) {
    kl.init(L.st, L.D, tid);
    vl.init(L.st, L.D, tid);
  }
  // tile kt of K / V into the registers (past the last one: the last again, never used)
  auto load_k = [&](int kt) { kl.load(rk, Kb, min(kt, n_kt - 1) * 32, L.T, L.D, L.st, tid); };
  auto load_v = [&](int kt) { vl.load(rv, Vb, min(kt, n_kt - 1) * 32, L.T, L.D, L.st, tid); };
  auto store_k = [&](unsigned* Kd) { kl.template store<false>(Kd, tid); };
  auto store_v = [&](unsigned* Vd) { vl.template store<true>(Vd, tid); };
  Frag3 qf[NKS];
  load_k(0);
  load_v(0);
  load_frags<NKS, VEC>(Q + base, qrow, L.T, L.D, L.st, lane, qf);
  store_k(K0);
  load_k(1);
  __syncthreads();
  store_k(K1);
  load_k(2);
  store_v(V0);
  load_v(1);

  // running maximum m (log2 units; finite from the first tile on, whose key 0
  // comes before every query), this lane's part of the row sum, O
  float m = -INFINITY, l = 0.f;
  floatx16 o[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) o[dt] = zero16();
  floatx16 s;

  // The scores of a tile against the wave's queries: MFMA i of 6 NKS, the small
  // products of every k-step, then the large ones.
  constexpr int NMS = 6 * NKS, NMO = 12 * NDT;
  auto score_step = [&](auto ic, const unsigned* Ks, Frag3 (&kf)[NKS], floatx16& acc) {
    constexpr int i = decltype(ic)::value;
    if constexpr (i < 5 * NKS) {
      constexpr int ks = i / 5, e = i % 5;
      if constexpr (e == 1 && ks + 1 < NKS) kf[ks + 1] = T3::rows_frag(Ks, ks + 1, lane);
      acc = mfma_small_step(e, kf[ks], qf[ks], acc);
    } else {
      acc = mfma_bf16(kf[i - 5 * NKS].h, qf[i - 5 * NKS].h, acc);
    }
  };
  {
    Frag3 kf[NKS];
    kf[0] = T3::rows_frag(K0, 0, lane);
    s = zero16();
    run_pieces<0, NMS>([&](auto i) { score_step(i, K0, kf, s); });
  }

  // Tile kt, whose scores s are there: softmax and O.  NEXT: with the scores of
  // tile kt + 1, whose MFMAs run beside the softmax of tile kt; the staging of
  // K tile kt + 2 and V tile kt + 1 runs beside the MFMAs of O.  The last tile
  // of a wave is the only one with keys past a query or the end.
  auto tile = [&](auto next, int kt, const unsigned* Kn, const unsigned* Vs, unsigned* Kst, unsigned* Vst) {
    constexpr bool NEXT = decltype(next)::value;
    const int k0 = kt * 32;
    // SAVE: quad pair x of the tile's scores (4), among the MFMAs of the next
    // one's.  A lane's four quads of 16 bytes lie 32 bytes apart; swapped with
    // the lane 16 on, four lanes hold 64 contiguous bytes of one row (kept
    // forward and backward of 16 x 8 heads of 512 x 48: 128.8 -> 126.0 us).
    // Rows past the padded length: an offset past the descriptor, not a branch --
    // where a store may have been stepped over the compiler waits for all stores
    // at the next use of a load.  Kept forward, stores under branches before the
    // MFMAs -> this, us: 4 x 4 heads of 1500 x 48 77.2 -> 65.0, 1 x 2 of 2000 x
    // 64 103.6 -> 86.4, 1 x 4 of 8192 x 64 433 -> 380, 4 x 32 of 2048 x 128
    // 943 -> 895, 8 x 12 of 1024 x 64 99.5 -> 100.2 (+-3).
    int at_lo = 0, at_hi = 0;
    floatx4 lo, hi;  // rows r0 and r0 + 16, keys 16u .. 16u + 15
    auto save = [&](auto xc) {
      constexpr int x = decltype(xc)::value, u = x >> 1;
      if constexpr (x == 0) {
        const int c = k0 >> 6, r0 = q0 + (lane & 15);
        const int at =
            (int)(((ds_block_row(c, L.T) - (int64_t)64 * c + r0) * 64 + (k0 & 63) + 8 * ((lane >> 4) & 1) + 4 * g) * 4);
        at_lo = r0 < Tp ? at : (int)0x80000000;
        at_hi = r0 + 16 < Tp ? at + 16 * 256 : (int)0x80000000;
      }
#pragma unroll
      for (int e = 2 * (x & 1); e < 2 * (x & 1) + 2; ++e) {
        const auto y = __builtin_amdgcn_permlane16_swap(__float_as_uint(s[8 * u + e]),
                                                        __float_as_uint(s[8 * u + 4 + e]), false, false);
        lo[e] = __uint_as_float(y[0]);
        hi[e] = __uint_as_float(y[1]);
      }
      if constexpr (x & 1) {
        buffer_store_quad(rsc, lo, at_lo + 64 * u, 0);
        buffer_store_quad(rsc, hi, at_hi + 64 * u, 0);
      }
    };
    constexpr int NPW = SAVE ? 4 : 0;
    if constexpr (SAVE && !NEXT) run_pieces<0, NPW>(save);
    if constexpr (!NEXT) {
      const int key_last = min(qrow, L.T - 1);
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = k0 + acc_row(i, g) > key_last ? -INFINITY : s[i];
    }
    // softmax in pieces: the maximum, then pairs of probabilities and their split
    float mx = 0.f, alpha = 0.f, sum = 0.f, p[16];
    uintx4 ph[2], pm[2], pl[2];
    auto softmax = [&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if constexpr (j == 0) {
        mx = vmax3(vmax3(vmax3(s[0], s[1], s[2]), s[3], s[4]), vmax3(s[5], s[6], s[7]), s[8]);
      } else if constexpr (j == 1) {
        mx = vmax3(vmax3(vmax3(mx, s[9], s[10]), s[11], s[12]), vmax3(s[13], s[14], s[15]), s[15]);
      } else if constexpr (j == 2) {
        mx = vmax2(m, pair_max32(mx) * sl2);
        alpha = fast_exp2(m - mx);
        m = mx;
      } else if constexpr (j < 19) {
        constexpr int k = (j - 3) >> 1;
        if constexpr (((j - 3) & 1) == 0) {
          p[2 * k] = fast_exp2(fmaf(s[2 * k], sl2, -m));
          p[2 * k + 1] = fast_exp2(fmaf(s[2 * k + 1], sl2, -m));
          pin(p[2 * k]);
          pin(p[2 * k + 1]);
        } else {
          sum += p[2 * k] + p[2 * k + 1];
          pin(sum);
          const SplitPair x = split_pair(p[2 * k], p[2 * k + 1]);
          unsigned xh = x.h, xm = x.m, xl = x.l;
          pin(xh);
          pin(xm);
          pin(xl);
          ph[k >> 2][k & 3] = xh;
          pm[k >> 2][k & 3] = xm;
          pl[k >> 2][k & 3] = xl;
        }
      } else {
        l = fmaf(l, alpha, sum);
      }
    };
    constexpr int NPS = 20;
    floatx16 sn;
    if constexpr (NEXT) {
      Frag3 kf[NKS];
      kf[0] = T3::rows_frag(Kn, 0, lane);
      sn = zero16();
      run_pieces<0, 2>(softmax);
      WHA_FENCE();
      interleave<NMS, NPS - 2 + NPW>(
          [&](auto i) {
            score_step(i, Kn, kf, sn);
            pin(sn);
          },
          [&](auto jc) {
            constexpr int j = decltype(jc)::value;
            if constexpr (j < NPW)
              save(jc);
            else
              softmax(std::integral_constant<int, j - NPW + 2>{});
          });
    } else {
      run_pieces<0, NPS>(softmax);
    }
    Frag3 pf[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      pf[ks] = Frag3{__builtin_bit_cast(bf16x8, ph[ks]), __builtin_bit_cast(bf16x8, pm[ks]),
                     __builtin_bit_cast(bf16x8, pl[ks])};
    // O^T[d][query] = alpha O^T + V^T P^T: per d-tile the small products of both
    // k-steps, then the large ones
    Frag3 vf[2 * NDT];
    vf[0] = T3::cols_frag(Vs, 0, 0, lane);
    floatx16 t[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) t[dt] = zero16();
    typename decltype(kl)::Pending kw;
    typename decltype(vl)::Pending vw;
    constexpr int PK = decltype(kl)::kPieces, PV = decltype(vl)::kPieces;
    interleave<NMO, PK + 1 + (V_TWO ? PV + 1 : 0)>(
        [&](auto ic) {
          constexpr int i = decltype(ic)::value, dt = i / 12, e = i % 12;
          if (e == 1) vf[2 * dt + 1] = T3::cols_frag(Vs, dt, 1, lane);
          if constexpr (e == 6 && dt + 1 < NDT) vf[2 * dt + 2] = T3::cols_frag(Vs, dt + 1, 0, lane);
          if constexpr (e < 10)
            t[dt] = mfma_small_step(e % 5, vf[2 * dt + e / 5], pf[e / 5], t[dt]);
          else
            t[dt] = mfma_bf16(vf[2 * dt + e - 10].h, pf[e - 10].h, t[dt]);
          pin(t[dt]);
          // the d-tile before, four elements per MFMA
          if constexpr (dt > 0 && e >= 2 && e < 6) {
#pragma unroll
            for (int x = 4 * (e - 2); x < 4 * (e - 1); ++x) o[dt - 1][x] = fmaf(o[dt - 1][x], alpha, t[dt - 1][x]);
          }
        },
        [&](auto jc) {
          constexpr int j = decltype(jc)::value;
          if constexpr (j < PK)
            kl.template store_piece<false>(j, kw, Kst, tid);
          else if constexpr (j == PK)
            load_k(kt + 3);
          else if constexpr (j < PK + 1 + PV)
            vl.template store_piece<true>(j - PK - 1, vw, Vst, tid);
          else
            load_v(kt + 2);
        });
#pragma unroll
    for (int x = 0; x < 16; ++x) o[NDT - 1][x] = fmaf(o[NDT - 1][x], alpha, t[NDT - 1][x]);
    if constexpr (NEXT) s = sn;
  };
  auto step = [&](int kt, const unsigned* Kn, const unsigned* Vs, unsigned* Kst, unsigned* Vst) {
    __syncthreads();  // K tile kt + 1 and V tile kt are in LDS; every wave is done with the other buffers
    if (kt + 1 < n_w) {
      tile(std::true_type{}, kt, Kn, Vs, Kst, Vst);
    } else if (kt < n_w) {
      tile(std::false_type{}, kt, Kn, Vs, Kst, Vst);
    } else {  // every key follows every query of the wave
      store_k(Kst);
      load_k(kt + 3);
      if constexpr (V_TWO) {
        store_v(Vst);
        load_v(kt + 2);
      }
    }
    if constexpr (!V_TWO) {
      if (kt + 1 < n_kt) {
        __syncthreads();  // every wave is done with V tile kt
        store_v(Vst);
        load_v(kt + 2);
      }
    }
  };
  for (int kt = 0; kt < n_kt; kt += 2) {
    step(kt, K1, V0, K0, V_TWO ? V1 : V0);
    if (kt + 1 < n_kt) step(kt + 1, K0, V_TWO ? V1 : V0, K1, V0);
  }

  const float l_sum = pair_sum32(l);
  float chk = 0.f * l_sum;  // NaN if the row's sum or any of its O is not finite
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int x = 0; x < 16; ++x) chk = fmaf(o[dt][x], 0.f, chk);
  const bool ok = chk == 0.f;
  if (qrow < L.T && ok) {
    store_cols<NDT, VEC>(O + base + (int64_t)qrow * L.st, L.D, g, o, 1.f / l_sum);
    if (LSE != nullptr && g == 0) LSE[(int64_t)bh * L.T + qrow] = fmaf(m, kLn2, logf(l_sum));
  }
  const uint64_t bad = __builtin_amdgcn_ballot_w64(qrow < L.T && !ok);
  if (bad != 0) {
    wait_vmem();  // the kept scores of these rows are written once more
    again<NKS, NDT, VEC, SAVE>(Q + base, Kb, Vb, O + base, LSE == nullptr ? nullptr : LSE + (int64_t)bh * L.T, rsc, q0,
                               (uint32_t)(bad | (bad >> 32)), L, sl2, lane);
  }
}

namespace {
template <int NKS, int NDT, int NW>
void fwd_t(const float* q, const float* k, const float* v, float* o, float* lse, float* sc, const View& L, bool vec,
           float sl2, hipStream_t stream) {
  const dim3 grid((unsigned)((int64_t)((L.T + 32 * NW - 1) / (32 * NW)) * L.B * L.H));
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(64 * NW), 0, stream, q, k, v, o, lse, sc, L, sl2);
  };
  if constexpr (NW == 4) {  // (two waves: 128-bit loads only)
    if (!vec)
      return sc != nullptr ? launch(attn_fwd_split_kernel<NKS, NDT, NW, false, true>)
                           : launch(attn_fwd_split_kernel<NKS, NDT, NW, false, false>);
  }
  sc != nullptr ? launch(attn_fwd_split_kernel<NKS, NDT, NW, true, true>)
                : launch(attn_fwd_split_kernel<NKS, NDT, NW, true, false>);
}
// Head dims above 64, where a CU holds one block of four waves: blocks of two
// waves (64 queries, two blocks a CU) for short rows that fill more than one
// round of four-wave blocks -- up to 256 positions, above head dim 96 only
// where they spare the empty half of a 128-query block.  Kept forward, us, the
// former fp32 MFMA kernel / four waves / two, at head dim 80: 512 heads of 40
// 11.7 / 18.4 / 12.4, 352 of 123 27.6 / 28.1 / 26.8, 320 of 130 37.6 / 42.0 /
// 31.5, 288 of 256 60.0 / 50.8 / 46.6; not 256 of 128 (one round) 20.1 / 16.7 /
// 17.9, 160 of 384 65.9 / 45.6 / 46.2, 40 of 1000 137 / 72 / 78.  At 128: 512 of
// 40 13.1 / 23.4 / 16.9, 320 of 130 39.0 / 51.2 / 42.2; not 352 of 123 29.0 /
// 34.3 / 37.4, 288 of 200 60.8 / 58.6 / 60.8.
bool two_waves(const View& L) {
  if ((int64_t)((L.T + 127) / 128) * L.B * L.H <= 256) return false;
  return L.D <= 96 ? L.T <= 256 : L.T <= 192 && (L.T - 1) % 128 < 64;
}
}  // namespace

hipError_t launch_attn_fwd_split(const float* q, const float* k, const float* v, float* o, float* lse, float* sc,
                                 const View& L, bool vec, float scale, hipStream_t stream) {
  // 32-bit byte offsets within a head's rows, the last tile's rows past T
  // included; otherwise the 64-bit element loads
  vec = vec && L.D % 4 == 0 && ((int64_t)L.T + 32) * L.st * 4 < ((int64_t)1 << 31);
  const float sl2 = (float)((double)scale * 1.4426950408889634);
  TimingScope ts("attn_fwd", stream);
  if (L.D <= 32)
    fwd_t<2, 1, 4>(q, k, v, o, lse, sc, L, vec, sl2, stream);
  else if (L.D <= 48)
    fwd_t<3, 2, 4>(q, k, v, o, lse, sc, L, vec, sl2, stream);
  else if (L.D <= 64)
    fwd_t<4, 2, 4>(q, k, v, o, lse, sc, L, vec, sl2, stream);
  else if (L.D <= 96)
    vec && two_waves(L) ? fwd_t<6, 3, 2>(q, k, v, o, lse, sc, L, vec, sl2, stream)
                         : fwd_t<6, 3, 4>(q, k, v, o, lse, sc, L, vec, sl2, stream);
  else
    vec && two_waves(L) ? fwd_t<8, 4, 2>(q, k, v, o, lse, sc, L, vec, sl2, stream)
                         : fwd_t<8, 4, 4>(q, k, v, o, lse, sc, L, vec, sl2, stream);
  return hipGetLastError();
}

}  // namespace wha
