// Dispatch of the causal attention forward, and the Delta pass of the
// from-probabilities backward.
#include <type_traits>

#include "wha_launch.hpp"

namespace wha {

// Delta_t = sum_j att[t][j] (dO_t . V_j) for head dims 36..128 (multiples of 4,
// 128-bit-aligned operands; 48, 64 and 128 exact, others padded up to them), on
// fp32 MFMAs.  A wave forms dP^T = V dO^T (keys on MFMA rows, its 16 queries on
// columns) and each lane takes sum_j att[q][j] dP[q][j] over its keys: att as
// given, read one sub-tile ahead as 16-byte loads along the row (AV: T % 4 == 0
// and att 16-byte aligned), masked entries selected away; the row's -Delta goes
// into the stats blocks of attn_bwd_dkv_dma_kernel (0 in the -LSE half and past
// T).  32-key sub-tiles of V (16-key at DP = 128) go from global memory straight
// into LDS (global_load_lds, swizzled Lds<DP> layout, two slots in separate
// arrays, loop unrolled by two, one barrier per sub-tile).  A block handles query
// tiles p and n_qt-1-p (n_qt+1 key tiles of work for every block); grid =
// B*H*ceil(n_qt/2).
#ifndef WHA_FWD_WPE
#define WHA_FWD_WPE __attribute__((amdgpu_waves_per_eu(3)))
#endif
template <int DP, bool PADQ, bool AV>
__global__ __launch_bounds__(256) WHA_FWD_WPE void probs_delta_dma_kernel(const float* __restrict__ dO,
                                                                         const float* __restrict__ V,
                                                                         float* __restrict__ STATS, View L,
                                                                         int unpaired,
                                                                         const float* __restrict__ ATT) {
  constexpr int DG = DP / 4;
  constexpr int QPR = DP / 4;                      // quads per row
  constexpr int BSUB = DP == 48 ? 32 : 2048 / DP;  // keys per sub-tile (8 KB per operand; 6 KB at 48)
  constexpr int NKT = BSUB / 16;                   // 16-key groups per sub-tile
  constexpr int TILE = BSUB * DP;                  // floats per operand sub-tile
  // 64-quad DMA chunks per operand sub-tile: 8 (each wave fetches two of K
  // and two of V) or, at DP = 48, 6 (waves 0-1 fetch K, waves 2-3 V, three each)
  constexpr int CH = BSUB * QPR / 64;
  constexpr bool SPLIT = CH == 6;
  constexpr int NU = SPLIT ? 3 : 2;                // chunks per wave and operand it fetches
  using LT = Lds<DP, true>;
  static_assert((CH == 8 || SPLIT) && LT::SWZ, "sub-tiles of 512 or 384 quads in the swizzled unpadded layout");
  __shared__ __align__(16) float Vs0[TILE], Vs1[TILE];

  const int BH = L.B * L.H;
  const int bh = blockIdx.x % BH;
  const int pair = (int)(blockIdx.x / BH);
  const int n_qt = (L.T + 63) / 64;
  const int b = bh / L.H, h = bh % L.H;
  const int64_t base = (int64_t)b * L.sb + (int64_t)h * L.sh;
  const char* vg = reinterpret_cast<const char*>(V + base);
  const int64_t sub_bytes = (int64_t)BSUB * L.st * 4;
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int lq = lane & 15, g = lane >> 4;

  // this lane's fetch: wave w fills LDS chunk ch(u) = 2w+u (u < 2), or at DP =
  // 48 (six chunks) waves 0-1 three each: quad p = 64 ch + lane is row p / QPR,
  // stored position p % QPR <- logical quad pq_inv(row, p % QPR); byte offsets
  // from the sub-tile's first row
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  int rrow[NU], rcol[NU];
  uint32_t roff[NU];
  bool pad[NU];  // PADQ: this lane's quad lies past the head dim (fetched from g_zero_quad)
  auto chunk = [&](int u) { return SPLIT ? 3 * (wv & 1) + u : 2 * wv + u; };
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int p = 64 * chunk(u) + lane;
    rrow[u] = p / QPR;
    rcol[u] = LT::pq_inv(rrow[u], p % QPR);
    pad[u] = PADQ && 4 * rcol[u] >= L.D;
    roff[u] = (uint32_t)(rrow[u] * L.st + 4 * rcol[u]) * 4u;
  }
  auto fetch = [&](int st, float* Vd) {
    if (SPLIT && wv >= 2) return;
    const int k0 = st * BSUB;
    const char* vs = vg + st * sub_bytes;
    uint32_t off[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) off[u] = roff[u];
    if (k0 + BSUB > L.T) {  // last sub-tile: rows past T read row T-1
#pragma unroll
      for (int u = 0; u < NU; ++u)
        off[u] = (uint32_t)((min(k0 + rrow[u], L.T - 1) - k0) * L.st + 4 * rcol[u]) * 4u;
    }
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const float* vp = reinterpret_cast<const float*>(vs + off[u]);
      if (PADQ && pad[u]) vp = g_zero_quad;
      dma_quad(vp, Vd + 256 * chunk(u));
    }
  };

  // paired: query tiles n_qt-1-p and p (equal work per block); unpaired: one
  // tile per block, the longest first (grids too small to fill every slot)
  const int n_pass = (!unpaired && n_qt - 1 - pair != pair) ? 2 : 1;
  // sub-tiles this block sweeps, and how many it has left
  auto subs_of = [&](int qt) { return (min(L.T, (qt + 1) * 64) + BSUB - 1) / BSUB; };
  const int work = subs_of(n_qt - 1 - pair) + (n_pass == 2 ? subs_of(pair) : 0);
  int left = work;
  for (int pass = 0; pass < n_pass; ++pass) {
    const int qt = pass == 0 ? n_qt - 1 - pair : pair;  // the longer row of tiles first
    const int q0 = qt * 64 + wave * 16;                  // first query of this wave
    const int qrow = q0 + lq;                            // this lane's query
    float of[DG];
    load_row_frag_dma<DP>(dO + base, qrow, L.T, L.D, L.st, g, 1.f, of);
    const int n_sub = (min(L.T, (qt + 1) * 64) + BSUB - 1) / BSUB;
    const int key_last = min(qrow, L.T - 1);  // keys above it are masked
    // this lane's att row (clamped into the tensor; rows past T are never stored)
    const float* att_row = ATT + ((int64_t)bh * L.T + min(qrow, L.T - 1)) * L.T;
    float d_acc = 0.f;
    floatx4 atA[NKT], atB[NKT];  // att of the even / odd sub-tiles
    auto load_att = [&](int st, floatx4 (&dst)[NKT]) {
#pragma unroll
      for (int mt = 0; mt < NKT; ++mt) {
        const int c = st * BSUB + 16 * mt + 4 * g;  // keys c..c+3, clamped into the row (masked past it)
        if constexpr (AV) {
          dst[mt] = *reinterpret_cast<const floatx4*>(att_row + min(c, L.T - 4));
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) dst[mt][i] = att_row[min(c + i, L.T - 1)];
        }
      }
    };

    auto compute = [&](auto masked, int k0, const float* Vs, const floatx4 (&at)[NKT]) {
      constexpr bool MASKED = decltype(masked)::value;
      // dP^T[key][query]: MFMA rows are keys 16mt + lq, columns the wave's queries
      floatx4 s[NKT];
#pragma unroll
      for (int mt = 0; mt < NKT; ++mt) {
        WHA_FENCE();
        s[mt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < DG / 4; ++j) {
          const float4 a = lds_read_quad<DP, true>(Vs, 16 * mt + lq, dma48_quad<DP>(g, j));
          s[mt] = mfma4(a.x, of[4 * j + 0], s[mt]);
          s[mt] = mfma4(a.y, of[4 * j + 1], s[mt]);
          s[mt] = mfma4(a.z, of[4 * j + 2], s[mt]);
          s[mt] = mfma4(a.w, of[4 * j + 3], s[mt]);
        }
      }
      WHA_FENCE();
      // lane element (mt,i): dP of key k0 + 16mt + 4g + i and query qrow
#pragma unroll
      for (int mt = 0; mt < NKT; ++mt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float t = at[mt][i] * s[mt][i];
          d_acc += (MASKED && k0 + 16 * mt + 4 * g + i > key_last) ? 0.f : t;
        }
      }
    };

    // one sub-tile: wait for its loads, start the next one's, then consume it
    auto step = [&](int st, int nx, const float* Vs, float* Vn, const floatx4 (&at)[NKT], floatx4 (&at_next)[NKT]) {
      wait_vmem();
      __syncthreads();  // sub-tile st is in LDS; every wave is done with the previous one
      prio_by_remaining(left--, work);
      if (nx >= 0) {  // the next sub-tile of the sweep
        fetch(nx, Vn);
        load_att(nx, at_next);
      }
      const int k0 = st * BSUB;
      if (k0 > q0 + 15) return;  // every key follows every query of the wave
      if (k0 + BSUB - 1 <= q0 && k0 + BSUB <= L.T)
        compute(std::false_type{}, k0, Vs, at);
      else
        compute(std::true_type{}, k0, Vs, at);
    };

    // Sweep order: the first pass (the longer query tile) runs from key 0
    // forward, the second from its diagonal back to key 0, so the blocks of one
    // head read at most two distinct V sub-tiles at any time.
    auto st_at = [&](int j) { return pass == 0 ? j : n_sub - 1 - j; };
    __syncthreads();  // the previous pass's last sub-tile has been read by every wave
    fetch(st_at(0), Vs0);
    load_att(st_at(0), atA);
    for (int j = 0; j < n_sub; j += 2) {
      step(st_at(j), j + 1 < n_sub ? st_at(j + 1) : -1, Vs0, Vs1, atA, atB);
      if (j + 1 < n_sub) step(st_at(j + 1), j + 2 < n_sub ? st_at(j + 2) : -1, Vs1, Vs0, atB, atA);
    }

    // -Delta of the row into its stats block (rows past T within the block get 0)
    const float delta = pair_sum32(pair_sum16(d_acc));
    const int Tb = (L.T + 31) / 32 * 32;
    if (g == 0 && qrow < Tb) {
      float* blk = STATS + ((int64_t)bh * (Tb / 32) + qrow / 32) * 64 + qrow % 32;
      blk[0] = 0.f;
      blk[32] = qrow < L.T ? -delta : 0.f;
    }
  }
}

bool scores_kept(const View& L, bool vec) {
  return vec && kept_head_dim(L.D) && ds_head_fits(L) && !small_problem(L);
}

namespace {
template <int DP, bool PADQ, bool AV>
void probs_delta_t(const float* d_o, const float* v, const float* att, float* stats, const View& L,
                   hipStream_t stream) {
  const int unp = dma_unpaired(L);
  const dim3 grid((unsigned)(dma_tiles(L, unp) * L.B * L.H));
  hipLaunchKernelGGL((probs_delta_dma_kernel<DP, PADQ, AV>), grid, dim3(256), 0, stream, d_o, v, stats, L, unp, att);
}
}  // namespace

hipError_t launch_probs_delta_dma(const float* d_o, const float* v, const float* att, float* stats, const View& L,
                                  bool av, hipStream_t stream) {
  if (!dma_head_dim(L.D)) return hipErrorInvalidValue;
#define WHA_PD(DP, PADQ)                                                 \
  (av ? probs_delta_t<DP, PADQ, true>(d_o, v, att, stats, L, stream)   \
      : probs_delta_t<DP, PADQ, false>(d_o, v, att, stats, L, stream))
  if (L.D == 48)
    WHA_PD(48, false);
  else if (L.D < 48)
    WHA_PD(48, true);
  else if (L.D == 64)
    WHA_PD(64, false);
  else if (L.D < 64)
    WHA_PD(64, true);
  else if (L.D == 128)
    WHA_PD(128, false);
  else
    WHA_PD(128, true);
#undef WHA_PD
  return hipGetLastError();
}

hipError_t launch_attn_fwd(const float* q, const float* k, const float* v, float* o, float* lse,
                           const View& L, bool vec, float scale, hipStream_t stream, float* scores) {
  if (scores != nullptr && !scores_kept(L, vec)) return hipErrorInvalidValue;
  if (scores == nullptr && small_problem(L)) return launch_attn_fwd_small(q, k, v, o, lse, L, scale, stream);
  if (padded_dim(L.D) == 0) return hipErrorInvalidValue;
  return launch_attn_fwd_split(q, k, v, o, lse, scores, L, vec, scale, stream);
}

}  // namespace wha
