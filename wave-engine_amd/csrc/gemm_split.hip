// The projections' GEMMs on the bf16 matrix cores, at fp32 precision: each fp32
// product as six bf16 ones (wha_split.hpp).  C[m][n] = bias[n] + sum_k A(m,k)
// B(k,n) with A and B given by strides, so the same kernel serves y = X W^T + b,
// dX = dY W and dW = dY^T X (reference: linear.hip).
//
// Output tiles of 128 x 128, 64 x 128, 128 x 64 or 64 x 64 per 256-thread block
// (gemm_pick); k stages staged through registers, where each element is split
// once, into two LDS buffers.  Split-K writes per-split partial tiles that
// gemm_reduce sums in a fixed order (deterministic).
//
// Bound by the matrix cores and their power: at M = 8192 with N = K = 4096 the
// kernel runs 196 TFLOP/s of fp32 products (1180 of bf16 ones; MFMA busy 65% at
// the 1.75 GHz the card then holds, where a bare loop of bf16 MFMAs on random
// data reaches 1900) against 139 of the fp32 MFMA kernels; its error against 64
// bits is a third of theirs (4.0e-7 against 1.1e-6; K = 768 1.6e-7 against
// 5.0e-7).
#include "wha_gemm.hpp"
#include "wha_split.hpp"

namespace wha {

// One operand's part of a k stage.  The k range is walked in stages of 32 and
// each stage in two sub-stages of 16: sub-stage s holds k = 8j + 4s + i
// (j, i < 4) of the stage at its slots 4j + i, so that 16-byte pieces of a
// k-contiguous operand serve both.  Element (r, k) of the source is
// p[r*s_r + k*s_k], contiguous along k (KC) or along r.
//
// Per sub-stage a thread holds RU rows x KU k: KC one float4 (k = 8j + 4s + i,
// j = tid % 4) of each of the rows tid/4 + 64u; otherwise the rows RU*q + u
// (q = tid / 8) of the two k at slots 2(tid % 8), one 128-bit (64 rows: 64-bit)
// load each.  It splits what it holds into three bf16 planes in LDS and at
// once loads the same piece of the stage after next.  (With two rows x 4 k in
// four 64-bit loads the weight gradients were bound by load instructions:
// 768 x 768 over 8192 rows 96 us against 73.)
//
// LDS plane: [ROWS][16] bf16, 32-byte rows of two quads (8 slots each); quad c
// of the row at position rho is stored at quad c ^ f.  KC: rho is the row, f =
// rho>>3 & 1; otherwise row RU*q + u sits at rho = 32u + (q + 2u) % 32 (64
// rows: 32u + q) with f = u & 1.  The operand reads (lane l: row l%32 of 32,
// quad l/32) then meet 16 different quads in each set of 16 lanes the LDS
// serves together, and the stores fill whole runs of rows: no bank-conflict
// cycles.
template <int ROWS, bool KC>
struct SplitStage {
  static constexpr int PLANE = ROWS * 8;  // dwords per plane
  static constexpr int SIZE = 3 * PLANE;  // dwords per sub-stage
  static constexpr int RU = KC ? ROWS / 64 : ROWS / 32, KU = KC ? 4 : 2;
  static_assert(ROWS == 64 || ROWS == 128, "a sub-stage splits evenly over 256 threads");
  float v[2][RU * KU];  // [sub-stage][row][k] (KC) or [k][row]
  int off[KC ? RU : 1];  // VEC: byte offset of the thread's piece at k = 0

  __device__ __forceinline__ static int quad(int r, int c) {  // dword offset of quad c of row r
    int rho = r, f = (r >> 3) & 1;
    if (!KC) {
      const int u = r % RU, q = r / RU;
      rho = 32 * u + (RU == 4 ? (q + 2 * u) & 31 : q);
      f = u & 1;
    }
    return rho * 8 + 4 * (c ^ f);
  }
  __device__ __forceinline__ static int row(int tid, int u) { return KC ? (tid >> 2) + 64 * u : RU * (tid >> 3) + u; }
  // k of the thread's first element within the stage, sub-stage 0
  __device__ __forceinline__ static int kpos(int tid) {
    return KC ? 8 * (tid & 3) : 8 * ((tid & 7) >> 1) + 2 * (tid & 1);
  }

  // Rows past the extent read the last ones; they feed outputs that are never stored.
  __device__ __forceinline__ void init(int64_t s_r, int64_t s_k, int r0, int R, int tid) {
    if (KC) {
#pragma unroll
      for (int u = 0; u < RU; ++u) off[u] = (int)(((int64_t)min(r0 + row(tid, u), R - 1) * s_r + kpos(tid)) * 4);
    } else {
      off[0] = (int)((min(r0 + row(tid, 0), R - RU) + (int64_t)kpos(tid) * s_k) * 4);
    }
  }

  // Sub-stage s of the stage at k0.  VEC: aligned pieces through the operand's
  // buffer descriptor (gemm_vec_ok), k past k_end reading as zero (a lane offset
  // past the descriptor's range; the offset that all lanes share stays on a row
  // of the operand, K its rows).  A piece lies in k where the operand is
  // contiguous along it (K is a multiple of four then), else within one k.
  // Otherwise one predicated load per element.
  template <bool VEC>
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rsrc, const float* p, int64_t s_r, int64_t s_k, int r0,
                                       int R, int k0, int s, int k_end, int K, int tid) {
    const int k = k0 + 4 * s + kpos(tid);
    if (VEC) {
      if (KC) {
#pragma unroll
        for (int u = 0; u < RU; ++u) {
          const float4 x = buffer_load_quad(rsrc, k >= k_end ? (int)0x80000000 : off[u], (k0 + 4 * s) * 4);
          v[s][4 * u + 0] = x.x, v[s][4 * u + 1] = x.y, v[s][4 * u + 2] = x.z, v[s][4 * u + 3] = x.w;
        }
      } else {
#pragma unroll
        for (int i = 0; i < KU; ++i) {
          const int vo = k + i >= k_end ? (int)0x80000000 : off[0];
          const int so = (int)(min(k0 + 4 * s + i, K - 1) * s_k * 4);
          if constexpr (RU == 4) {
            const float4 x = buffer_load_quad(rsrc, vo, so);
            v[s][4 * i + 0] = x.x, v[s][4 * i + 1] = x.y, v[s][4 * i + 2] = x.z, v[s][4 * i + 3] = x.w;
          } else {
            const uintx2 x = __builtin_bit_cast(uintx2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, vo, so, 0));
            v[s][RU * i] = __uint_as_float(x.x), v[s][RU * i + 1] = __uint_as_float(x.y);
          }
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < RU; ++u) {
        const int r = r0 + row(tid, u);
#pragma unroll
        for (int i = 0; i < KU; ++i)
          v[s][KC ? KU * u + i : RU * i + u] =
              (r < R && k + i < k_end) ? p[(int64_t)r * s_r + (int64_t)(k + i) * s_k] : 0.f;
      }
    }
  }

  __device__ __forceinline__ void store(unsigned* lds, int s, int tid) const {
#pragma unroll
    for (int u = 0; u < RU; ++u) {
      if (KC) {
        const int j = tid & 3, at = quad(row(tid, u), j >> 1) + 2 * (j & 1);
        const SplitPair a = split_pair(v[s][4 * u], v[s][4 * u + 1]), b = split_pair(v[s][4 * u + 2], v[s][4 * u + 3]);
        *reinterpret_cast<uintx2*>(lds + at) = uintx2{a.h, b.h};
        *reinterpret_cast<uintx2*>(lds + PLANE + at) = uintx2{a.m, b.m};
        *reinterpret_cast<uintx2*>(lds + 2 * PLANE + at) = uintx2{a.l, b.l};
      } else {
        const int j = tid & 7, at = quad(row(tid, u), j >> 2) + (j & 3);
        const SplitPair a = split_pair(v[s][u], v[s][RU + u]);
        lds[at] = a.h;
        lds[PLANE + at] = a.m;
        lds[2 * PLANE + at] = a.l;
      }
    }
  }

  // Sum of this thread's elements of sub-stage s per row (not KC).
  __device__ __forceinline__ void add_to(float (&rs)[4], int s, bool take) const {
#pragma unroll
    for (int u = 0; u < RU; ++u) rs[u] += take ? v[s][u] + v[s][RU + u] : 0.f;
  }

  // MFMA operand of rows row0 .. row0+31, slots 8*(lane/32) + j.
  __device__ __forceinline__ static Frag3 frag(const unsigned* lds, int row0, int lane) {
    const unsigned* q = lds + quad(row0 + (lane & 31), lane >> 5);
    return Frag3{*reinterpret_cast<const bf16x8*>(q), *reinterpret_cast<const bf16x8*>(q + PLANE),
                 *reinterpret_cast<const bf16x8*>(q + 2 * PLANE)};
  }
};

// BM x BN output tile per 256-thread block, WM x WN waves.  One barrier per
// sub-stage: while sub-stage t is multiplied out of one LDS buffer, sub-stage
// t+1 is split into the other one and sub-stage t+3 is loaded into the
// registers that held it.  MFMA rows are output columns n, MFMA columns output
// rows m, so a lane ends with runs of four consecutive n of one row: 128-bit
// stores.  VEC: both operands' pieces are 16-byte aligned (gemm_vec_ok).
template <int BM, int BN, int WM, int WN, bool A_KC, bool B_KC, bool VEC, bool PARTIAL>
__global__ __launch_bounds__(256, 2) void gemm_split_kernel(GemmArgs g) {
  static_assert(WM * WN == 4 && BM % (32 * WM) == 0 && BN % (32 * WN) == 0, "four waves of 32 x 32 MFMA tiles");
  using SA = SplitStage<BM, A_KC>;
  using SB = SplitStage<BN, B_KC>;
  constexpr int NT = BN / WN / 32, MT = BM / WM / 32;
  __shared__ __align__(16) unsigned As0[SA::SIZE], As1[SA::SIZE];
  __shared__ __align__(16) unsigned Bs0[SB::SIZE], Bs1[SB::SIZE];
  // XCD-aware order: blocks are dealt round-robin to the 8 XCDs by linear id,
  // and each XCD takes a contiguous run of the (batch, split, m-tile, n-tile)
  // order: it reuses a band's A rows, and a split's whole k range, from its
  // own L2.
  const int total = (int)(gridDim.x * gridDim.y * gridDim.z);
  int tile = (int)((blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x);
  tile = (tile % 8) * (total / 8) + min(tile % 8, total % 8) + tile / 8;
  const int n0 = (tile % (int)gridDim.x) * BN;
  tile /= (int)gridDim.x;
  const int m0 = (tile % (int)gridDim.y) * BM;
  const int z = tile / (int)gridDim.y, bt = z / g.splits;
  const int k_begin = (z % g.splits) * g.k_chunk;
  const float* A = g.a + bt * g.a_sb;
  const float* Bm = g.b + bt * g.b_sb;
  const int k_end = min(g.K, k_begin + g.k_chunk);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, wm = wave / WN;

  floatx16 big[NT][MT], small[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) big[i][j] = small[i][j] = zero16();
  float rs[4] = {0.f, 0.f, 0.f, 0.f};

  SA sa;
  SB sb;
  const __amdgpu_buffer_rsrc_t ra = buffer_rsrc(A, VEC ? g.a_bytes : 0u), rb = buffer_rsrc(Bm, VEC ? g.b_bytes : 0u);
  if (VEC) {
    sa.init(g.a_sm, g.a_sk, m0, g.M, tid);
    sb.init(g.b_sn, g.b_sk, n0, g.N, tid);
  }
  const int nst = k_end > k_begin ? (k_end - k_begin + 31) / 32 : 0;
  // (past the last stage the loads start again at stage 0: in bounds, never used)
  auto load = [&](int st, int s) {
    const int k0 = k_begin + (st < nst ? st : 0) * 32;
    sa.template load<VEC>(ra, A, g.a_sm, g.a_sk, m0, g.M, k0, s, k_end, g.K, tid);
    sb.template load<VEC>(rb, Bm, g.b_sn, g.b_sk, n0, g.N, k0, s, k_end, g.K, tid);
  };
  auto store = [&](int s, unsigned* Ad, unsigned* Bd) {
    sa.store(Ad, s, tid);
    // One operand's split at a time: together they take registers from the
    // loads in flight (M = 4096, us: 128 x 128 weight gradients of 2304 x 768 134.9
    // -> 122.7, 64 x 128 input gradients of 1280 x 1280 108 -> 97) -- but not in
    // the 128 x 128 input gradient, where the fence costs (2304 x 768 99 -> 104).
    if constexpr (!(BM == 128 && BN == 128 && A_KC)) WHA_FENCE();
    sb.store(Bd, s, tid);
  };
  auto multiply = [&](const unsigned* Ac, const unsigned* Bc) {
    Frag3 a[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) a[mt] = SA::frag(Ac, 32 * (MT * wm + mt), lane);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const Frag3 b = SB::frag(Bc, 32 * (NT * wn + nt), lane);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        big[nt][mt] = mfma_bf16(b.h, a[mt].h, big[nt][mt]);
        small[nt][mt] = mfma_small(b, a[mt], small[nt][mt]);
      }
    }
  };
  if (nst > 0) {
    load(0, 0);
    load(0, 1);
    store(0, As0, Bs0);
    if (!A_KC) sa.add_to(rs, 0, true);
    load(1, 0);
    for (int st = 0; st < nst; ++st) {
      __syncthreads();  // sub-stage 0 is in LDS; every wave is done with the other buffers
      store(1, As1, Bs1);
      if (!A_KC) sa.add_to(rs, 1, true);
      load(st + 1, 1);
      multiply(As0, Bs0);
      __syncthreads();
      store(0, As0, Bs0);  // (after the last stage: stored, never read or summed)
      if (!A_KC) sa.add_to(rs, 0, st + 1 < nst);
      load(st + 2, 0);
      multiply(As1, Bs1);
    }
  }

  // Bias gradient of the weight-gradient GEMM, by the blocks of the first
  // column tile: a row's sum lies in the eight threads that staged it (two k
  // of a sub-stage each), added in a fixed order.
  float* rdst = PARTIAL ? g.rowsum_part : g.rowsum;
  if (!A_KC && n0 == 0 && rdst != nullptr) {
    rdst += PARTIAL ? (int64_t)z * g.M : bt * g.rowsum_sb;
#pragma unroll
    for (int u = 0; u < SA::RU; ++u) {
      float t = rs[u];
      t += __shfl_xor(t, 1, 64);
      t += __shfl_xor(t, 2, 64);
      t += __shfl_xor(t, 4, 64);
      const int m = m0 + SA::row(tid, u);
      if ((tid & 7) == 0 && m < g.M) rdst[m] = t;
    }
  }

  // C[m][n], m = m0 + 32(MT wm + mt) + lane%32, n = n0 + 32(NT wn + nt) + 8u + 4(lane/32) + e
  const bool vec = PARTIAL ? (g.N % 4 == 0) : g.c_vec;
  const float* bias = (!PARTIAL && g.bias != nullptr) ? g.bias + bt * g.bias_sb : nullptr;
  // An infinite operand element, one that rounds to infinity or a product past
  // the fp32 range leaves infinity or NaN (wha_split.hpp) where fp32 arithmetic
  // may have another result.  A wave that meets one forms its tile again on the
  // fp32 MFMA, straight from memory, and takes those elements from there.  All
  // NaN, 4096 x 768 <- 768: 0.29 ms where finite operands take 0.044 (summed
  // element by element it was 4.2).
  auto finite = [](float x) { return __builtin_fabsf(x) < INFINITY; };
  bool again = false;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        big[nt][mt][i] += small[nt][mt][i];
        again |= !finite(big[nt][mt][i]);
      }
  if (__builtin_amdgcn_ballot_w64(again) != 0) {
    const float *ap[MT], *bp[NT];  // this lane's rows (past the extent: the last, never stored)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      ap[mt] = A + (int64_t)min(m0 + 32 * (MT * wm + mt) + (lane & 31), g.M - 1) * g.a_sm;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      bp[nt] = Bm + (int64_t)min(n0 + 32 * (NT * wn + nt) + (lane & 31), g.N - 1) * g.b_sn;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) small[nt][mt] = zero16();
    }
#pragma unroll 4
    for (int k0 = k_begin; k0 < k_end; k0 += 2) {
      const int k = k0 + (lane >> 5);
      float a[MT], b[NT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) a[mt] = k < k_end ? ap[mt][(int64_t)k * g.a_sk] : 0.f;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        b[nt] = k < k_end ? bp[nt][(int64_t)k * g.b_sk] : 0.f;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) small[nt][mt] = mfma_f32(b[nt], a[mt], small[nt][mt]);
      }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          big[nt][mt][i] = finite(big[nt][mt][i]) ? big[nt][mt][i] : small[nt][mt][i];
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = m0 + 32 * (MT * wm + mt) + (lane & 31);
    if (m >= g.M) continue;
    float* row =
        PARTIAL ? g.c + ((int64_t)z * g.M + m) * g.N : g.c + bt * g.c_sb + (int64_t)m * g.ldc;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int n = n0 + 32 * (NT * wn + nt) + 8 * u + 4 * (lane >> 5);
        if (n >= g.N) continue;
        float r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = big[nt][mt][4 * u + e];
        float* dst = row + n;
        if (bias != nullptr) {
#pragma unroll
          for (int e = 0; e < 4; ++e) r[e] = (n + e < g.N ? bias[n + e] : 0.f) + r[e];
        }
        if (vec && n + 3 < g.N) {
          if (!PARTIAL && g.accumulate) {
            const float4 o = *reinterpret_cast<const float4*>(dst);
            r[0] += o.x, r[1] += o.y, r[2] += o.z, r[3] += o.w;
          }
          *reinterpret_cast<float4*>(dst) = make_float4(r[0], r[1], r[2], r[3]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < g.N) dst[e] = (!PARTIAL && g.accumulate) ? r[e] + dst[e] : r[e];
        }
      }
    }
  }
}

namespace {

// 128-bit (row-contiguous operands: 64-bit) buffer loads: every row 16-byte
// aligned along its operand's contiguous direction (a_vec, b_vec), that
// direction's extent a multiple of four (pieces do not straddle the end), and
// each operand's reachable extent (one batch) below 2 GiB (32-bit offsets).
// Otherwise one load per element.  Weight gradients, where both operands are
// row-contiguous, take any number of positions.
template <bool A_KC, bool B_KC>
bool gemm_vec_ok(GemmArgs& g) {
  if (!(g.a_vec && g.b_vec && ((!A_KC && !B_KC) || g.K % 4 == 0) && (A_KC || g.M % 4 == 0) && (B_KC || g.N % 4 == 0)))
    return false;
  const int64_t a_ext = 4 * (A_KC ? (int64_t)(g.M - 1) * g.a_sm + g.K : (int64_t)(g.K - 1) * g.a_sk + g.M);
  const int64_t b_ext = 4 * (B_KC ? (int64_t)(g.N - 1) * g.b_sn + g.K : (int64_t)(g.K - 1) * g.b_sk + g.N);
  if (a_ext >= ((int64_t)1 << 31) || b_ext >= ((int64_t)1 << 31)) return false;
  g.a_bytes = (uint32_t)a_ext;
  g.b_bytes = (uint32_t)b_ext;
  return true;
}

template <int BM, int BN, int WM, int WN, bool A_KC, bool B_KC, bool PARTIAL>
void gemm_enqueue(GemmArgs& g, const dim3& grid, hipStream_t stream) {
  if (gemm_vec_ok<A_KC, B_KC>(g))
    hipLaunchKernelGGL((gemm_split_kernel<BM, BN, WM, WN, A_KC, B_KC, true, PARTIAL>), grid, dim3(256), 0, stream, g);
  else
    hipLaunchKernelGGL((gemm_split_kernel<BM, BN, WM, WN, A_KC, B_KC, false, PARTIAL>), grid, dim3(256), 0, stream, g);
}

template <int BM, int BN, int WM, int WN, bool A_KC, bool B_KC>
hipError_t gemm_launch(GemmArgs g, float* ws, int splits, const char* name, hipStream_t stream) {
  const dim3 grid((g.N + BN - 1) / BN, (g.M + BM - 1) / BM, splits * g.batch);
  g.splits = splits;
  const int per = (g.K + splits - 1) / splits;
  g.k_chunk = ((per + 31) / 32) * 32;
  TimingScope ts(name, stream);
  if (splits == 1) {
    gemm_enqueue<BM, BN, WM, WN, A_KC, B_KC, false>(g, grid, stream);
    return hipGetLastError();
  }
  GemmArgs p = g;
  p.c = ws;
  p.bias = nullptr;
  gemm_enqueue<BM, BN, WM, WN, A_KC, B_KC, true>(p, grid, stream);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return gemm_reduce(g, ws, stream);
}

}  // namespace

// Output tile and split-K factor of one GEMM, by estimated time: the k steps of
// the blocks of the CU that gets most of them, times what a k step of the tile
// costs (128 x 128: 0.054 us with every CU busy; the smaller tiles stage more
// per product: 0.55 of it for half the tile, 0.32 for a quarter of it, 0.45
// where an operand is contiguous along its rows and its pieces get narrower),
// plus, with a split, writing and adding up the partial tiles.  Measured at M =
// 8192 (us; 128 x 128, 64 x 128, 64 x 64): 768 <- 768 forward 75, 64, 71; 2304
// <- 768 186, 179, 208; 1536 <- 1536 220, 228, 263; 216 <- 768 39, 29, 27; and
// for the 768 x 768 weight gradient in 128 x 128 tiles split 4, 7, 10, 14 ways
// 98, 71, 81, 72.
constexpr int kCUs = 256;
GemmPick gemm_pick(int M, int N, int K, int batch, bool rows_contiguous, int max_splits, int min_k) {
  GemmPick best{64, 64, 1};
  double best_us = 1e30;
  const int tiles[4][2] = {{128, 128}, {64, 128}, {128, 64}, {64, 64}};
  for (const auto& t : tiles) {
    const double w = t[0] + t[1] == 256 ? 1. : t[0] + t[1] == 192 ? 0.55 : rows_contiguous ? 0.45 : 0.32;
    const int64_t blocks = (int64_t)((M + t[0] - 1) / t[0]) * ((N + t[1] - 1) / t[1]) * batch;
    for (int s = 1; s <= max_splits; ++s) {
      if (s > 1 && K / s < min_k) break;
      const int per = ((K + s - 1) / s + 31) / 32 * 32;
      double us = (double)((blocks * s + kCUs - 1) / kCUs) * w * 0.054 * (per + 32);
      if (s > 1) us += 2. + (double)s * M * N * batch * 1e-6;
      if (us < best_us) {
        best_us = us;
        best = GemmPick{t[0], t[1], s};
      }
    }
  }
  return best;
}

// Products below 2^24 multiply-adds stay on the fp32 MFMA kernels of linear.hip:
// their time is launch and latency, and they were no slower there (us, fp32
// MFMA against split: 1000 x 100 <- 77 forward / dx / dW 8.7 / 8.9 / 21.5
// against 9.8 / 11.1 / 22.9; above, 1024 x 504 <- 168 13.2 / 14.7 / 13.7
// against 11.2 / 13.4 / 16.5, 32 x 768 <- 768 32 / 31 / 10.8 against 18 / 20 /
// 12).  Above, the fp32 kernels are the faster ones by 5-25% (about 1 us) for
// forwards of at most 256 columns over at most 160 k and for input gradients of
// at most 256 columns below 2^26 (4312 x 192 <- 128 8.4 against 9.0, dx of 1500 x
// 192 <- 128 5.7 against 7.8), and by up to 13% for some operands whose rows are
// not aligned (4001 x 513 <- 512 dx 38.8 against 45.2); the rule leaves those
// here for the error, a third of the fp32 MFMA's.
bool gemm_split_ok(int64_t M, int64_t N, int64_t K, int64_t batch) {
  return (double)M * (double)N * (double)K * (double)batch >= (double)(1 << 24);
}
// Weight gradients from 2^29 on: below, their few output tiles and the split-K
// sum set the time (us, fp32 MFMA against split, M x N x K: 1024 x 504 x 168
// 13.7 / 16.5, 4096 x 504 x 168 19.9 / 20.9, 2048 x 384 x 384 21.2 / 21.1, 12
// heads of 8192 x 64 x 64 16.1 / 22.7; above, 8192 x 256 x 256 23.0 / 24.0, 4096 x
// 768 x 256 27.6 / 27.7, 4096 x 384 x 384 32.3 / 24.1, 1024 x 768 x 768 31.9 / 24.4,
// 8192 x 216 x 768 47.3 / 39.3): the line lies where the smallest outputs are
// no slower, those of more tiles gain from a little below it.
bool gemm_split_dw_ok(int64_t M, int64_t N, int64_t K, int64_t batch) {
  return (double)M * (double)N * (double)K * (double)batch >= (double)(1 << 29);
}

template <bool A_KC, bool B_KC>
hipError_t gemm_split(const GemmArgs& args, const GemmPick& t, float* ws, const char* name, hipStream_t stream) {
  GemmArgs g = args;
  // 128-bit loads need every row start along the contiguous direction 16-byte aligned
  g.a_vec = aligned16(g.a) && g.a_sb % 4 == 0 && (A_KC ? g.a_sm % 4 == 0 : g.a_sk % 4 == 0);
  g.b_vec = aligned16(g.b) && g.b_sb % 4 == 0 && (B_KC ? g.b_sn % 4 == 0 : g.b_sk % 4 == 0);
  if (t.bn == 64)
    return t.bm == 128 ? gemm_launch<128, 64, 4, 1, A_KC, B_KC>(g, ws, t.splits, name, stream)
                       : gemm_launch<64, 64, 2, 2, A_KC, B_KC>(g, ws, t.splits, name, stream);
  return t.bm == 128 ? gemm_launch<128, 128, 2, 2, A_KC, B_KC>(g, ws, t.splits, name, stream)
                     : gemm_launch<64, 128, 2, 2, A_KC, B_KC>(g, ws, t.splits, name, stream);
}

template hipError_t gemm_split<true, true>(const GemmArgs&, const GemmPick&, float*, const char*, hipStream_t);
template hipError_t gemm_split<true, false>(const GemmArgs&, const GemmPick&, float*, const char*, hipStream_t);
template hipError_t gemm_split<false, false>(const GemmArgs&, const GemmPick&, float*, const char*, hipStream_t);

}  // namespace wha
