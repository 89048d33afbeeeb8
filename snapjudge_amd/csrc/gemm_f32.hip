// gemm_f32.hip -- fp32-product GEMM for gfx950: out[M, N] = epi(A[M, K] . W[N, K]^T).
//
// Serves the fp32 numerics mode, the decision tail (scorer and act head, fp32
// in every mode), LoRA, and the bf16 shapes that the bf16 kernels' tiling does
// not cover (they are widened exactly on load).  Products and sums are fp32
// throughout: v_mfma_f32_16x16x4_f32.
//
// What bounds it.  The fp32 matrix rate is a sixteenth of the bf16 one (a
// 16x16x4 block takes 32 cycles), so operand bandwidth is not the limit once
// the loads are coalesced.
//  - gemm_f32_staged_kernel: 64x64 or 32x64 tiles, four waves, 32-deep K steps
//    in which eight lanes take 32 consecutive values of a row, moved by
//    direct-to-LDS loads through a three-stage ring, or through registers for
//    bf16 operands, rows no vector load can read and K of a few steps.
//  - gemm_f32_split_kernel, for products too small to give every CU such a
//    tile: 16x64 or 16x16 tiles whose eight waves each take an eighth of K and
//    add their sums through LDS in wave order, so that the weights stream
//    through as many CUs as there are and a wave's few steps are all in flight
//    at once.  Operands go straight to registers in the MFMA's own layout; 16
//    neighbouring lanes then read 16 different rows, which the vector cache
//    serves at a quarter of its rate or less (64x64 tiles loaded this way ran
//    the 1536 x 768 x 768 scorer in 51 us), so it is used only where latency,
//    not that rate, is the limit.
// Measured against the 64x64x16 FMA tiles both replace: the scorer's product of
// one request, 16 x 768 x 768, 83 (mean of the tail's four products) -> 7.4 us;
// of 96 questions, 1536 x 768 x 768, 85 (mean) -> 30 us (60 TFLOP/s; 8192 x
// 3072 x 768 reaches 107 of the 154 that a large fp32 product of the vendor
// library does); QKV of 569 rows 112 -> 32 us, the residual products 107 -> 21.
// Through registers: bf16 8000 x 768 x 777 304 -> 110 us (the split kernel 573),
// fp32 2000 x 768 x 769 126 -> 35, and 20000 x 768 x 8, a LoRA update, 36 -> 30.
// Both take the k values of a 16-deep group in the lanes' own order: lane
// (r, q) holds row r's values 4 q + [0, 4) and MFMA j of the group takes the
// lanes' j-th values, the same k on both sides.  The epilogue runs on the fp32
// tile in LDS.
#include <algorithm>
#include <type_traits>

#include "sjh_common.hpp"
#include "sjh_host.hpp"
#include "sjh_kernels.hpp"

namespace sjh {

namespace {

// ---- epilogue over an fp32 BMxBN tile staged in LDS (row stride ldcs) ----
template <int BM, int BN, int NT, typename OutT>
__device__ __forceinline__ void tile_epilogue(const float* Cs, int ldcs, int m0, int tile_n,
                                              const GemmArgs g) {
  const int tid = threadIdx.x;
  if (g.epi == EPI_GEGLU) {
    constexpr int HB = BN / 2;
    const int j0 = tile_n * HB;
    OutT* out = static_cast<OutT*>(g.out);
    for (int idx = tid; idx < BM * HB; idx += NT) {
      const int r = idx / HB, c = idx - r * HB;
      const int m = m0 + r, j = j0 + c;
      if (m < g.M && j < g.N) {
        const float in = Cs[r * ldcs + c], gate = Cs[r * ldcs + HB + c];
        store_f32(out + static_cast<int64_t>(m) * g.ldo + j, gelu_out<OutT>(in) * gate);
      }
    }
    return;
  }
  const int n0 = tile_n * BN;
  for (int idx = tid; idx < BM * BN; idx += NT) {
    const int r = idx / BN, c = idx - r * BN;
    const int m = m0 + r, n = n0 + c;
    if (m >= g.M || n >= g.N) continue;
    float v = Cs[r * ldcs + c];
    if (g.epi == EPI_RESID) {
      if (g.bias) v += g.bias[n];
      g.X[static_cast<int64_t>(m) * g.ldx + n] += v;
      continue;
    }
    if (g.epi == EPI_ROPE) {
      if (n < 2 * g.rope_dim) {
        const int hd = g.head_dim, half = hd >> 1;
        const int dd = n % hd;
        const int64_t p = min(max(g.pos[m], 0), g.rope_rows - 1);
        if (dd < half) {
          const float x1 = Cs[r * ldcs + c + half];
          const float cs = g.rope_cos[p * half + dd], sn = g.rope_sin[p * half + dd];
          v = rope_lo(v, x1, cs, sn);
        } else {
          const int d2 = dd - half;
          const float x0 = Cs[r * ldcs + c - half];
          const float cs = g.rope_cos[p * half + d2], sn = g.rope_sin[p * half + d2];
          v = rope_hi(x0, v, cs, sn);
        }
        if (n < g.rope_dim) v *= g.q_scale;
      }
    } else {
      if (g.bias) v += g.bias[n];
      if (g.act == 1)
        v = gelu_out<OutT>(v);
      else if (g.act == 2)
        v = fmaxf(v, 0.f);
    }
    store_f32(static_cast<OutT*>(g.out) + static_cast<int64_t>(m) * g.ldo + n, v);
  }
}

// W row feeding tile row i of column tile tile_n (GEGLU: first half of the
// tile = input rows, second half = gate rows of the reference's [2F, K] Wi).
template <int BN>
__device__ __forceinline__ int64_t w_row(const GemmArgs g, int tile_n, int i) {
  if (g.epi == EPI_GEGLU) {
    constexpr int HB = BN / 2;
    const int j = tile_n * HB + (i < HB ? i : i - HB);
    const int jc = j < g.N ? j : g.N - 1;
    return i < HB ? jc : static_cast<int64_t>(g.N) + jc;
  }
  const int n = tile_n * BN + i;
  return n < g.N ? n : g.N - 1;
}

// Four k values of one operand row as fp32 (16- or 8-byte load).
__device__ __forceinline__ f32x4_t load4(const float* p) { return *reinterpret_cast<const f32x4_t*>(p); }
__device__ __forceinline__ f32x4_t load4(const bf16_t* p) {
  const u32x2_t v = *reinterpret_cast<const u32x2_t*>(p);
  return f32x4_t{__uint_as_float(v[0] << 16), __uint_as_float(v[0] & 0xffff0000u), __uint_as_float(v[1] << 16),
                 __uint_as_float(v[1] & 0xffff0000u)};
}
template <typename T>
__device__ __forceinline__ f32x4_t load4_upto(const T* p, int n) {
  f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (j < n) v[j] = load_f32(p + j);
  return v;
}

// Workgroups of a grid's row: a grid dimension holds fewer than 2^32 threads
// (512 of them here at most), so that more tiles take several rows.
constexpr unsigned kGridX = 1u << 22;

// Tile of this workgroup, or false past the last one.  XCDs get contiguous runs
// of tiles (workgroups go round-robin over the 8 XCDs); the operand with fewer
// rows is the one that every XCD reads whole.
template <int BM, int BN>
__device__ __forceinline__ bool pick_tile(const GemmArgs& g, int launch_m, int& tile_m, int& tile_n) {
  const int tiles_n = g.epi == EPI_GEGLU ? (g.N + BN / 2 - 1) / (BN / 2) : (g.N + BN - 1) / BN;
  const int tiles_m = (launch_m + BM - 1) / BM;
  const int nb = tiles_m * tiles_n;
  const unsigned wg = blockIdx.y * kGridX + blockIdx.x;
  if (wg >= static_cast<unsigned>(nb)) return false;
  const int bid = static_cast<int>(wg);
  const int xcd = bid & 7, per = nb >> 3, rem = nb & 7;
  const int tile = xcd * per + min(xcd, rem) + (bid >> 3);
  if (launch_m < g.N) {
    tile_n = tile / tiles_m;
    tile_m = tile - tile_n * tiles_m;
  } else {
    tile_m = tile / tiles_n;
    tile_n = tile - tile_m * tiles_n;
  }
  return true;
}

// 16 x 16 TJ tiles, K cut into WGK slices of whole 16-deep steps, one wave
// each, PD steps of operands in flight per wave.  vec_steps: leading steps that
// may use vector loads (aligned rows).
template <typename InT, typename OutT, int TJ, int WGK, int PD>
__global__ __launch_bounds__(64 * WGK) void gemm_f32_split_kernel(GemmArgs g0, int vec_steps) {
  GemmArgs g = g0;
  if (g.M_dev) g.M = *g.M_dev;
  constexpr int BM = 16, BN = 16 * TJ, NT = 64 * WGK, LDC = BN + 4;
  __shared__ float Cs[WGK * BM * LDC];
  int tile_m, tile_n;
  if (!pick_tile<BM, BN>(g, g0.M, tile_m, tile_n)) return;  // (uniform)
  const int m0 = tile_m * BM;
  if (m0 >= g.M) return;  // a row tile past the device row count (uniform)

  const int tid = threadIdx.x, lane = tid & 63, wk = tid >> 6;
  const int r16 = lane & 15, q4 = (lane >> 4) * 4;
  const InT* ap = static_cast<const InT*>(g.A) + static_cast<int64_t>(min(m0 + r16, g.M - 1)) * g.lda + q4;
  const InT* wp[TJ];
#pragma unroll
  for (int j = 0; j < TJ; ++j)
    wp[j] = static_cast<const InT*>(g.W) + w_row<BN>(g, tile_n, j * 16 + r16) * g.ldw + q4;

  f32x4_t acc[TJ];
#pragma unroll
  for (int j = 0; j < TJ; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  f32x4_t a[PD], w[PD][TJ];
  auto mac = [&](int u) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int j = 0; j < TJ; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][c], w[u][j][c], acc[j], 0, 0, 0);
  };
  auto load = [&](int s, int u) {
    a[u] = load4(ap + 16 * s);
#pragma unroll
    for (int j = 0; j < TJ; ++j) w[u][j] = load4(wp[j] + 16 * s);
  };

  // steps [s0, s1) of this wave: vector loads up to vec_steps, then guarded
  // scalar loads (unaligned rows, and the step that K ends in)
  const int steps = (g.K + 15) >> 4, chunk = (steps + WGK - 1) / WGK;
  const int s0 = wk * chunk, s1 = min(s0 + chunk, steps);
  const int n = min(s1, vec_steps) - s0;
  int i = 0;
#pragma unroll
  for (int u = 0; u < PD; ++u)
    if (u < n) load(s0 + u, u);
  for (; i + 2 * PD <= n; i += PD)
#pragma unroll
    for (int u = 0; u < PD; ++u) {
      mac(u);
      load(s0 + i + u + PD, u);
    }
#pragma unroll
  for (int u = 0; u < PD; ++u)
    if (i + u < n) {
      mac(u);
      if (i + u + PD < n) load(s0 + i + u + PD, u);
    }
#pragma unroll
  for (int u = 0; u < PD; ++u)
    if (i + PD + u < n) mac(u);
  for (int s = max(s0, vec_steps); s < s1; ++s) {
    const int left = g.K - 16 * s - q4;  // k values of this lane's four that exist
    a[0] = load4_upto(ap + 16 * s, left);
#pragma unroll
    for (int j = 0; j < TJ; ++j) w[0][j] = load4_upto(wp[j] + 16 * s, left);
    mac(0);
  }

  // accumulator lane (r, q): column r, rows 4 q + [0, 4) of a block
  float* C = Cs + wk * BM * LDC;
#pragma unroll
  for (int j = 0; j < TJ; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) C[(q4 + e) * LDC + j * 16 + r16] = acc[j][e];
  __syncthreads();
  for (int idx = tid; idx < BM * BN; idx += NT) {  // the slices' sums, in order
    const int o = (idx / BN) * LDC + idx % BN;
    float v = Cs[o];
#pragma unroll
    for (int k = 1; k < WGK; ++k) v += Cs[k * BM * LDC + o];
    Cs[o] = v;
  }
  __syncthreads();
  tile_epilogue<BM, BN, NT, OutT>(Cs, LDC, m0, tile_n, g);
}

// BM x 64 tiles, four waves in 2 x 2.  DIRECT (fp32, 16-byte aligned rows): whole
// K steps go straight to LDS, two ahead of their use.  Otherwise, and for the
// last partial step, a step's values pass through registers (widened there, the
// next step's in flight meanwhile) into one LDS buffer; vec: rows aligned to four
// values, which one load then takes.
template <typename InT, typename OutT, int BM, bool DIRECT>
__global__ __launch_bounds__(256) void gemm_f32_staged_kernel(GemmArgs g0, int vec) {
  static_assert(!DIRECT || std::is_same<InT, float>::value, "direct loads move fp32 rows");
  GemmArgs g = g0;
  if (g.M_dev) g.M = *g.M_dev;
  constexpr int BN = 64, BK = 32, NS = DIRECT ? 3 : 1, RB = BK * 4, ROWS = BM + BN, LDC = BN + 4;
  constexpr int TI = BM / 32, TJ = 2, G = ROWS / 32;  // load instructions (8 rows each) per wave and stage
  constexpr int STAGE = ROWS * RB;
  constexpr int LDS = NS * STAGE > BM * LDC * 4 ? NS * STAGE : BM * LDC * 4;  // the epilogue's tile reuses the ring
  __shared__ __attribute__((aligned(16))) char ring[LDS];
  int tile_m, tile_n;
  if (!pick_tile<BM, BN>(g, g0.M, tile_m, tile_n)) return;  // (uniform)
  const int m0 = tile_m * BM;
  if (m0 >= g.M) return;  // a row tile past the device row count (uniform)

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1, r16 = lane & 15, q = lane >> 4;
  const InT* A = static_cast<const InT*>(g.A);
  const InT* W = static_cast<const InT*>(g.W);
  auto row_ptr = [&](int r) {
    return r < BM ? A + static_cast<int64_t>(min(m0 + r, g.M - 1)) * g.lda : W + w_row<BN>(g, tile_n, r - BM) * g.ldw;
  };
  // 16-byte chunk c of row r sits at slot c ^ swz(r): 16 consecutive rows at one
  // chunk then fall into 16 different 16-byte bank groups
  auto swz = [](int r) { return (r >> 1) & 7; };
  f32x4_t acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int key = swz(r16);  // (a block's first row is a multiple of 16)
  const char* a_row = ring + (wm * TI * 16 + r16) * RB;
  const char* w_rowp = ring + (BM + wn * TJ * 16 + r16) * RB;
  auto compute = [&](int slot) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int off = slot * STAGE + ((4 * h + q) ^ key) * 16;
      f32x4_t a[TI], w[TJ];
#pragma unroll
      for (int i = 0; i < TI; ++i) a[i] = *reinterpret_cast<const f32x4_t*>(a_row + i * 16 * RB + off);
#pragma unroll
      for (int j = 0; j < TJ; ++j) w[j] = *reinterpret_cast<const f32x4_t*>(w_rowp + j * 16 * RB + off);
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < TJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][c], w[j][c], acc[i][j], 0, 0, 0);
    }
  };

  int k0 = 0;
  if constexpr (DIRECT) {
    const float* src[G];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int r = 8 * (wave + 4 * i) + (lane >> 3);
      src[i] = row_ptr(r) + 4 * ((lane & 7) ^ swz(r));
    }
    auto issue = [&](int kt, int slot) {
#pragma unroll
      for (int i = 0; i < G; ++i) load_lds16(src[i] + kt * BK, ring + slot * STAGE + (wave + 4 * i) * 1024);
    };
    const int nk = g.K / BK;
#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
      if (s < nk) issue(s, s);
    int slot = 0;
    for (int kt = 0; kt < nk; ++kt) {
      if (kt + 1 < nk)
        wait_vmcnt<G*(NS - 2)>();
      else
        wait_vmcnt<0>();
      wait_lgkm0();  // this wave's reads of the slot that is refilled next
      __builtin_amdgcn_s_barrier();
      if (kt + NS - 1 < nk) issue(kt + NS - 1, slot == 0 ? NS - 1 : slot - 1);
      compute(slot);
      slot = slot + 1 == NS ? 0 : slot + 1;
    }
    k0 = nk * BK;
  }
  if (k0 < g.K) {
    constexpr int NP = ROWS * 8 / 256;  // four-value pieces per thread and step
    const int c = tid & 7;
    const InT* row[NP];
    f32x4_t v[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) row[i] = row_ptr((tid >> 3) + 32 * i) + 4 * c;
    auto fetch = [&](int k) {
      const int left = g.K - k - 4 * c;  // k values of this thread's four that exist
      if (left < 4) {
#pragma unroll
        for (int i = 0; i < NP; ++i) v[i] = load4_upto(row[i] + k, left);
      } else if (vec) {
#pragma unroll
        for (int i = 0; i < NP; ++i) v[i] = load4(row[i] + k);
      } else {
#pragma unroll
        for (int i = 0; i < NP; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) v[i][j] = load_f32(row[i] + k + j);
      }
    };
    fetch(k0);
    for (; k0 < g.K; k0 += BK) {
      __syncthreads();  // the reads of the step before
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int r = (tid >> 3) + 32 * i;
        *reinterpret_cast<f32x4_t*>(ring + r * RB + (c ^ swz(r)) * 16) = v[i];
      }
      __syncthreads();
      if (k0 + BK < g.K) fetch(k0 + BK);
      compute(0);
    }
  }
  __syncthreads();
  float* Cs = reinterpret_cast<float*>(ring);
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        Cs[((wm * TI + i) * 16 + 4 * q + e) * LDC + (wn * TJ + j) * 16 + r16] = acc[i][j][e];
  __syncthreads();
  tile_epilogue<BM, BN, 256, OutT>(Cs, LDC, m0, tile_n, g);
}

unsigned tiles_of(const GemmArgs& g, int BM, int BN) {
  const int64_t tiles_n = g.epi == EPI_GEGLU ? (g.N + BN / 2 - 1) / (BN / 2) : (g.N + BN - 1) / BN;
  const int64_t tiles = tiles_n * ((g.M + BM - 1) / BM);
  require(tiles < (int64_t{1} << 31), "gemm: too many tiles");
  return static_cast<unsigned>(tiles);
}

dim3 grid_of(unsigned tiles) { return dim3(std::min(tiles, kGridX), (tiles + kGridX - 1) / kGridX); }

template <typename InT, typename OutT, bool DIRECT>
void launch_staged(const GemmArgs& g, int vec, unsigned t32, hipStream_t st) {
  if (t32 >= 8 * static_cast<unsigned>(num_cus()))
    gemm_f32_staged_kernel<InT, OutT, 64, DIRECT><<<grid_of(tiles_of(g, 64, 64)), 256, 0, st>>>(g, vec);
  else
    gemm_f32_staged_kernel<InT, OutT, 32, DIRECT><<<grid_of(t32), 256, 0, st>>>(g, vec);
}

template <typename InT, typename OutT>
void launch_typed(const GemmArgs& g, hipStream_t st) {
  const uintptr_t align = 4 * sizeof(InT) - 1;
  const bool vec = g.lda % 4 == 0 && g.ldw % 4 == 0 && (reinterpret_cast<uintptr_t>(g.A) & align) == 0 &&
                   (reinterpret_cast<uintptr_t>(g.W) & align) == 0;
  // Staged tiles once there are enough for three CUs in four (N = 768, 575
  // rows: 21 us a product against 28 split); 64 rows each where there are
  // several rounds of them anyway (fewer operand bytes per product), 32 below,
  // so that the last round is shorter.
  const unsigned t32 = tiles_of(g, 32, 64), cus = static_cast<unsigned>(num_cus());
  if (t32 >= 3 * cus / 4) {
    // direct-to-LDS steps where rows allow them and there are enough steps to
    // pay for the ring: with several rounds of tiles its 48 KB leave three
    // workgroups on a CU instead of eight to cover each other's start and
    // epilogue (18432 x 3072 x 256: 323 us direct, 289 through registers; 8192 x
    // 768 at K = 384 55.5 and 55.8, 512 66.9 and 68.9).  One round has no such
    // cover to lose (1000 x 768 x 64 6.5 and 7.0, 768 20.6 and 22.0).  The same bits.
    if constexpr (std::is_same<InT, float>::value)
      if (vec && g.K >= (t32 >= 8 * cus ? 384 : 64)) {
        launch_staged<InT, OutT, true>(g, vec, t32, st);
        return;
      }
    launch_staged<InT, OutT, false>(g, vec, t32, st);
    return;
  }
  // 16x16 tiles where 16x64 ones would leave CUs idle and the epilogue (bias,
  // activation, residual) needs no pairs of columns
  const int vec_steps = vec ? g.K / 16 : 0;
  if (tiles_of(g, 16, 64) < cus && (g.epi == EPI_STORE || g.epi == EPI_RESID))
    gemm_f32_split_kernel<InT, OutT, 1, 8, 6><<<grid_of(tiles_of(g, 16, 16)), 512, 0, st>>>(g, vec_steps);
  else
    gemm_f32_split_kernel<InT, OutT, 4, 8, 6><<<grid_of(tiles_of(g, 16, 64)), 512, 0, st>>>(g, vec_steps);
}

}  // namespace

void launch_gemm_f32(const GemmArgs& g, hipStream_t st) {
  const bool bf_out = g.out_dtype == DT_BF16;
  if (g.in_dtype == DT_BF16)
    bf_out ? launch_typed<bf16_t, bf16_t>(g, st) : launch_typed<bf16_t, float>(g, st);
  else
    bf_out ? launch_typed<float, bf16_t>(g, st) : launch_typed<float, float>(g, st);
}

}  // namespace sjh
