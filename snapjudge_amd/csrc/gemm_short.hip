// gemm_short.hip -- projection GEMMs of short batches for gfx950.
//
// What bounds them.  A batch of up to a few hundred rows does so little work
// per layer that its time is that of its launches, each a chain of memory
// round trips: a compute unit takes the tens of KB of operands that a tile
// needs at ~25 GB/s from memory and ~65 GB/s from its L2, and a launch has a
// fixed cost of a few microseconds.  So:
//  - as many of a tile's loads as fit are in flight at once, issued by four
//    waves (or one wave per K slice) before the first use;
//  - the RoPE rows and the residual stream that an epilogue reads are loaded
//    with them, not after the products (the bias and fp8 scales are: a few bytes
//    per tile, whose loads the sums' way through LDS mostly covers);
//  - no kernel reads the batch's row count first: every row of the launch is
//    computed (the buffers hold them), whatever is in the surplus ones (but for a
//    residual stream in the caller's memory, whose rows end with the batch);
//  - residual products cut K over the waves of one workgroup and add the
//    slices there, in slice order, so that no partial sums travel through
//    memory to the LayerNorm that would add them.
//
// Measured per launch at 128 rows of a 768-wide layer (start to start in a
// replayed graph, against the 64x32 and split-K tiles these replace there): QKV
// + RoPE 8.0 -> 5.1 us (5.4 while its tables waited for the operands), Wi + GEGLU
// 7.9 -> 5.0, Wo2 with the LayerNorm after it 10.9 -> 8.0; at 256 rows Wo2 12.3 ->
// 10.1 (the others: plain_pays).  At 640 rows
// the 64x64 tiles are the faster ones (10.6 against 11.9, 10.9 against 11.3).
// With fp8 weights, which had one 256x256 tile shape, four layers of 128 rows
// take 175 us and 256 rows 224 us, against 636.  The LayerNorm before a product
// computed inside it (rows of the fp32 stream normalised by every column tile)
// took 10.6 us against 5.4 + 3.5 for the two launches: its statistics cost more
// than the launch.
//
// v_mfma_f32_16x16x32_bf16 adds its products to the accumulator in the order
// of two v_mfma_f32_32x32x16_bf16 over the same k values (the same bits on the
// device over 24 chained steps of random values), so a product here has the
// bits of the other bf16 kernels': sum over K in order for plain, RoPE and
// GEGLU products; for residual ones the K slices of split_k_slices().  With fp8
// weights the residual products of more rows sum K in one chain, so that a row's
// bits differ between batches of up to 256 rows and larger ones, as bf16 rows' do.
#include <algorithm>
#include <type_traits>

#include "sjh_common.hpp"
#include "sjh_host.hpp"
#include "sjh_kernels.hpp"

namespace sjh {

namespace {

typedef __attribute__((ext_vector_type(2))) float f32x2_t;

// W row of tile row i.  Columns that an epilogue combines meet in one tile: a
// RoPE dim and its partner 32 higher (head_dim 64), a GEGLU input and its gate,
// BN / 2 rows apart.
template <int BN, int EPI>
__device__ __forceinline__ int short_w_row(const GemmArgs& g, int tile_n, int i) {
  if constexpr (EPI == EPI_ROPE) {
    const int p = tile_n * (BN / 2) + (i & (BN / 2 - 1));
    return (p >> 5) * 64 + (p & 31) + (i >= BN / 2 ? 32 : 0);
  } else if constexpr (EPI == EPI_GEGLU) {
    const int j = tile_n * (BN / 2) + (i & (BN / 2 - 1));
    return i >= BN / 2 ? g.N + j : j;
  } else {
    return min(tile_n * BN + i, g.N - 1);
  }
}

// Row tiles fastest, XCDs taking contiguous runs of tiles: the row tiles that
// read one W tile share an XCD's L2.
__device__ __forceinline__ void short_tile(int tiles_m, int& tile_m, int& tile_n) {
  const int nb = static_cast<int>(gridDim.x), bid = static_cast<int>(blockIdx.x);
  const int xcd = bid & 7, tile = xcd * (nb >> 3) + min(xcd, nb & 7) + (bid >> 3);
  tile_n = tile / tiles_m;
  tile_m = tile - tile_n * tiles_m;
}

// ---- plain, RoPE and GEGLU products: the whole K per wave -------------------
// BM x 32 tiles, four waves in 2 x 2.  K = 64 GR NG, moved into LDS in NG groups
// of GR 64-deep stages through a ring of R groups (R == NG: all of K is in
// flight from the start).
template <int BM, int GR, int NG, int R, bool W8>
struct STile {
  static constexpr int BN = 32;
  static constexpr int A_STAGE = BM * 128, W_STAGE = W8 ? BN * 64 : BN * 128, STAGE = A_STAGE + W_STAGE;
  static constexpr int INSTR = STAGE / 1024;       // load instructions per stage
  static constexpr int PER_GROUP = GR * INSTR / 4;  // ... per group and wave
  static constexpr int LDC = BN + 4;
  static constexpr int LDS = R * GR * STAGE > BM * LDC * 4 ? R * GR * STAGE : BM * LDC * 4;
  static_assert(R <= NG && GR * INSTR % 4 == 0, "loads split evenly over the waves");
  static_assert(LDS <= 160 * 1024, "LDS");
};

template <int BM, int GR, int NG, int R, bool W8, int EPI>
__global__ __launch_bounds__(256) void gemm_short_kernel(GemmArgs g) {
  using T = STile<BM, GR, NG, R, W8>;
  constexpr int BN = T::BN, TI = BM / 32, LDC = T::LDC;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  int tile_m, tile_n;
  short_tile(g.M / BM, tile_m, tile_n);
  const int m0 = tile_m * BM;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // epilogue items: two neighbouring columns (of a pair's lower half) each
  constexpr int EC = EPI == EPI_STORE ? BN / 2 : BN / 4, ES = BM * EC / 256;
  static_assert(BM * EC % 256 == 0, "epilogue items");
  // A RoPE tile's positions come through the scalar cache, eight rows per wave, so
  // that the table loads wait for them and for no operand (a vector load's wait
  // would drain those issued after it as well).
  int pos[ES];
  if constexpr (EPI == EPI_ROPE) {
    static_assert(EC == 8, "eight rows of items per wave");
#pragma unroll
    for (int s = 0; s < ES; ++s) {
      const int* pr = g.pos + m0 + 32 * s + 8 * wave;  // uniform
      pos[s] = __builtin_amdgcn_readfirstlane(pr[0]);
#pragma unroll
      for (int i = 1; i < 8; ++i) {
        const int p = __builtin_amdgcn_readfirstlane(pr[i]);  // (else the selected address is loaded, by lane)
        pos[s] = (lane >> 3) == i ? p : pos[s];
      }
    }
  }

  // operand loads: instruction j of a stage moves 1 KB, 8 rows of 128 bytes (16
  // of 64 for fp8 W rows).  A row's 16-byte chunk c goes to slot c ^ key(row),
  // so that 16 consecutive rows at one chunk fall into 16 different bank groups.
  auto issue_group = [&](int grp) {
#pragma unroll
    for (int i = 0; i < T::PER_GROUP; ++i) {
      const int j = i * 4 + wave;  // uniform
      const int stage = j / T::INSTR, w = j - stage * T::INSTR, kt = grp * GR + stage;
      char* dst = lds + ((grp % R) * GR + stage) * T::STAGE + w * 1024;
      if (w < T::A_STAGE / 1024) {
        const int r = w * 8 + (lane >> 3);
        load_lds16(static_cast<const bf16_t*>(g.A) + (m0 + r) * g.lda + kt * 64 + ((lane & 7) ^ ((r >> 1) & 7)) * 8, dst);
      } else if constexpr (W8) {
        const int r = (w - T::A_STAGE / 1024) * 16 + (lane >> 2);
        load_lds16(static_cast<const uint8_t*>(g.W) + short_w_row<BN, EPI>(g, tile_n, r) * g.ldw + kt * 64 +
                       ((lane & 3) ^ ((r >> 2) & 3)) * 16,
                   dst);
      } else {
        const int r = (w - T::A_STAGE / 1024) * 8 + (lane >> 3);
        load_lds16(static_cast<const bf16_t*>(g.W) + short_w_row<BN, EPI>(g, tile_n, r) * g.ldw + kt * 64 +
                       ((lane & 7) ^ ((r >> 1) & 7)) * 8,
                   dst);
      }
    }
  };
#pragma unroll
  for (int grp = 0; grp < R; ++grp) issue_group(grp);
  __builtin_amdgcn_sched_barrier(0);
  f32x2_t cs[ES], sn[ES];
  if constexpr (EPI == EPI_ROPE) {
#pragma unroll
    for (int s = 0; s < ES; ++s) {
      const int c = 2 * ((tid + 256 * s) % EC);
      const int64_t o = static_cast<int64_t>(min(max(pos[s], 0), g.rope_rows - 1)) * 32 + ((tile_n * (BN / 2) + c) & 31);
      cs[s] = *reinterpret_cast<const f32x2_t*>(g.rope_cos + o);
      sn[s] = *reinterpret_cast<const f32x2_t*>(g.rope_sin + o);
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  const int wm = wave >> 1, wn = wave & 1, r16 = lane & 15, q = lane >> 4;
  // 8-value chunk of a 32-deep step that this lane's quarter takes: in order,
  // or 0, 2, 1, 3 for fp8 weights (the persistent kernel's order)
  const int qc = W8 ? (q == 1 ? 2 : q == 2 ? 1 : q) : q;
  f32x4_t acc[TI];
#pragma unroll
  for (int t = 0; t < TI; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto step = [&](auto grp_tag) {
    constexpr int grp = decltype(grp_tag)::value;
    // operand loads of this wave issued after group grp's: the later groups of the
    // first R and the refills so far (one per group consumed).  The table loads are
    // not counted: how many the compiler makes of them, and where it puts them,
    // must not decide whether a group has landed.
    constexpr int last = grp - 1 + R < NG - 1 ? grp - 1 + R : NG - 1;
    wait_vmcnt<(last - grp) * T::PER_GROUP>();
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int s = 0; s < GR; ++s) {
      const char* sa = lds + ((grp % R) * GR + s) * T::STAGE + (wm * (BM / 2) + r16) * 128;
      const char* sw = lds + ((grp % R) * GR + s) * T::STAGE + T::A_STAGE;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        bf16x8_t w;
        if constexpr (W8) {
          const int r = wn * 16 + r16, c = 4 * h + qc;  // 8-byte piece c of the row's eight
          const u32x2_t v = *reinterpret_cast<const u32x2_t*>(sw + r * 64 + ((c >> 1) ^ ((r >> 2) & 3)) * 16 + (c & 1) * 8);
          w = fp8x8_to_bf16(v[0], v[1]);
        } else {
          w = *reinterpret_cast<const bf16x8_t*>(sw + (wn * 16 + r16) * 128 + ((4 * h + qc) ^ ((r16 >> 1) & 7)) * 16);
        }
#pragma unroll
        for (int t = 0; t < TI; ++t) {
          const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(sa + t * 2048 + ((4 * h + qc) ^ ((r16 >> 1) & 7)) * 16);
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w, acc[t], 0, 0, 0);
        }
      }
    }
    if constexpr (grp + R < NG) {
      wait_lgkm0();  // this wave's reads of the slots that are refilled next
      __builtin_amdgcn_s_barrier();
      issue_group(grp + R);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  step(std::integral_constant<int, 0>{});
  if constexpr (NG > 1) step(std::integral_constant<int, 1>{});
  if constexpr (NG > 2) step(std::integral_constant<int, 2>{});
  if constexpr (NG > 3) step(std::integral_constant<int, 3>{});
  static_assert(NG <= 4, "groups");

  // ---- epilogue on the tile in LDS
  __syncthreads();
  float* C = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int t = 0; t < TI; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) C[(wm * (BM / 2) + t * 16 + 4 * q + e) * LDC + wn * 16 + r16] = acc[t][e];
  __syncthreads();
  auto two = [&](int r, int c) {
    f32x2_t v = *reinterpret_cast<const f32x2_t*>(C + r * LDC + c);
    if constexpr (W8) {
      v[0] *= g.w_scale[short_w_row<BN, EPI>(g, tile_n, c)];
      v[1] *= g.w_scale[short_w_row<BN, EPI>(g, tile_n, c + 1)];
    }
    return v;
  };
  bf16_t* out = static_cast<bf16_t*>(g.out);
#pragma unroll
  for (int s = 0; s < ES; ++s) {
    const int r = (tid + 256 * s) / EC, c = 2 * ((tid + 256 * s) % EC);
    bf16_t* orow = out + static_cast<int64_t>(m0 + r) * g.ldo;
    if constexpr (EPI == EPI_ROPE) {
      const f32x2_t x0 = two(r, c), x1 = two(r, c + BN / 2);
      const int n = short_w_row<BN, EPI>(g, tile_n, c);
      float lo[2], hi[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const bool rot = n < 2 * g.rope_dim;
        lo[k] = rot ? rope_lo(x0[k], x1[k], cs[s][k], sn[s][k]) : x0[k];
        hi[k] = rot ? rope_hi(x0[k], x1[k], cs[s][k], sn[s][k]) : x1[k];
        if (n < g.rope_dim) lo[k] *= g.q_scale, hi[k] *= g.q_scale;
      }
      *reinterpret_cast<uint32_t*>(orow + n) = pack_bf16x2(lo[0], lo[1]);
      *reinterpret_cast<uint32_t*>(orow + n + 32) = pack_bf16x2(hi[0], hi[1]);
    } else if constexpr (EPI == EPI_GEGLU) {
      const f32x2_t in = two(r, c), gate = two(r, c + BN / 2);
      *reinterpret_cast<uint32_t*>(orow + tile_n * (BN / 2) + c) =
          pack_bf16x2(gelu_as(in[0]) * gate[0], gelu_as(in[1]) * gate[1]);
    } else {
      const int n = tile_n * BN + c;
      if (n >= g.N) continue;  // (N is even)
      f32x2_t v = two(r, c);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        if (g.bias) v[k] += g.bias[n + k];
        v[k] = g.act == 1 ? gelu_as(v[k]) : g.act == 2 ? fmaxf(v[k], 0.f) : v[k];
      }
      *reinterpret_cast<uint32_t*>(orow + n) = pack_bf16x2(v[0], v[1]);
    }
  }
}

template <int BM, int GR, int NG, int R, bool W8, int EPI>
void launch_tile(const GemmArgs& g, hipStream_t st) {
  using T = STile<BM, GR, NG, R, W8>;
  constexpr int per = EPI == EPI_GEGLU ? T::BN / 2 : T::BN;
  auto kern = gemm_short_kernel<BM, GR, NG, R, W8, EPI>;
  static const bool attr_set = [&] {  // per instantiation; the attribute is per function
    hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS),
              "gemm: LDS attribute");
    return true;
  }();
  (void)attr_set;
  kern<<<static_cast<unsigned>((g.N + per - 1) / per * (g.M / BM)), 256, T::LDS, st>>>(g);
}

template <int BM, int GR, int NG, int R, bool W8>
void launch_epi(const GemmArgs& g, hipStream_t st) {
  switch (g.epi) {
    case EPI_ROPE: launch_tile<BM, GR, NG, R, W8, EPI_ROPE>(g, st); break;
    case EPI_GEGLU: launch_tile<BM, GR, NG, R, W8, EPI_GEGLU>(g, st); break;
    default: launch_tile<BM, GR, NG, R, W8, EPI_STORE>(g, st); break;
  }
}

template <int BM, int R, bool W8>
void launch_k(const GemmArgs& g, hipStream_t st) {
  switch (g.K / 256) {
    case 1: launch_epi<BM, 4, 1, 1, W8>(g, st); break;
    case 2: launch_epi<BM, 4, 2, 2, W8>(g, st); break;
    case 3: launch_epi<BM, 4, 3, R < 3 ? R : 3, W8>(g, st); break;
    default: launch_epi<BM, 4, 4, R, W8>(g, st); break;
  }
}

int plain_tiles(const GemmArgs& g) {
  return (g.epi == EPI_GEGLU ? (g.N + 15) / 16 : (g.N + 31) / 32) * (g.M / 32);
}

// How many tiles these kernels take of a product, by whole layers in replayed graphs
// against the 64x32 tiles (fp8: 64x64): all that run at once, two per CU (192 rows of
// a 768-wide layer, 432 tiles: QKV 2.3 us less, Wi + GEGLU 2.2). A second round
// saves less (Wi + GEGLU of 192 rows at K = 1024, 984 tiles: 0.5, with fp8 weights
// 0.6), and loses where the third begins (256 rows, 1312 tiles: 0.4 and 1.4 more).
// It loses at once for biased products (the decision head's at 256 rows, 576 and 768
// tiles: ~1.5 more) and QKV at K up to 768 (256 rows, 576 tiles: 0.6 more; at K =
// 1024, 768 tiles, 1.3 less, with fp8 weights 2.1-2.5 less).  Wi + GEGLU of the same
// 256 rows at K = 768 gains 0.5 on the other tiles while QKV stays here, but both
// there lose 1.2, so that one of the two goes.
bool plain_pays(const GemmArgs& g) {
  const bool one_round = g.epi == EPI_STORE || (g.epi == EPI_ROPE && g.K <= 768 && g.w_dtype != DT_FP8);
  return plain_tiles(g) <= (one_round ? 2 : 4) * num_cus();
}

template <bool W8>
void launch_plain(const GemmArgs& g, hipStream_t st) {
  // the whole K in flight (96 KB of LDS at K = 768) while every tile has a CU of
  // its own; else half the ring, so that two tiles share a CU (128 rows, 288
  // tiles: QKV 5.4 us, against 6.3 with 64-row tiles of the whole K)
  if (plain_tiles(g) <= num_cus())
    launch_k<32, 4, W8>(g, st);
  else
    launch_k<32, 2, W8>(g, st);
}

// ---- residual products: a K slice per wave -----------------------------------
// 32 x 16 tiles; wave s takes slice s, C units of 64 k values, loads it into
// registers (coalesced, 128 bytes of a row per 8 lanes), passes each unit
// through its own LDS patch into the MFMA's layout, and leaves its sum in the
// patch.  X += ((slice 0 + slice 1) + ...) + bias, as the split-K epilogue.
template <int C, bool W8>
__global__ __launch_bounds__(1024) void gemm_short_resid_kernel(GemmArgs g) {
  constexpr int BM = 32, BN = 16, LDC = BN + 4, PATCH = (BM + BN) * 128;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  int tile_m, tile_n;
  short_tile(g.M / BM, tile_m, tile_n);
  const int m0 = tile_m * BM;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slices = static_cast<int>(blockDim.x) >> 6, units = g.K >> 6;
  const int u0 = wave * C, nu = min(C, units - u0);  // >= 1

  // the residual stream's two columns of this thread's item
  // (rows past a device row count do not exist: the last one's are read again)
  const int er = (tid & 255) / 8, en = tile_n * BN + 2 * (tid & 7);
  const int rows = g.M_dev ? *g.M_dev : g.M;
  float* xp = g.X + static_cast<int64_t>(min(m0 + er, rows - 1)) * g.ldx + min(en, g.N - 2);
  const f32x2_t x = *reinterpret_cast<const f32x2_t*>(xp);

  u32x4_t av[C][4], wv[C][W8 ? 1 : 2];
  const int l8 = lane & 7;
  const bf16_t* ab = static_cast<const bf16_t*>(g.A) + m0 * g.lda + u0 * 64;
  const uint32_t ao = static_cast<uint32_t>((lane >> 3) * static_cast<int>(g.lda) + l8 * 8);
#pragma unroll
  for (int i = 0; i < C; ++i)
    if (i < nu) {
#pragma unroll
      for (int a = 0; a < 4; ++a) av[i][a] = *reinterpret_cast<const u32x4_t*>(ab + 8 * a * g.lda + i * 64 + ao);
      if constexpr (W8) {
        wv[i][0] = *reinterpret_cast<const u32x4_t*>(
            static_cast<const uint8_t*>(g.W) + static_cast<int64_t>(min(tile_n * BN + (lane >> 2), g.N - 1)) * g.ldw +
            (u0 + i) * 64 + (lane & 3) * 16);
      } else {
#pragma unroll
        for (int a = 0; a < 2; ++a)
          wv[i][a] = *reinterpret_cast<const u32x4_t*>(
              static_cast<const bf16_t*>(g.W) +
              static_cast<int64_t>(min(tile_n * BN + 8 * a + (lane >> 3), g.N - 1)) * g.ldw + (u0 + i) * 64 + l8 * 8);
      }
    }

  char* pa = lds + wave * PATCH;
  char* pw = pa + BM * 128;
  auto swz = [](int r) { return (r >> 1) & 7; };
  // orders this wave's LDS accesses for the compiler (the hardware keeps them)
  auto order = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  f32x4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  const int r16 = lane & 15, q = lane >> 4;
#pragma unroll
  for (int i = 0; i < C; ++i) {
    if (i >= nu) break;
    order();
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int r = 8 * a + (lane >> 3);
      *reinterpret_cast<u32x4_t*>(pa + r * 128 + (l8 ^ swz(r)) * 16) = av[i][a];
    }
    if constexpr (W8) {
      const int r = lane >> 2, c = (lane & 3) * 2;
      *reinterpret_cast<bf16x8_t*>(pw + r * 128 + (c ^ swz(r)) * 16) = fp8x8_to_bf16(wv[i][0][0], wv[i][0][1]);
      *reinterpret_cast<bf16x8_t*>(pw + r * 128 + ((c + 1) ^ swz(r)) * 16) = fp8x8_to_bf16(wv[i][0][2], wv[i][0][3]);
    } else {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const int r = 8 * a + (lane >> 3);
        *reinterpret_cast<u32x4_t*>(pw + r * 128 + (l8 ^ swz(r)) * 16) = wv[i][a];
      }
    }
    order();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int o = r16 * 128 + ((4 * h + q) ^ swz(r16)) * 16;
      const bf16x8_t w = *reinterpret_cast<const bf16x8_t*>(pw + o);
#pragma unroll
      for (int t = 0; t < 2; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8_t*>(pa + t * 2048 + o), w, acc[t],
                                                         0, 0, 0);
    }
  }
  order();
  float* P = reinterpret_cast<float*>(pa);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) P[(t * 16 + 4 * q + e) * LDC + r16] = acc[t][e];
  __syncthreads();
  if (tid < 256 && en < g.N && m0 + er < rows) {
    f32x2_t v = {0.f, 0.f};
    const char* p = lds + (er * LDC + 2 * (tid & 7)) * 4;
    for (int s = 0; s < slices; ++s) {
      const f32x2_t t = *reinterpret_cast<const f32x2_t*>(p + s * PATCH);
      v[0] += t[0];
      v[1] += t[1];
    }
    if constexpr (W8) {
      v[0] *= g.w_scale[en];
      v[1] *= g.w_scale[en + 1];
    }
    if (g.bias) {
      v[0] += g.bias[en];
      v[1] += g.bias[en + 1];
    }
    *reinterpret_cast<f32x2_t*>(xp) = f32x2_t{x[0] + v[0], x[1] + v[1]};
  }
}

template <int C, bool W8>
void launch_resid(const GemmArgs& g, int slices, hipStream_t st) {
  constexpr int PATCH = 48 * 128;
  auto kern = gemm_short_resid_kernel<C, W8>;
  static const bool attr_set = [&] {
    hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  16 * PATCH),
              "gemm: LDS attribute");
    return true;
  }();
  (void)attr_set;
  kern<<<static_cast<unsigned>((g.N + 15) / 16 * (g.M / 32)), 64 * slices, slices * PATCH, st>>>(g);
}

bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

}  // namespace

bool gemm_short_ok(const GemmArgs& g) {
  const bool w8 = g.w_dtype == DT_FP8;
  if (g.ln_stats_in || g.ln_y || g.rln_y) return false;  // (no LayerNorm in these epilogues)
  if (g.M_dev && g.epi != EPI_RESID) return false;
  if (g.M <= 0 || g.M % 32 != 0 || g.M > kShortMaxRows || g.N < 2 || g.N % 2 != 0 || g.K <= 0 || g.K % 64 != 0)
    return false;
  if (g.in_dtype != DT_BF16 || !g.A || !aligned(g.A, 16) || g.lda % 8 != 0 || g.lda < g.K || g.lda >= (int64_t{1} << 28))
    return false;
  if (!g.W || !aligned(g.W, 16) || g.ldw < g.K || (!w8 && g.w_dtype != DT_BF16)) return false;
  if (w8 ? !(g.w_scale && g.ldw % 16 == 0) : g.ldw % 8 != 0) return false;
  if (g.epi == EPI_RESID) {
    int slices = 0, chunk = 0;
    split_k_slices(g.M, g.N, g.K, slices, chunk);
    return chunk <= 4 && slices >= 4 && slices <= 16 && g.X && aligned(g.X, 8) && g.ldx % 2 == 0 && g.ldx >= g.N;
  }
  if (g.K % 256 != 0 || g.K > 1024 || !g.out || g.out_dtype != DT_BF16 || !aligned(g.out, 4) || g.ldo % 2 != 0 || g.ldo < g.N)
    return false;
  if (g.epi == EPI_ROPE)
    return g.head_dim == 64 && g.N % 64 == 0 && g.rope_dim % 64 == 0 && g.pos && g.rope_cos && g.rope_sin &&
           aligned(g.rope_cos, 8) && aligned(g.rope_sin, 8) && g.rope_rows > 0 && 2 * g.rope_dim <= g.N && plain_pays(g);
  return (g.epi == EPI_STORE || (g.epi == EPI_GEGLU && g.N % 16 == 0)) && plain_pays(g);
}

void launch_gemm_short(const GemmArgs& g, hipStream_t st) {
  require(gemm_short_ok(g), "gemm: arguments outside the short-batch kernels' range");
  const bool w8 = g.w_dtype == DT_FP8;
  if (g.epi == EPI_RESID) {
    int slices = 0, chunk = 0;
    split_k_slices(g.M, g.N, g.K, slices, chunk);
    switch (chunk) {
      case 1: w8 ? launch_resid<1, true>(g, slices, st) : launch_resid<1, false>(g, slices, st); break;
      case 2: w8 ? launch_resid<2, true>(g, slices, st) : launch_resid<2, false>(g, slices, st); break;
      case 3: w8 ? launch_resid<3, true>(g, slices, st) : launch_resid<3, false>(g, slices, st); break;
      default: w8 ? launch_resid<4, true>(g, slices, st) : launch_resid<4, false>(g, slices, st); break;
    }
  } else {
    w8 ? launch_plain<true>(g, st) : launch_plain<false>(g, st);
  }
  check_launch("gemm_short");
}

}  // namespace sjh
