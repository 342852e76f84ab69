// FP32 GEMM C = A W^T + bias on gfx950 fp32 MFMA (v_mfma_f32_16x16x4f32),
// with optional GELU or residual-add epilogue.
//
// Replaces esm::kernels::Linear (reference src/kernels/gemm_fp32.cpp:33-46
// LinearRef, :272-294 LinearAvx512) for the all-fp32 8M model and for the
// fp32 lm head (dense d->d, tied decoder d->vocab; src/model.cpp:1192-1239).
// Products are exact fp32 products accumulated in fp32, so results differ
// from the sequential reference sum only by summation order.
//
// Three kernels (launch_gemm_f32 picks), and the decoder's:
//   - gemm_f32_tile_kernel: aligned rows with K % 16 == 0; LDS tiles of 32x32
//     to 128x64, direct global -> LDS stage loads;
//   - gemm_f32_pair_kernel: the same operands and the same sums bit for bit, for
//     grids too small for that one: two waves to a 16x16 tile;
//   - gemm_f32_kernel: any other shape (128x128 tiles through registers);
//   - gemm_narrow_kernel and gemm_narrow_rows_kernel: N <= 48, the sums of eight
//     ranges of K, by eight waves or one after the other.
// Which order a row is summed in is chosen by N, K and the alignment alone,
// never by M: a sequence's logits do not depend on what it is batched with.
//
// gemm_f32_kernel's tiling: 128x128 workgroup tile, four waves of 64x64,
// 32-wide K stages in LDS (row pitch 36 floats). Within a stage, lane group g
// (lane / 16) owns the eight consecutive k values [8g, 8g+8): MFMA step j
// multiplies A and W at k = 8g + j for every lane group, which keeps A and W
// consistent and lets each lane fetch its k values with two 16-byte LDS reads.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace esm_gfx950 {
namespace {

constexpr int BM = 128, BN = 128, BK = 32;
constexpr int kPitch = BK + 4;  // floats
constexpr int kThreads = 256;
constexpr int kStage = (BM + BN) * kPitch;

template <bool VEC>
__device__ __forceinline__ void load_stage(const float* __restrict__ base, int ld, int rows,
                                           int row0, int k0, int K, float4 (&r)[4]) {
  const int t = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int idx = t + kThreads * i;
    const int row = idx >> 3;
    const int c = (idx & 7) * 4;
    int gr = row0 + row;
    gr = gr < rows ? gr : rows - 1;
    const int kk = k0 + c;
    const float* src = base + static_cast<size_t>(gr) * ld + kk;
    if constexpr (VEC) {
      r[i] = kk < K ? *reinterpret_cast<const float4*>(src) : make_float4(0.f, 0.f, 0.f, 0.f);
    } else {
      r[i].x = kk + 0 < K ? src[0] : 0.f;
      r[i].y = kk + 1 < K ? src[1] : 0.f;
      r[i].z = kk + 2 < K ? src[2] : 0.f;
      r[i].w = kk + 3 < K ? src[3] : 0.f;
    }
  }
}

__device__ __forceinline__ void store_stage(float* s, const float4 (&r)[4]) {
  const int t = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int idx = t + kThreads * i;
    *reinterpret_cast<float4*>(s + (idx >> 3) * kPitch + (idx & 7) * 4) = r[i];
  }
}

template <int EPI, bool VEC>
__global__ __launch_bounds__(kThreads, 2) void gemm_f32_kernel(const GemmF32Args p) {
  __shared__ __attribute__((aligned(16))) float smem[2 * kStage];
  const int tiles_n = (p.N + BN - 1) / BN;
  const int m0 = (blockIdx.x / tiles_n) * BM;
  const int n0 = (blockIdx.x % tiles_n) * BN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int lr = lane & 15, lg = lane >> 4;

  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  float4 ra[4], rb[4];
  const int nk = (p.K + BK - 1) / BK;
  load_stage<VEC>(p.A, p.lda, p.M, m0, 0, p.K, ra);
  load_stage<VEC>(p.W, p.ldw, p.N, n0, 0, p.K, rb);
  store_stage(smem, ra);
  store_stage(smem + BM * kPitch, rb);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const float* cur = smem + (kt & 1) * kStage;
    const bool more = kt + 1 < nk;
    if (more) {
      load_stage<VEC>(p.A, p.lda, p.M, m0, (kt + 1) * BK, p.K, ra);
      load_stage<VEC>(p.W, p.ldw, p.N, n0, (kt + 1) * BK, p.K, rb);
    }
    float fa[4][8], fb[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* pa = cur + (wm * 64 + i * 16 + lr) * kPitch + lg * 8;
      const float* pb = cur + BM * kPitch + (wn * 64 + i * 16 + lr) * kPitch + lg * 8;
      const float4 a0 = *reinterpret_cast<const float4*>(pa);
      const float4 a1 = *reinterpret_cast<const float4*>(pa + 4);
      const float4 b0 = *reinterpret_cast<const float4*>(pb);
      const float4 b1 = *reinterpret_cast<const float4*>(pb + 4);
      fa[i][0] = a0.x; fa[i][1] = a0.y; fa[i][2] = a0.z; fa[i][3] = a0.w;
      fa[i][4] = a1.x; fa[i][5] = a1.y; fa[i][6] = a1.z; fa[i][7] = a1.w;
      fb[i][0] = b0.x; fb[i][1] = b0.y; fb[i][2] = b0.z; fb[i][3] = b0.w;
      fb[i][4] = b1.x; fb[i][5] = b1.y; fb[i][6] = b1.z; fb[i][7] = b1.w;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int n = 0; n < 4; ++n)
          acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[i][j], fb[n][j], acc[i][n], 0, 0, 0);
    if (more) {
      float* nxt = smem + ((kt + 1) & 1) * kStage;
      store_stage(nxt, ra);
      store_stage(nxt + BM * kPitch, rb);
    }
    __syncthreads();
  }

  const int rb0 = m0 + wm * 64, cb0 = n0 + wn * 64;
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const int col = cb0 + n * 16 + lr;
    if (col >= p.N) continue;
    const float b = p.bias ? p.bias[col] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = rb0 + i * 16 + lg * 4 + r;
        if (row >= p.M) continue;
        float v = acc[i][n][r] + b;
        float* dst = p.C + static_cast<size_t>(row) * p.ldc + col;
        if constexpr (EPI == kF32Gelu) v = gelu_erf(v);
        if constexpr (EPI == kF32Resid) {
          *dst += v;
        } else {
          *dst = v;
        }
      }
  }
}

// ---- Tiled fp32 GEMM (K % 16 == 0, 16-byte aligned rows): 2 x 2 waves of
// 16 MB x 16 NB outputs, a 32 MB x 32 NB workgroup tile.
//
// Staging is the INT8 kernel's: K advances 128 bytes (32 floats) a stage, one
// global_load_lds_dwordx4 per 8 rows x 128 bytes, chunk c of row r at c ^ r
// within its 1 KB block, two or three stage buffers and one barrier a stage.
// A lane reads 16 bytes, k = 16 h + 4 lg .. + 4 of row lr, per half h of the
// stage; MFMA step j multiplies k = 16 h + 4 lg + j. The operands are swapped
// (W rows in the M dimension), so a lane's four accumulators are four
// consecutive columns of one row and go out as one 16-byte store.
//
// v_mfma_f32_16x16x4_f32 takes 32 cycles for 512 operand bytes, so neither LDS
// nor the stage loads bound the loop; what does is the matrix rate times how
// evenly the tiles fall on the CUs (tile_of). 1280 x 1280 at 7,777 rows:
// 303 us with 128x128 tiles staged through registers, 199 here (128 TFLOP/s;
// 165 us at the rate of a large fp32 library product); at 66 rows and K = N =
// 320, 33 -> 4.8 us.
// X3: the split-fp16 GEMM on the same stages. A row of A or W holds, for each
// 32 k, 64 bytes of hi parts and 64 bytes of lo parts (GemmX3Args), so a
// 128-byte piece is again one K stage: chunk lg is a lane's eight hi halves, k
// = 8 lg .. + 8, and chunk 4 + lg its lo halves, the operands of one
// v_mfma_f32_16x16x32_f16 each; three of them per 16x16 block and stage (hi hi
// + lo hi + hi lo). They take 48 cycles where the fp32 MFMAs take 256, so here
// the stage traffic bounds the loop and the tiles want to be large. With A
// split while it was staged through registers (128x128 tiles, 64-byte rows) the
// ESM-2 650M lm dense took 58 / 62 / 409 us at 301 / 2,048 / 31,107 rows; 15 /
// 35 / 359 here.
//
// The order of an output's sum depends on K alone: over kSumStages stages one
// sum of the first and one of the second halves, the two added, and those added
// in turn. The last half stage of a K that is an odd multiple of 16 is a sum of its
// own, added last, its operands read straight into registers (f32_tail).
// gemm_f32_pair_kernel has the same. Sums of 160 products keep the
// error of the eight-way split that small grids had before, at K = 1280 0.36 of
// one long sum's standard deviation, and cost the large tiles 1% (2560 x 2560 at
// 16,000 rows 1,488 -> 1,501 us). A second sum also keeps a 32x32 tile's wave off
// a single chain of dependent MFMAs.
constexpr int kSumStages = 10;
template <int MB, int NB>
struct F32Tile {
  static constexpr int BM = 32 * MB, BN = 32 * NB;
  static constexpr int kBlocks = (BM + BN) / 8;  // 1 KB blocks per stage
  static constexpr int kPer = kBlocks / 4;       // per wave
  static constexpr int kStage = kBlocks * 1024;
  // More buffers only cost resident workgroups (1280 x 1280 at 1,000 rows,
  // 32x32 tiles: 33 us with three, 39 with five).
  static constexpr int kNStage = kStage <= 16384 ? 3 : 2;
};

// Output of four consecutive columns of one row, the epilogue applied.
// X3: the sums are first multiplied by c_unscale, in one rounding with the bias.
template <int EPI, bool X3>
__device__ __forceinline__ void f32_store4(const GemmF32Args& p, int row, int col, f32x4 v, bool vec_c) {
  if (row >= p.M || col >= p.N) return;
  float* dst = p.C + static_cast<size_t>(row) * p.ldc + col;
  const int n = min(4, p.N - col);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float b = p.bias && e < n ? p.bias[col + e] : 0.0f;
    v[e] = X3 ? __builtin_fmaf(v[e], p.c_unscale, b) : v[e] + b;
    if constexpr (EPI == kF32Gelu) v[e] = gelu_erf(v[e]);
  }
  if (vec_c && n == 4) {
    if constexpr (EPI == kF32Resid) v = *reinterpret_cast<const f32x4*>(dst) + v;
    *reinterpret_cast<f32x4*>(dst) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < n) dst[e] = EPI == kF32Resid ? dst[e] + v[e] : v[e];
  }
}

// kF32QkvRope, 16-wide heads: a 16-column block is one head, the lane's four
// columns dims 4 lg .. + 4 of it, and the other half of its rotary pairs is in
// lane ^ 32. The products of launch_rope_f32, in its fused forms; a pass of its
// own per layer and operand took 2.6 / 4.7 us each at 66 / 1,768 rows.
__device__ __forceinline__ f32x4 rope16(const GemmF32Args& p, int row, int col, f32x4 v) {
  const int n0 = __builtin_amdgcn_readfirstlane(col) & ~15;
  if (n0 >= 2 * p.d_model) return v;
  const int lane = threadIdx.x & 63, d0 = 4 * (lane >> 4);
  const size_t at = static_cast<size_t>(p.pos[min(row, p.M - 1)]) * 16 + d0;
  const f32x4 c = *reinterpret_cast<const f32x4*>(p.rope_cos + at);
  const f32x4 s = *reinterpret_cast<const f32x4*>(p.rope_sin + at);
  const float f = n0 < p.d_model ? p.q_scale : 1.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    // The swap leaves dim d0 % 8 + e's value first, its partner's second, in
    // both halves of the wave.
    const LanePair x = lane_xor32(v[e] * f);
    v[e] = lane < 32 ? __builtin_fmaf(x.a, c[e], -(x.b * s[e])) : __builtin_fmaf(x.b, c[e], x.a * s[e]);
  }
  return v;
}

// Four consecutive columns of one row, as a wave holds a 16x16 block (lane (lr,
// lg): row lr, columns 4 lg .. + 4; every lane reaches this).
template <int EPI, bool X3>
__device__ __forceinline__ void f32_out(const GemmF32Args& p, int row, int col, f32x4 v, bool vec_c) {
  if constexpr (EPI == kF32QkvRope) {
    // N is a multiple of 16 (gemm_f32_rope_ok), so a block is in or out.
    if (col >= p.N) return;
    if (p.bias) v += *reinterpret_cast<const f32x4u*>(p.bias + col);
    v = rope16(p, row, col, v);
    if (row < p.M) *reinterpret_cast<f32x4*>(p.C + static_cast<size_t>(row) * p.ldc + col) = v;
  } else {
    f32_store4<EPI, X3>(p, row, col, v, vec_c);
  }
}

// A lane's operands of the last 16 k: 4 lg .. + 4 of them, of a row of A or W.
__device__ __forceinline__ f32x4 f32_tail(const float* base, int ld, int row, int K) {
  return *reinterpret_cast<const f32x4*>(base + static_cast<size_t>(row) * ld + (K - 16 + 4 * ((threadIdx.x >> 4) & 3)));
}

// TAIL: K is an odd multiple of 16 (640 x 528 at 66 / 301 / 8,000 rows 4.2 / 7.0 / 54
// us; 48.8 / 48.8 / 93.9 in the general kernel). A kernel of its own: the same
// test made at run time cost the others four registers and up to 10%.
template <bool X3, int MB, int NB, bool TAIL, int EPI>
__global__ __launch_bounds__(256, MB * NB == 16 ? 1 : 3) void gemm_f32_tile_kernel(const GemmF32Args p, bool vec_c) {
  using TL = F32Tile<MB, NB>;
  constexpr int BM = TL::BM, BN = TL::BN, kPer = TL::kPer, kStage = TL::kStage, kNStage = TL::kNStage;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kNStage * kStage];
  int m0, n0;
  tile_origin_of(blockIdx.x, p.M, p.N, BM, BN, &m0, &n0);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int lr = lane & 15, lg = lane >> 4;

  // Blocks wave * kPer .. of a stage: [0, BM / 8) are A row groups, the rest
  // W row groups; rows past the edge re-read the last valid row.
  uint32_t goff[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int b = wave * kPer + i;
    const int r = lane >> 3, c = (lane & 7) ^ r;
    const bool is_a = b < BM / 8;
    const int row = is_a ? min(m0 + b * 8 + r, p.M - 1) : min(n0 + (b - BM / 8) * 8 + r, p.N - 1);
    goff[i] = (static_cast<uint32_t>(row) * static_cast<uint32_t>(is_a ? p.lda : p.ldw) + c * 4) * 4u;
  }
  const uint32_t lds0 = lds_byte_addr(smem);
  auto load_stage = [&](int kt, int buf) {
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      lds_dma16((wave * kPer + i < BM / 8 ? p.A : p.W) + kt * 32, goff[i],
                lds0 + static_cast<uint32_t>(buf * kStage + (wave * kPer + i) * 1024));
  };
  const int nk = p.K / 32;
#pragma unroll
  for (int st = 0; st < kNStage - 1; ++st)
    if (st < nk) load_stage(st, st);

  // fp32: one sum of the first and one of the second halves of the stages.
  constexpr int kChains = X3 ? 1 : 2;
  f32x4 acc[kChains][MB][NB];
  // Row R's chunk c of a stage: block R / 8, slot c ^ (R % 8).
  const int arow = wm * 16 * MB + lr, wrow = BM + wn * 16 * NB + lr;
  using Frag = std::conditional_t<X3, f16x8, f32x4>;
  auto frag = [&](const uint8_t* st, int R, int h) {
    return *reinterpret_cast<const Frag*>(st + (R >> 3) * 1024 + (R & 7) * 128 + (((4 * h + lg) ^ (R & 7)) << 4));
  };
  int buf = 0;
  // first: the sums start with this stage.
  auto stage = [&](int kt, auto first) {
    constexpr bool FIRST = decltype(first)::value;
    // Stage kt has landed (this wave's loads, then everyone's behind the
    // barrier), and every wave is done with stage kt - 1, whose buffer
    // receives stage kt + kNStage - 1.
    if (kNStage == 3 && kt + 1 < nk)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kPer) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (kt + kNStage - 1 < nk) load_stage(kt + kNStage - 1, buf == 0 ? kNStage - 1 : buf - 1);
    const uint8_t* st = smem + buf * kStage;
    buf = buf + 1 == kNStage ? 0 : buf + 1;
    if constexpr (X3) {
      f16x8 ah[MB], al[MB], wh[NB], wl[NB];
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        ah[i] = frag(st, arow + 16 * i, 0);
        al[i] = frag(st, arow + 16 * i, 1);
      }
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        wh[j] = frag(st, wrow + 16 * j, 0);
        wl[j] = frag(st, wrow + 16 * j, 1);
      }
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          f32x4 c = FIRST ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[0][i][j];
          c = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[j], ah[i], c, 0, 0, 0);
          c = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[j], al[i], c, 0, 0, 0);
          acc[0][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wl[j], ah[i], c, 0, 0, 0);
        }
    } else {
      // A single-block wave advances both sums together: one alone is a chain
      // of dependent MFMAs, 52 cycles each instead of the 32 they occupy the
      // matrix core. Otherwise one half of the stage at a time keeps fewer
      // fragments live.
      constexpr int kPair = MB * NB == 1 ? 2 : 1;
#pragma unroll
      for (int h0 = 0; h0 < 2; h0 += kPair) {
        f32x4 fa[kPair][MB], fw[kPair][NB];
#pragma unroll
        for (int x = 0; x < kPair; ++x) {
#pragma unroll
          for (int i = 0; i < MB; ++i) fa[x][i] = frag(st, arow + 16 * i, h0 + x);
#pragma unroll
          for (int j = 0; j < NB; ++j) fw[x][j] = frag(st, wrow + 16 * j, h0 + x);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int x = 0; x < kPair; ++x)
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
              for (int j = 0; j < NB; ++j) {
                const f32x4 c = FIRST && e == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[h0 + x][i][j];
                acc[h0 + x][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[x][j][e], fa[x][i][e], c, 0, 0, 0);
              }
      }
    }
  };
  constexpr int kSum = X3 ? 1 << 30 : kSumStages;
  f32x4 total[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int kb = 0; kb < nk; kb += kSum) {
    stage(kb, std::true_type{});
    for (int kt = kb + 1; kt < min(kb + kSum, nk); ++kt) stage(kt, std::false_type{});
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        f32x4 v = acc[0][i][j];
        if constexpr (!X3) v += acc[1][i][j];
        total[i][j] += v;
      }
  }
  if constexpr (TAIL) {
    f32x4 fa[MB], fw[NB];
#pragma unroll
    for (int i = 0; i < MB; ++i) fa[i] = f32_tail(p.A, p.lda, min(m0 + arow + 16 * i, p.M - 1), p.K);
#pragma unroll
    for (int j = 0; j < NB; ++j) fw[j] = f32_tail(p.W, p.ldw, min(n0 + wrow - BM + 16 * j, p.N - 1), p.K);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) v = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[j][e], fa[i][e], v, 0, 0, 0);
        total[i][j] += v;
      }
  }
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const f32x4 v = total[i][j];
      const int row = m0 + wm * 16 * MB + 16 * i + lr, col = n0 + wn * 16 * NB + 16 * j + 4 * lg;
      f32_out<EPI, X3>(p, row, col, v, vec_c);
    }
}

// ---- The same sums for grids of few tiles: a 16x16 output tile per workgroup
// of two waves, one for the first and one for the second halves of the stages,
// which leave their sums in LDS for the first wave to add up. A wave's
// operands of a K stage are 16 bytes a lane of A and of W (lane (lr, lg): k =
// 16 h + 4 lg .. + 4 of row lr), so it keeps a ring of D stages of its own in
// LDS, filled by direct loads and read back lane by lane, with no barrier
// before the two sums meet: what the launch takes is the chain of dependent
// MFMAs and one load latency. N = 320 at 66 rows: K = 320 / 640 / 1280 in 3.3 /
// 4.4 / 6.7 us, where 32x32 tiles take 4.9 / 7.3 / 12.5. (A ring in registers
// took 3.6 / 4.7 / 8.6, before the sums were cut: the compiler waits for every
// load in flight at the loop's head. A wave for each sum, its operands straight
// into registers, took 3.3 / 4.4 / 6.8 to 7.8.)
constexpr int kPairSums = 32;  // at most, without the last half stage's: K <= 32 kSumStages kPairSums
template <int D, bool TAIL, int EPI>
__global__ __launch_bounds__(128) void gemm_f32_pair_kernel(const GemmF32Args p, bool vec_c) {
  constexpr int kStage = 2048;  // 1 KB of A, 1 KB of W
  __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * D * kStage];
  __shared__ f32x4 sums[2][kPairSums][64];
  const int lane = threadIdx.x & 63, half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int m0 = blockIdx.x * 16, n0 = blockIdx.y * 16;
  const float* a = p.A + static_cast<size_t>(m0) * p.lda + 16 * half;
  const float* w = p.W + static_cast<size_t>(n0) * p.ldw + 16 * half;
  const uint32_t aoff = (static_cast<uint32_t>(min(lr, p.M - 1 - m0)) * static_cast<uint32_t>(p.lda) + 4 * lg) * 4u;
  const uint32_t woff = (static_cast<uint32_t>(min(lr, p.N - 1 - n0)) * static_cast<uint32_t>(p.ldw) + 4 * lg) * 4u;
  uint8_t* ring = smem + half * D * kStage;
  const uint32_t lds = lds_byte_addr(ring);
  auto load = [&](int kt, int slot) {
    lds_dma16(a + 32 * kt, aoff, lds + static_cast<uint32_t>(slot * kStage));
    lds_dma16(w + 32 * kt, woff, lds + static_cast<uint32_t>(slot * kStage + 1024));
  };
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 fa, fw;
  auto read = [&](int slot) {
    fa = *reinterpret_cast<const f32x4*>(ring + slot * kStage + lane * 16);
    fw = *reinterpret_cast<const f32x4*>(ring + slot * kStage + 1024 + lane * 16);
  };
  // The last half stage, first to be loaded, belongs to the first wave.
  f32x4 ta, tw;
  if (TAIL && half == 0) {
    ta = f32_tail(p.A, p.lda, min(m0 + lr, p.M - 1), p.K);
    tw = f32_tail(p.W, p.ldw, min(n0 + lr, p.N - 1), p.K);
  }
  const int nk = p.K / 32;
  int slot = 0, in_sum = 0, nsum = 0;
  auto multiply = [&] {
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[e], fa[e], acc, 0, 0, 0);
    slot = slot + 1 == D ? 0 : slot + 1;
    if (++in_sum == kSumStages) {
      sums[half][nsum++][lane] = acc;
      acc = f32x4{0.f, 0.f, 0.f, 0.f};
      in_sum = 0;
    }
  };
#pragma unroll
  for (int u = 0; u < D; ++u)
    if (u < nk) load(u, u);
  // Stage kt is read into registers, its slot refilled (once the reads are
  // back), and then multiplied.
  for (int kt = 0; kt + D < nk; ++kt) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (D - 1)) : "memory");
    read(slot);
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(fa), "+v"(fw)::"memory");
    load(kt + D, slot);
    multiply();
  }
  // The last min(D, nk) stages are on their way, `later` of them after this one.
#pragma unroll
  for (int later = D - 1; later >= 0; --later)
    if (later < nk) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * later) : "memory");
      read(slot);
      multiply();
    }
  if (in_sum > 0) sums[half][nsum++][lane] = acc;
  __syncthreads();
  if (half == 1) return;
  f32x4 total = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int x = 0; x < nsum; ++x) total += sums[0][x][lane] + sums[1][x][lane];
  if constexpr (TAIL) {
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) v = __builtin_amdgcn_mfma_f32_16x16x4f32(tw[e], ta[e], v, 0, 0, 0);
    total += v;
  }
  f32_out<EPI, false>(p, m0 + lr, n0 + 4 * lg, total, vec_c);
}

// ---- Narrow fp32 GEMM (N <= 48, the tied decoder; K % 16 == 0): a 16 MB x 48
// output tile whose K is split over the workgroup's eight waves. Each wave
// loads its 16-wide K steps straight into registers (lane (lr, lg): k = 16 s +
// 4 lg .. + 4 of row lr), CH steps in flight at once, and the waves' sums meet
// in LDS in wave order.
constexpr int kNarrowBlocks = 3;
constexpr int kNarrowWaves = 8;
template <int MB, int CH>
__global__ __launch_bounds__(kNarrowWaves * 64) void gemm_narrow_kernel(const GemmF32Args p, bool vec_c) {
  constexpr int NB = kNarrowBlocks;
  __shared__ f32x4 part[kNarrowWaves][MB * NB][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int m0 = blockIdx.x * 16 * MB;
  const float* arow[MB];
  const float* wrow[NB];
#pragma unroll
  for (int i = 0; i < MB; ++i) arow[i] = p.A + static_cast<size_t>(min(m0 + 16 * i + lr, p.M - 1)) * p.lda + 4 * lg;
#pragma unroll
  for (int j = 0; j < NB; ++j) wrow[j] = p.W + static_cast<size_t>(min(16 * j + lr, p.N - 1)) * p.ldw + 4 * lg;
  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = p.K / 16;
  const int s0 = steps * wave / kNarrowWaves, s1 = steps * (wave + 1) / kNarrowWaves;
  for (int s = s0; s < s1; s += CH) {
    f32x4 fa[CH][MB], fw[CH][NB];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int k0 = 16 * min(s + u, s1 - 1);  // past the range: its last step again, unused
#pragma unroll
      for (int i = 0; i < MB; ++i) fa[u][i] = *reinterpret_cast<const f32x4*>(arow[i] + k0);
#pragma unroll
      for (int j = 0; j < NB; ++j) fw[u][j] = *reinterpret_cast<const f32x4*>(wrow[j] + k0);
    }
#pragma unroll
    for (int u = 0; u < CH; ++u)
      if (s + u < s1) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[u][j][e], fa[u][i][e], acc[i][j], 0, 0, 0);
      }
  }
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) part[wave][i * NB + j][lane] = acc[i][j];
  __syncthreads();
  // Wave w finishes block w.
  if (wave >= MB * NB) return;
  f32x4 v = part[0][wave][lane];
#pragma unroll
  for (int w = 1; w < kNarrowWaves; ++w) v += part[w][wave][lane];
  f32_store4<kF32Store, false>(p, m0 + 16 * (wave / NB) + lr, 16 * (wave % NB) + 4 * lg, v, vec_c);
}

// The same sums for many rows (K % 32 == 0): with enough of them to fill the chip
// K need not be split, and eight waves that each read 64 bytes of a row at a
// time only cost. Four waves of 16 rows share stages of 32 k (A's rows and the 48
// of W) moved and laid out as in the tiled kernel; a wave walks the eight ranges
// of K one after the other and adds each to its total. 31,107 x 33 x 1280: 72 ->
// 39 us, 4.1 TB/s of A; its MFMAs alone are 26. (32 rows a wave leave a CU one
// workgroup and nothing to cover its barriers: 46 us.)
constexpr int kNarrowRows = 64;
__global__ __launch_bounds__(256, 2) void gemm_narrow_rows_kernel(const GemmF32Args p, bool vec_c) {
  constexpr int NB = kNarrowBlocks, BM = kNarrowRows;
  constexpr int kBlocks = BM / 8 + 2 * NB;
  constexpr int kPer = (kBlocks + 3) / 4;  // the last ones move W's last row again
  constexpr int kStage = 4 * kPer * 1024, kNStage = 3;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kNStage * kStage];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int m0 = blockIdx.x * BM;
  const float* a = p.A + static_cast<size_t>(m0) * p.lda;
  uint32_t goff[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int b = wave * kPer + i;
    const int r = lane >> 3, c = (lane & 7) ^ r;
    const bool is_a = b < BM / 8;
    const int row = is_a ? min(b * 8 + r, p.M - 1 - m0) : min((b - BM / 8) * 8 + r, p.N - 1);
    goff[i] = (static_cast<uint32_t>(row) * static_cast<uint32_t>(is_a ? p.lda : p.ldw) + c * 4) * 4u;
  }
  const uint32_t lds0 = lds_byte_addr(smem);
  auto load_stage = [&](int kt, int buf) {
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      lds_dma16((wave * kPer + i < BM / 8 ? a : p.W) + kt * 32, goff[i],
                lds0 + static_cast<uint32_t>(buf * kStage + (wave * kPer + i) * 1024));
  };
  const int nk = p.K / 32;
#pragma unroll
  for (int st = 0; st < kNStage - 1; ++st)
    if (st < nk) load_stage(st, st);
  const int arow = wave * 16 + lr, wrow = BM + lr;
  auto frag = [&](const uint8_t* st, int R, int h) {
    return *reinterpret_cast<const f32x4*>(st + (R >> 3) * 1024 + (R & 7) * 128 + (((4 * h + lg) ^ (R & 7)) << 4));
  };
  f32x4 acc[NB], total[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) acc[j] = total[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = 2 * nk;
  int range = 0, end = steps / kNarrowWaves, buf = 0;
  for (int kt = 0; kt < nk; ++kt) {
    // As in the tiled kernel: stage kt has landed, and the buffer of stage kt - 1
    // receives stage kt + kNStage - 1.
    if (kt + 1 < nk)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kPer) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (kt + kNStage - 1 < nk) load_stage(kt + kNStage - 1, buf == 0 ? kNStage - 1 : buf - 1);
    const uint8_t* st = smem + buf * kStage;
    buf = buf + 1 == kNStage ? 0 : buf + 1;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // The ranges that end before this step (with K < 128 some are empty: zero).
      while (2 * kt + h == end) {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          total[j] = range == 0 ? acc[j] : total[j] + acc[j];
          acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        ++range;
        end = steps * (range + 1) / kNarrowWaves;
      }
      const f32x4 fa = frag(st, arow, h);
      f32x4 fw[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) fw[j] = frag(st, wrow + 16 * j, h);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[j][e], fa[e], acc[j], 0, 0, 0);
    }
  }
  // The eighth range ends with K.
#pragma unroll
  for (int j = 0; j < NB; ++j)
    f32_store4<kF32Store, false>(p, m0 + arow, 16 * j + 4 * lg, total[j] + acc[j], vec_c);
}

}  // namespace

namespace {

bool f32_vec_c(const GemmF32Args& p) { return p.ldc % 4 == 0 && reinterpret_cast<uintptr_t>(p.C) % 16 == 0; }

// One EPI of a kernel template instantiated for each fp32 epilogue.
#define ESM_F32_EPI(KERNEL, ...)                                                              \
  switch (epi) {                                                                              \
    case kF32Store: hipLaunchKernelGGL((KERNEL<__VA_ARGS__, kF32Store>), grid, block, 0, s, p, vec_c); break; \
    case kF32Gelu: hipLaunchKernelGGL((KERNEL<__VA_ARGS__, kF32Gelu>), grid, block, 0, s, p, vec_c); break;   \
    case kF32Resid: hipLaunchKernelGGL((KERNEL<__VA_ARGS__, kF32Resid>), grid, block, 0, s, p, vec_c); break; \
    default: return hipErrorInvalidValue;                                                     \
  }                                                                                           \
  return hipGetLastError()

template <bool X3, int MB, int NB, bool TAIL = false>
hipError_t launch_f32_tile(const GemmF32Args& p, int epi, hipStream_t s) {
  using TL = F32Tile<MB, NB>;
  const bool vec_c = f32_vec_c(p);
  const dim3 grid(((p.M + TL::BM - 1) / TL::BM) * ((p.N + TL::BN - 1) / TL::BN)), block(256);
  if constexpr (!X3 && !TAIL) {
    if (p.K % 32 != 0) return launch_f32_tile<false, MB, NB, true>(p, epi, s);
    if (epi == kF32QkvRope) {
      hipLaunchKernelGGL((gemm_f32_tile_kernel<false, MB, NB, false, kF32QkvRope>), grid, block, 0, s, p, vec_c);
      return hipGetLastError();
    }
  }
  ESM_F32_EPI(gemm_f32_tile_kernel, X3, MB, NB, TAIL);
}

hipError_t launch_f32_pair(const GemmF32Args& p, int epi, hipStream_t s) {
  const bool vec_c = f32_vec_c(p);
  const dim3 grid((p.M + 15) / 16, (p.N + 15) / 16), block(128);
  constexpr int kAhead = 4;  // 16 KB of LDS; 8, 12 or 16 were no faster
  if (epi == kF32QkvRope) {
    hipLaunchKernelGGL((gemm_f32_pair_kernel<kAhead, false, kF32QkvRope>), grid, block, 0, s, p, vec_c);
    return hipGetLastError();
  }
  if (p.K % 32 != 0) {
    ESM_F32_EPI(gemm_f32_pair_kernel, kAhead, true);
  }
  ESM_F32_EPI(gemm_f32_pair_kernel, kAhead, false);
}

template <int MB, int CH>
hipError_t launch_narrow(const GemmF32Args& p, hipStream_t s) {
  hipLaunchKernelGGL((gemm_narrow_kernel<MB, CH>), dim3((p.M + 16 * MB - 1) / (16 * MB)), dim3(kNarrowWaves * 64), 0, s,
                     p, f32_vec_c(p));
  return hipGetLastError();
}

hipError_t launch_narrow_rows(const GemmF32Args& p, hipStream_t s) {
  hipLaunchKernelGGL(gemm_narrow_rows_kernel, dim3((p.M + kNarrowRows - 1) / kNarrowRows), dim3(256), 0, s, p,
                     f32_vec_c(p));
  return hipGetLastError();
}

constexpr uint64_t kOffsetLimit = 1ull << 32;  // bytes that 32-bit lane offsets reach

// 16-byte aligned rows of A and W.
bool f32_rows_ok(const GemmF32Args& p) {
  return p.lda % 4 == 0 && p.ldw % 4 == 0 &&
         (reinterpret_cast<uintptr_t>(p.A) | reinterpret_cast<uintptr_t>(p.W)) % 16 == 0;
}

// The tiled kernel's (and the pair kernel's) operands: whole and half K stages of
// aligned rows, W within the stage loads' offsets. A beyond them goes in pieces
// (f32_pieces), so which order a row is summed in does not depend on M.
bool f32_tile_ok(const GemmF32Args& p) {
  return p.K > 0 && p.K % 16 == 0 && f32_rows_ok(p) && static_cast<uint64_t>(p.N) * p.ldw * 4 <= kOffsetLimit &&
         static_cast<uint64_t>(p.lda) * 4 <= kOffsetLimit;
}

// Runs launch on pieces of rows of A that 32-bit offsets reach.
template <class F>
hipError_t f32_pieces(const GemmF32Args& p, F launch) {
  const int most = static_cast<int>(std::min<uint64_t>(1 << 30, kOffsetLimit / (static_cast<uint64_t>(p.lda) * 4)));
  for (int m0 = 0; m0 < p.M; m0 += most) {
    GemmF32Args q = p;
    q.A += static_cast<size_t>(m0) * p.lda;
    q.C += static_cast<size_t>(m0) * p.ldc;
    if (q.pos) q.pos += m0;
    q.M = std::min(most, p.M - m0);
    const hipError_t e = launch(q);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// Tiles 0 .. n - 1 of {32x32, 64x64, 128x64, 128x128}: the one whose grid
// takes the least time, (the most tiles any CU gets + the ends of its work, in
// tiles) x the tile's outputs x its cost per output.
constexpr int kTileRows[4] = {32, 64, 128, 128}, kTileCols[4] = {32, 64, 64, 128};
template <class Ends>
int tile_of(int M, int N, int n, const double* cost, Ends ends) {
  const int cus = device_cus();
  int best = 0;
  double best_t = 0.0;
  for (int t = 0; t < n; ++t) {
    const long tiles = static_cast<long>((M + kTileRows[t] - 1) / kTileRows[t]) * ((N + kTileCols[t] - 1) / kTileCols[t]);
    const long most = (tiles + cus - 1) / cus;
    const double c = (static_cast<double>(most) + ends(most)) * kTileRows[t] * kTileCols[t] * cost[t];
    if (t == 0 || c < best_t) {
      best = t;
      best_t = c;
    }
  }
  return best;
}

// fp32: the first loads and the last stores of a CU's tiles take about three K
// stages, and a CU with a single tile leaves its matrix cores waiting longer.
// 32x32 / 64x64 / 128x64 tiles: 2560 x 2560 at 16,000 rows 1,718 / 1,535 / 1,506
// us; 1280 x 1280 at 1,000 rows 32 / 44 / 49 us, at 1,768 53 / 62 / 80, at 3,000
// 86 / 86 / 81, at 7,777 214 / 202 / 197, at 16,000 429 / 396 / 391. Over 20 row
// counts of 66 .. 16,000 at nine N x K of 320 .. 3840 x 96 .. 2560 the choice is
// 0.3% off the fastest on average, 9% at 16,000 x 320 x 320 and 8% at 16,000 x
// 320 x 1280, where 32x32 is, and 4% at most elsewhere. (64x32 and 128x128 tiles
// were never more than 8% faster.)
constexpr double kF32Cost[3] = {1.14, 1.02, 1.0};

int f32_tile(const GemmF32Args& p) {
  return tile_of(p.M, p.N, 3, kF32Cost, [&](long most) { return 3.0 * 32 / p.K + (most == 1 ? 0.2 : 0.0); });
}

// Split-fp16, bound by the stage traffic: 1280 x 1280 takes 15 / 21 / 35 / 48 us
// at 301 rows, 45 / 35 / 38 / 50 at 2,048, 148 / 103 / 91 / 110 at 7,562, - / 423
// / 376 / 359 at 31,107; 2560 x 2560 at 7,562 rows 617 / 358 / 339 / 305.
// The last round, in which a CU's few remaining workgroups wait for their loads,
// counts for half a tile.
constexpr double kX3Cost[4] = {2.2, 1.18, 1.07, 1.0};

hipError_t launch_x3_tile(const GemmF32Args& p, int epi, hipStream_t s) {
  switch (tile_of(p.M, p.N, 4, kX3Cost, [](long) { return 0.5; })) {
    case 0: return launch_f32_tile<true, 1, 1>(p, epi, s);
    case 1: return launch_f32_tile<true, 2, 2>(p, epi, s);
    case 2: return launch_f32_tile<true, 4, 2>(p, epi, s);
    default: return launch_f32_tile<true, 4, 4>(p, epi, s);
  }
}

}  // namespace

hipError_t launch_gemm_narrow(const GemmF32Args& p, hipStream_t s) {
  if (p.M <= 0 || p.N <= 0) return hipSuccess;
  if (p.N > 16 * kNarrowBlocks || p.K <= 0 || p.K % 16 != 0 || !f32_rows_ok(p)) return hipErrorInvalidValue;
  // 16 rows a workgroup while there is one for every CU, then 32, and past one of
  // those for every CU no K split. N = 33, K = 1280 with 16 / 32 / no split: 11.4
  // / 18.3 / 25.8 us at 3,000 rows, 21.0 / 19.5 / 26.0 at 6,400, 30.9 / 36.7 / 26.5
  // at 10,000, 81.0 / 71.9 / 38.6 at 31,107; K = 320 6.3 / 7.1 / 9.3, 9.9 / 7.3 /
  // 9.4, 13.8 / 12.1 / 9.7 and 33.4 / 22.8 / 14.1.
  const int cus = device_cus();
  if (p.M <= 16 * cus) return launch_narrow<1, 5>(p, s);
  if (p.M <= 32 * cus || p.K % 32 != 0) return launch_narrow<2, 4>(p, s);
  return launch_narrow_rows(p, s);
}

hipError_t launch_gemm_x3(const GemmX3Args& x, int epi, hipStream_t s) {
  if (x.M <= 0 || x.N <= 0) return hipSuccess;
  if (x.K <= 0 || x.K % 32 != 0) return hipErrorInvalidValue;
  // Larger operands than the stage loads' offsets reach go in pieces.
  const int most = static_cast<int>(std::min<uint64_t>(1 << 30, kOffsetLimit / (static_cast<uint64_t>(x.K) * 4)));
  for (int n0 = 0; n0 < x.N; n0 += most) {
    GemmF32Args p;
    // Rows of K / 32 pieces of 128 bytes: the fp32 kernel's pitches.
    p.A = reinterpret_cast<const float*>(x.A);
    p.W = reinterpret_cast<const float*>(x.W) + static_cast<size_t>(n0) * x.K;
    p.lda = p.ldw = p.K = x.K;
    p.c_unscale = x.w_unscale;
    p.bias = x.bias ? x.bias + n0 : nullptr;
    p.C = x.C + n0;
    p.ldc = x.ldc;
    p.M = x.M;
    p.N = std::min(most, x.N - n0);
    if (!f32_tile_ok(p)) return hipErrorInvalidValue;
    const hipError_t e = f32_pieces(p, [&](const GemmF32Args& q) { return launch_x3_tile(q, epi, s); });
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

namespace {

// At most two 16x16 tiles a CU, whose waves then have a SIMD each. N = 320, K =
// 320 / 1280: 4.4 / 11.2 us at 301 rows (380 tiles) against 4.9 / 12.6 in 32x32
// tiles, 5.5 / 15.7 at 450 rows (580 tiles) against 5.0 / 12.8.
bool f32_takes_pair(const GemmF32Args& p) {
  const long tiles16 = static_cast<long>((p.M + 15) / 16) * ((p.N + 15) / 16);
  return tiles16 <= 2 * device_cus() && p.K <= 32 * kSumStages * kPairSums;
}

}  // namespace

bool gemm_f32_rope_ok(const GemmF32Args& p, int head_dim) {
  return head_dim == 16 && p.N % 16 == 0 && p.K % 32 == 0 && f32_vec_c(p) && f32_tile_ok(p);
}

void gemm_f32_tile(int M, int N, int K, int* rows, int* cols) {
  GemmF32Args p;
  p.lda = p.ldw = p.K = K;
  p.M = M;
  p.N = N;
  *rows = *cols = 0;
  if (M <= 0 || N <= 0 || !f32_tile_ok(p)) return;
  const int t = f32_takes_pair(p) ? -1 : f32_tile(p);
  *rows = t < 0 ? 16 : kTileRows[t];
  *cols = t < 0 ? 16 : kTileCols[t];
}

hipError_t launch_gemm_f32(const GemmF32Args& p, int epi, hipStream_t s) {
  if (p.M <= 0 || p.N <= 0) return hipSuccess;
  if (epi == kF32QkvRope && !gemm_f32_rope_ok(p, 16)) return hipErrorInvalidValue;
  if (f32_tile_ok(p)) {
    if (f32_takes_pair(p)) return launch_f32_pair(p, epi, s);
    return f32_pieces(p, [&](const GemmF32Args& q) {
      switch (f32_tile(q)) {
        case 0: return launch_f32_tile<false, 1, 1>(q, epi, s);
        case 1: return launch_f32_tile<false, 2, 2>(q, epi, s);
        default: return launch_f32_tile<false, 4, 2>(q, epi, s);
      }
    });
  }
  const int tiles = ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
  const dim3 grid(tiles), block(kThreads);
  const bool vec = (p.K % 4 == 0) && (p.lda % 4 == 0) && (p.ldw % 4 == 0);
#define ESM_F32_LAUNCH(E)                                                          \
  if (vec) hipLaunchKernelGGL((gemm_f32_kernel<E, true>), grid, block, 0, s, p);   \
  else hipLaunchKernelGGL((gemm_f32_kernel<E, false>), grid, block, 0, s, p);
  switch (epi) {
    case kF32Store: ESM_F32_LAUNCH(kF32Store) break;
    case kF32Gelu: ESM_F32_LAUNCH(kF32Gelu) break;
    case kF32Resid: ESM_F32_LAUNCH(kF32Resid) break;
    default: return hipErrorInvalidValue;
  }
#undef ESM_F32_LAUNCH
  return hipGetLastError();
}

}  // namespace esm_gfx950
