// FP32 GEMM C = A W^T + bias on gfx950 fp32 MFMA (v_mfma_f32_16x16x4f32),
// with optional GELU or residual-add epilogue.
//
// Replaces esm::kernels::Linear (reference src/kernels/gemm_fp32.cpp:33-46
// LinearRef, :272-294 LinearAvx512) for the all-fp32 8M model and for the
// fp32 lm head (dense d->d, tied decoder d->vocab; src/model.cpp:1192-1239).
// Products are exact fp32 products accumulated in fp32, so results differ
// from the sequential reference sum only by summation order.
//
// Three kernels (launch_gemm_f32 picks):
//   - gemm_f32_tile_kernel: aligned rows with K % 32 == 0; LDS tiles of 32x32
//     to 128x64, direct global -> LDS stage loads;
//   - gemm_f32_skinny_kernel: grids too small for that one (and the decoder's
//     N <= 48): eight waves split K, operands straight into registers;
//   - gemm_f32_kernel: any other shape (128x128 tiles through registers).
//
// gemm_f32_kernel's tiling: 128x128 workgroup tile, four waves of 64x64,
// 32-wide K stages in LDS (row pitch 36 floats). Within a stage, lane group g
// (lane / 16) owns the eight consecutive k values [8g, 8g+8): MFMA step j
// multiplies A and W at k = 8g + j for every lane group, which keeps A and W
// consistent and lets each lane fetch its k values with two 16-byte LDS reads.
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

// ---- Split-fp16 GEMM (fp32 accuracy on fp16 MFMA), same 128x128 tile and
// wave layout as above on v_mfma_f32_16x16x32_f16: each lane holds eight
// consecutive k of one row for A and W, so one MFMA covers a 32-wide K stage.
// A (fp32) is split into hi / lo fp16 planes while it is staged in LDS; W's
// planes come split. LDS rows are 64 bytes (four 16-byte chunks), chunk c of
// row r stored at position c ^ ((r / 4) mod 4): the 16-byte fragment reads
// of 16 rows at one chunk then cover all 64 banks once, and so do the stage
// writes of four consecutive rows (an 80-byte padded pitch kept the reads
// conflict-free but made every write pass conflict).
constexpr int kX3Pitch = 64;                    // bytes per 32-half row
constexpr int kX3Plane = 128 * kX3Pitch;        // one 128-row plane
constexpr int kX3Stage = 4 * kX3Plane;          // A hi, A lo, W hi, W lo

// Byte offset of 16-byte chunk c of row r in a plane.
__device__ __forceinline__ int x3_off(int r, int c) { return r * kX3Pitch + ((c ^ ((r >> 2) & 3)) << 4); }

__device__ __forceinline__ uint2 pack_f16x4(float a, float b, float c, float d) {
  return make_uint2(static_cast<uint32_t>(f32_to_f16_bits(a)) | (static_cast<uint32_t>(f32_to_f16_bits(b)) << 16),
                    static_cast<uint32_t>(f32_to_f16_bits(c)) | (static_cast<uint32_t>(f32_to_f16_bits(d)) << 16));
}

// One K stage of the tile from global memory: A 128 rows x 32 floats (four
// float4 per thread), W planes 128 rows x 32 halves each (two 16-byte pieces
// per plane per thread). Rows past the edge re-read the last valid row;
// their results are never stored.
__device__ __forceinline__ void x3_load(const GemmX3Args& p, int m0, int n0, int k0, f32x4 (&ra)[4],
                                        i32x4 (&rh)[2], i32x4 (&rl)[2]) {
  const int t = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int idx = t + kThreads * i;
    const int row = min(m0 + (idx >> 3), p.M - 1);
    ra[i] = *reinterpret_cast<const f32x4*>(p.A + static_cast<size_t>(row) * p.lda + k0 + (idx & 7) * 4);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int idx = t + kThreads * i;
    const int row = min(n0 + (idx >> 2), p.N - 1);
    const size_t off = static_cast<size_t>(row) * p.ldw + k0 + (idx & 3) * 8;
    rh[i] = *reinterpret_cast<const i32x4*>(p.w_hi + off);
    rl[i] = *reinterpret_cast<const i32x4*>(p.w_lo + off);
  }
}

// The stage into LDS: A split into hi / lo planes, W planes as loaded.
__device__ __forceinline__ void x3_store(uint8_t* st, const f32x4 (&ra)[4], const i32x4 (&rh)[2],
                                         const i32x4 (&rl)[2]) {
  const int t = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int idx = t + kThreads * i;
    const int off = x3_off(idx >> 3, (idx & 7) >> 1) + (idx & 1) * 8;
    const f32x4 x = ra[i];
    const float hx = f16_bits_to_f32(f32_to_f16_bits(x[0])), hy = f16_bits_to_f32(f32_to_f16_bits(x[1]));
    const float hz = f16_bits_to_f32(f32_to_f16_bits(x[2])), hw = f16_bits_to_f32(f32_to_f16_bits(x[3]));
    *reinterpret_cast<uint2*>(st + off) = pack_f16x4(hx, hy, hz, hw);
    *reinterpret_cast<uint2*>(st + kX3Plane + off) = pack_f16x4(x[0] - hx, x[1] - hy, x[2] - hz, x[3] - hw);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int idx = t + kThreads * i;
    const int off = x3_off(idx >> 2, idx & 3);
    *reinterpret_cast<i32x4*>(st + 2 * kX3Plane + off) = rh[i];
    *reinterpret_cast<i32x4*>(st + 3 * kX3Plane + off) = rl[i];
  }
}

template <int EPI>
__global__ __launch_bounds__(kThreads, 2) void gemm_x3_kernel(const GemmX3Args p) {
  __shared__ __attribute__((aligned(16))) uint8_t smem[2 * kX3Stage];
  const int tiles_n = (p.N + BN - 1) / BN;
  const int m0 = (blockIdx.x / tiles_n) * BM;
  const int n0 = (blockIdx.x % tiles_n) * BN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int lr = lane & 15, lg = lane >> 4;

  f32x4 ra[4];
  i32x4 rh[2], rl[2];
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int nk = p.K / 32;
  x3_load(p, m0, n0, 0, ra, rh, rl);
  x3_store(smem, ra, rh, rl);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const uint8_t* cur = smem + (kt & 1) * kX3Stage;
    const bool more = kt + 1 < nk;
    if (more) x3_load(p, m0, n0, (kt + 1) * 32, ra, rh, rl);
    f16x8 ah[4], al[4], bh[4], bl[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ao = x3_off(wm * 64 + i * 16 + lr, lg);
      const int bo = x3_off(wn * 64 + i * 16 + lr, lg);
      ah[i] = *reinterpret_cast<const f16x8*>(cur + ao);
      al[i] = *reinterpret_cast<const f16x8*>(cur + kX3Plane + ao);
      bh[i] = *reinterpret_cast<const f16x8*>(cur + 2 * kX3Plane + bo);
      bl[i] = *reinterpret_cast<const f16x8*>(cur + 3 * kX3Plane + bo);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        f32x4 c = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], bh[n], acc[i][n], 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[i], bh[n], c, 0, 0, 0);
        acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], bl[n], c, 0, 0, 0);
      }
    if (more) x3_store(smem + ((kt + 1) & 1) * kX3Stage, ra, rh, rl);
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
        float v = __builtin_fmaf(acc[i][n][r], p.w_unscale, b);
        if constexpr (EPI == kF32Gelu) v = gelu_erf(v);
        float* dst = p.C + static_cast<size_t>(row) * p.ldc + col;
        if constexpr (EPI == kF32Resid) {
          *dst += v;
        } else {
          *dst = v;
        }
      }
  }
}

// ---- Tiled fp32 GEMM (K % 32 == 0, 16-byte aligned rows): 2 x 2 waves of
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
// evenly the tiles fall on the CUs (f32_tile_of). 1280 x 1280 at 7,777 rows:
// 303 us with 128x128 tiles staged through registers, 199 here (128 TFLOP/s;
// 165 us at the rate of a large fp32 library product); at 66 rows and K = N =
// 320, 33 -> 4.8 us.
template <int MB, int NB>
struct F32Tile {
  static constexpr int BM = 32 * MB, BN = 32 * NB;
  static constexpr int kBlocks = (BM + BN) / 8;  // 1 KB blocks per stage
  static constexpr int kPer = kBlocks / 4;       // per wave
  static constexpr int kStage = kBlocks * 1024;
  // More buffers only cost resident workgroups (1280 x 1280 at 1,000 rows,
  // 32x32 tiles: 33 us with three, 39 with five).
  static constexpr int kNStage = kStage <= 16384 ? 3 : 2;
  // A single 16x16 block per wave would be one chain of dependent MFMAs, 52
  // cycles each instead of the 32 they occupy the matrix core: its halves of a
  // stage go to two accumulators.
  static constexpr int kChains = MB * NB == 1 ? 2 : 1;
};

// One 16-byte-per-lane global -> LDS load, as in the INT8 kernel: uniform
// base, 32-bit lane offset, LDS byte address in M0; awaited by the explicit
// vmcnt before the barrier that publishes the stage.
__device__ __forceinline__ void f32_dma16(const void* base, uint32_t off, uint32_t lds) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t m0v = __builtin_amdgcn_readfirstlane(lds);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(m0v)
               : "memory", "m0");
#endif
}

// Output of four consecutive columns of one row, the epilogue applied.
template <int EPI>
__device__ __forceinline__ void f32_store4(const GemmF32Args& p, int row, int col, f32x4 v, bool vec_c) {
  if (row >= p.M || col >= p.N) return;
  float* dst = p.C + static_cast<size_t>(row) * p.ldc + col;
  const int n = min(4, p.N - col);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] += p.bias && e < n ? p.bias[col + e] : 0.0f;
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

template <int MB, int NB, int EPI>
__global__ __launch_bounds__(256) void gemm_f32_tile_kernel(const GemmF32Args p, bool vec_c) {
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
  const uint32_t lds0 = static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)smem));
  auto load_stage = [&](int kt, int buf) {
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      f32_dma16((wave * kPer + i < BM / 8 ? p.A : p.W) + kt * 32, goff[i],
                lds0 + static_cast<uint32_t>(buf * kStage + (wave * kPer + i) * 1024));
  };
  const int nk = p.K / 32;
#pragma unroll
  for (int st = 0; st < kNStage - 1; ++st)
    if (st < nk) load_stage(st, st);

  constexpr int kChains = TL::kChains;
  f32x4 acc[kChains][MB][NB];
#pragma unroll
  for (int x = 0; x < kChains; ++x)
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[x][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Row R's chunk c of a stage: block R / 8, slot c ^ (R % 8).
  const int arow = wm * 16 * MB + lr, wrow = BM + wn * 16 * NB + lr;
  auto frag = [&](const uint8_t* st, int R, int h) {
    return *reinterpret_cast<const f32x4*>(st + (R >> 3) * 1024 + (R & 7) * 128 + (((4 * h + lg) ^ (R & 7)) << 4));
  };
  int buf = 0;
  for (int kt = 0; kt < nk; ++kt) {
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
    // The chains of a single-block wave advance together; otherwise one half
    // of the stage at a time keeps fewer fragments live.
#pragma unroll
    for (int h0 = 0; h0 < 2; h0 += kChains) {
      f32x4 fa[kChains][MB], fw[kChains][NB];
#pragma unroll
      for (int x = 0; x < kChains; ++x) {
#pragma unroll
        for (int i = 0; i < MB; ++i) fa[x][i] = frag(st, arow + 16 * i, h0 + x);
#pragma unroll
        for (int j = 0; j < NB; ++j) fw[x][j] = frag(st, wrow + 16 * j, h0 + x);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int x = 0; x < kChains; ++x)
#pragma unroll
          for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
              acc[x][i][j] =
                  __builtin_amdgcn_mfma_f32_16x16x4f32(fw[x][j][e], fa[x][i][e], acc[x][i][j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      f32x4 v = acc[0][i][j];
      if constexpr (kChains == 2) v += acc[1][i][j];
      f32_store4<EPI>(p, m0 + wm * 16 * MB + 16 * i + lr, n0 + wn * 16 * NB + 16 * j + 4 * lg, v, vec_c);
    }
}

// ---- Skinny fp32 GEMM (K % 16 == 0): a 16 MB x 16 NB output tile whose K is
// split over the workgroup's eight waves. Each wave loads its 16-wide K steps
// straight into registers (lane (lr, lg): k = 16 s + 4 lg .. + 4 of row lr), CH
// steps in flight at once, and the waves' sums meet in LDS in wave order. It
// is for grids of few tiles, where one wave's walk over all of K, a load
// latency per step, is what the launch takes.
constexpr int kSkinnyWaves = 8;
template <int MB, int NB, int CH, int EPI>
__global__ __launch_bounds__(kSkinnyWaves * 64) void gemm_f32_skinny_kernel(const GemmF32Args p, bool vec_c) {
  __shared__ f32x4 part[kSkinnyWaves][MB * NB][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int m0 = blockIdx.x * 16 * MB, n0 = blockIdx.y * 16 * NB;
  const float* arow[MB];
  const float* wrow[NB];
#pragma unroll
  for (int i = 0; i < MB; ++i) arow[i] = p.A + static_cast<size_t>(min(m0 + 16 * i + lr, p.M - 1)) * p.lda + 4 * lg;
#pragma unroll
  for (int j = 0; j < NB; ++j) wrow[j] = p.W + static_cast<size_t>(min(n0 + 16 * j + lr, p.N - 1)) * p.ldw + 4 * lg;
  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = p.K / 16;
  const int s0 = steps * wave / kSkinnyWaves, s1 = steps * (wave + 1) / kSkinnyWaves;
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
  for (int w = 1; w < kSkinnyWaves; ++w) v += part[w][wave][lane];
  f32_store4<EPI>(p, m0 + 16 * (wave / NB) + lr, n0 + 16 * (wave % NB) + 4 * lg, v, vec_c);
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

template <int MB, int NB>
hipError_t launch_f32_tile(const GemmF32Args& p, int epi, hipStream_t s) {
  using TL = F32Tile<MB, NB>;
  const bool vec_c = f32_vec_c(p);
  const dim3 grid(((p.M + TL::BM - 1) / TL::BM) * ((p.N + TL::BN - 1) / TL::BN)), block(256);
  ESM_F32_EPI(gemm_f32_tile_kernel, MB, NB);
}

template <int MB, int NB, int CH>
hipError_t launch_f32_skinny(const GemmF32Args& p, int epi, hipStream_t s) {
  const bool vec_c = f32_vec_c(p);
  const dim3 grid((p.M + 16 * MB - 1) / (16 * MB), (p.N + 16 * NB - 1) / (16 * NB)), block(kSkinnyWaves * 64);
  ESM_F32_EPI(gemm_f32_skinny_kernel, MB, NB, CH);
}

bool f32_skinny_ok(const GemmF32Args& p) {
  return p.K > 0 && p.K % 16 == 0 && p.lda % 4 == 0 && p.ldw % 4 == 0;
}

// The stage loads take 16-byte aligned rows and 32-bit lane offsets.
bool f32_tile_ok(const GemmF32Args& p) {
  constexpr uint64_t kLimit = 1ull << 32;
  return p.K > 0 && p.K % 32 == 0 && p.lda % 4 == 0 && p.ldw % 4 == 0 &&
         (reinterpret_cast<uintptr_t>(p.A) | reinterpret_cast<uintptr_t>(p.W)) % 16 == 0 &&
         static_cast<uint64_t>(p.M) * p.lda * 4 <= kLimit && static_cast<uint64_t>(p.N) * p.ldw * 4 <= kLimit;
}

// Index into {32x32, 64x64, 128x64}: the tile whose grid takes the least
// time, (the most tiles any CU gets + 1/2) x the tile's outputs x its cost per
// output. The costs are those of many rounds (2560 x 2560 at 16,000 rows:
// 1,727 / 1,529 / 1,498 us); the half tile is the last round, in which a CU's
// few remaining workgroups leave its matrix cores waiting. It follows the
// measured order at 1280 x 1280: 33 / 44 / 48 us at 1,000 rows, 56 / 62 / 79 at
// 1,768, 94 / 84 / 81 at 3,000, 224 / 199 / 230 at 7,777, 457 / 393 / 389 at
// 16,000. (64x32 and 128x128 tiles were never more than 8% faster.)
int f32_tile_of(int M, int N) {
  static constexpr int kBM[3] = {32, 64, 128}, kBN[3] = {32, 64, 64};
  static constexpr double kCost[3] = {1.17, 1.02, 1.0};
  const int cus = device_cus();
  int best = 0;
  double best_t = 0.0;
  for (int t = 0; t < 3; ++t) {
    const long tiles = static_cast<long>((M + kBM[t] - 1) / kBM[t]) * ((N + kBN[t] - 1) / kBN[t]);
    const double c = (static_cast<double>((tiles + cus - 1) / cus) + 0.5) * kBM[t] * kBN[t] * kCost[t];
    if (t == 0 || c < best_t) {
      best = t;
      best_t = c;
    }
  }
  return best;
}

}  // namespace

hipError_t launch_gemm_narrow(const GemmF32Args& p, hipStream_t s) {
  if (p.M <= 0 || p.N <= 0) return hipSuccess;
  if (p.N > 48 || !f32_skinny_ok(p)) return hipErrorInvalidValue;
  // 32 rows a workgroup halve the reads of W once there are enough of them.
  if (p.M > 4096) return launch_f32_skinny<2, 3, 4>(p, kF32Store, s);
  return launch_f32_skinny<1, 3, 5>(p, kF32Store, s);
}

hipError_t launch_gemm_x3(const GemmX3Args& p, int epi, hipStream_t s) {
  if (p.M <= 0 || p.N <= 0) return hipSuccess;
  if (p.K <= 0 || p.K % 32 != 0 || p.lda % 4 != 0 || p.ldw % 8 != 0) return hipErrorInvalidValue;
  const int tiles = ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
  const dim3 grid(tiles), block(kThreads);
  switch (epi) {
    case kF32Store: hipLaunchKernelGGL((gemm_x3_kernel<kF32Store>), grid, block, 0, s, p); break;
    case kF32Gelu: hipLaunchKernelGGL((gemm_x3_kernel<kF32Gelu>), grid, block, 0, s, p); break;
    case kF32Resid: hipLaunchKernelGGL((gemm_x3_kernel<kF32Resid>), grid, block, 0, s, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_gemm_f32(const GemmF32Args& p, int epi, hipStream_t s) {
  if (p.M <= 0 || p.N <= 0) return hipSuccess;
  // At most one 16x16-tile workgroup a CU and a K long enough to be worth
  // splitting: N = 320 at 66 rows takes 6.4 / 6.5 / 6.6 / 6.7 us skinny for K
  // = 320 / 480 / 960 / 1280 against 4.8 / 6.0 / 9.7 / 12.2 in 32x32 tiles; a
  // second round of workgroups (301 rows) 11.4 against 12.4 at K = 1280.
  const long tiles16 = static_cast<long>((p.M + 15) / 16) * ((p.N + 15) / 16);
  if (f32_skinny_ok(p) && p.K >= 512 && tiles16 <= device_cus()) return launch_f32_skinny<1, 1, 10>(p, epi, s);
  if (f32_tile_ok(p)) {
    switch (f32_tile_of(p.M, p.N)) {
      case 0: return launch_f32_tile<1, 1>(p, epi, s);
      case 1: return launch_f32_tile<2, 2>(p, epi, s);
      default: return launch_f32_tile<4, 2>(p, epi, s);
    }
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
