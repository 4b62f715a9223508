// FP8 block-scaled linear for few tokens (at most 32): one launch that streams
// each weight byte once, in whole 1 KiB pieces of its rows.
//
// Replaces the same two Triton kernels as fp8_linear.hip for decode-sized
// calls (nanovllm/kernels/fp8_linear.py:11-71, launched at :116-138).
//
// The weights are nearly all of the bytes, so their stream is what the kernel
// is built around.  Loads in the MFMA operand's layout (16 rows x 64 bytes an
// instruction) reach 3.2 TB/s on 6,144 x 4,096 weights and 4.3 on 24,576 x
// 4,096, loads of 1 KiB of one row 4.6 and 6.4 (loads alone, all CUs), so a
// wave brings 16 rows x 1 KiB (a chunk: eight K blocks) to LDS by sixteen
// direct-to-LDS loads and reads the operands back from there.
//
// A workgroup owns 16 features over all of K; its waves take the chunks in
// turn (wave w: chunks w, w + nw, ..), each into its own 16 KiB of LDS, so no
// wave waits for another until the partial sums meet in LDS at the end: a
// barrier per K block is what a tile grid of this shape spends its time on.
// The waves of one or two workgroups keep 64 to 128 KiB per CU in flight.
//  - activations, XI == 0: the quantised rows, loaded to registers in the
//    operand layout ahead of the chunk (L2 hits: every workgroup reads them);
//  - activations, XI > 0: the wave quantises the chunk's groups of the raw
//    activations itself (XI passes of four 16-lane groups, loaded ahead of the
//    weights and done while those are in flight) into its own LDS slice.  The
//    activation launch, its round trip through memory and its place in the
//    queue go away; worth it while every workgroup repeats little work.
// One MFMA per 16 x 16 fragment per K block and acc += P * (sx * sw), as in
// the tile kernels; the waves' partial sums are added in wave order.
#include <algorithm>
#include <atomic>

#include "fp8_common.h"
#include "fp8_quant.h"
#include "kernels.h"
#include "lds_dma.h"

namespace nvamd {

namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));

constexpr int kThinChunk = 1024;                 // bytes of a row in a chunk
constexpr int kThinSlot = 16 * kThinChunk;       // LDS of a chunk: 16 rows
constexpr int kThinKb = kThinChunk / kFp8Block;  // K blocks of a chunk
constexpr int kThinMaxWaves = 8;

constexpr uint32_t kOutOfRange = 0xFFFFFFF0u;  // a buffer offset that reads zeros

// A wave's slice of quantised activations (XI > 0): rows of one chunk, padded
// by a granule, then the chunk's scales (fp32).
constexpr int kThinXPitch = kThinChunk + 16;
__host__ __device__ constexpr int thin_x_bytes(int M) { return M * (kThinXPitch + 4 * kThinKb); }

// LDS of a launch: the waves' chunks, then their activation slices; the
// partial fragments [wave][MF][64 lanes] f32x4 (at most 4 KiB a wave) reuse
// the chunks.
__host__ __device__ constexpr int thin_lds_bytes(int nw, int M, int xi) {
  return nw * (kThinSlot + (xi > 0 ? thin_x_bytes(M) : 0));
}

template <int MF, int XI, bool F16_IN>
__global__ __launch_bounds__(64 * kThinMaxWaves) void thin_linear_kernel(Fp8GemmParams p, const uint16_t* __restrict__ x,
                                                                       int64_t x_stride, int f16_out) {
  static_assert(XI == 0 || MF == 1, "a call that quantises its activations has one token fragment");
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_uniform(tid >> 6);
  const int nw = (int)blockDim.x >> 6;
  const int q = lane >> 4, r16 = lane & 15;
  const int n0 = (int)blockIdx.x * 16;
  const int Kc = p.Kc, M = (int)p.M;
  const int chunks = (p.K + kThinChunk - 1) / kThinChunk;

  const u32x4 rw = rsrc_words(p.w + (int64_t)n0 * p.w_stride, (uint32_t)(16 * p.w_stride));
  const uint16_t* sw_row = p.w_scale + (int64_t)(n0 / kFp8Block) * Kc;  // the workgroup's 128-row block
  const uint32_t slot = wave_uniform((int)lds_addr(smem)) + (uint32_t)(wave * kThinSlot);
  const uint8_t* slot_p = smem + wave * kThinSlot;
  // Granule g (of 64) of chunk row r sits at position g ^ 2r: an operand read
  // takes granules q and q + 4 of a K block of 16 rows, so the 32 lanes served
  // together (two values of q) hit 32 different granules of a 512-byte window.
  const uint32_t rd0 = (uint32_t)(r16 * kThinChunk + 16 * (q ^ (2 * r16)));

  const __amdgpu_buffer_rsrc_t rxq =
      make_rsrc(p.xq, (uint32_t)(M - 1) * p.x_row + (uint32_t)(Kc - 1) * p.x_blk + (uint32_t)kFp8Block);
  const __amdgpu_buffer_rsrc_t rsx =
      make_rsrc(p.x_scale, ((uint32_t)(M - 1) * p.sx_row + (uint32_t)(Kc - 1) * p.sx_blk + 1u) * 2u);
  uint8_t* xs = smem + nw * kThinSlot + wave * thin_x_bytes(M);
  float* ss = reinterpret_cast<float*>(xs + M * kThinXPitch);

  u32x4 xr[XI > 0 ? XI : 1], xb[XI > 0 ? 1 : kThinKb][MF][2];
  uint32_t sx2[MF];  // lane (q, token): scales of the chunk's K blocks 2q (low half) and 2q + 1
  auto load_x = [&](int d, int kc) {  // quantised rows of K block kc, in the operand layout
#pragma unroll
    for (int j = 0; j < MF; ++j) {
      const uint32_t row = (uint32_t)(16 * j + r16);
      const bool in = kc < Kc && row < (uint32_t)M;  // rows past M: no traffic
      const uint32_t off = row * p.x_row + (uint32_t)kc * p.x_blk + 16u * (uint32_t)q;
      xb[d][j][0] = buf_load16(rxq, in ? off : kOutOfRange);
      xb[d][j][1] = buf_load16(rxq, in ? off + 64u : kOutOfRange);
    }
  };
  auto load_sx = [&](int kc0) {  // (blocks past K: P is 0, and the row's last scale stands in)
    const uint32_t k0 = (uint32_t)min(kc0 + 2 * q, Kc - 1) * p.sx_blk, k1 = (uint32_t)min(kc0 + 2 * q + 1, Kc - 1) * p.sx_blk;
#pragma unroll
    for (int j = 0; j < MF; ++j) {
      const uint32_t row = (uint32_t)(16 * j + r16) * p.sx_row;
      sx2[j] = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rsx, (int)((row + k0) * 2u), 0, 0) |
               ((uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rsx, (int)((row + k1) * 2u), 0, 0) << 16);
    }
  };

  f32x4 acc[MF];
#pragma unroll
  for (int j = 0; j < MF; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int c = wave; c < chunks; c += nw) {
    const int kc0 = c * kThinKb;
    // activations first (loads complete in order), then the weights
    const uint32_t sw_bits = sw_row[min(kc0 + (lane & (kThinKb - 1)), Kc - 1)];  // lane kb: scale of block kc0 + kb
    if constexpr (XI > 0) {
#pragma unroll
      for (int i = 0; i < XI; ++i) {  // group 4 i + q: token (4 i + q) / 8, K block kc0 + (4 i + q) % 8
        // (past K: a block of the same token again, against weights of zero)
        const int m = min((4 * i + q) / kThinKb, M - 1), kc = min(kc0 + (4 * i + q) % kThinKb, Kc - 1);
        xr[i] = *reinterpret_cast<const u32x4*>(x + m * x_stride + kc * kFp8Block + 8 * r16);
      }
    } else {
      load_sx(kc0);
#pragma unroll
      for (int d = 0; d < kThinKb; ++d) load_x(d, kc0 + d);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const uint32_t k = (uint32_t)(c * kThinChunk + 16 * (lane ^ (2 * r)));
      dma_load16(rw, k < (uint32_t)p.K ? (uint32_t)r * (uint32_t)p.w_stride + k : kOutOfRange, slot + 1024u * r);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (XI > 0) {
#pragma unroll
      for (int i = 0; i < XI; ++i) {
        const int m = (4 * i + q) / kThinKb, kb = (4 * i + q) % kThinKb;
        float scale;
        const u32x2 b = quant_group8<F16_IN>(xr[i], scale);
        if (m < M) {
          *reinterpret_cast<u32x2*>(xs + m * kThinXPitch + kb * kFp8Block + 8 * r16) = b;
          if (r16 == 0) ss[m * kThinKb + kb] = bf16_bits_to_f32(scale_bf16_bits(scale));
        }
      }
    }
    wait_vmcnt<0>();
    // this wave's chunk and slice are in LDS; no other wave touches them
    asm volatile("" ::: "memory");
    // blocks past K count as zero, not with the last block's scale (it may be
    // infinite, and 0 * inf is NaN)
    const float sw_lane = kc0 + (lane & (kThinKb - 1)) < Kc ? bf16_bits_to_f32(sw_bits) : 0.f;
#pragma unroll
    for (int kb = 0; kb < kThinKb; ++kb) {
      const float sw = readlane_f32(sw_lane, kb);
      const uint32_t rd = rd0 ^ (uint32_t)(kFp8Block * kb);
      const u32x4 lo = *reinterpret_cast<const u32x4*>(slot_p + rd), hi = *reinterpret_cast<const u32x4*>(slot_p + (rd ^ 64u));
      const i32x8 a = {(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
#pragma unroll
      for (int j = 0; j < MF; ++j) {
        u32x4 blo, bhi;
        float s;
        if constexpr (XI > 0) {
          const int m = min(r16, M - 1);  // columns past M hold a copy and are not stored
          const uint8_t* row = xs + m * kThinXPitch + kb * kFp8Block + 16 * q;
          blo = *reinterpret_cast<const u32x4*>(row);
          bhi = *reinterpret_cast<const u32x4*>(row + 64);
          s = ss[m * kThinKb + kb] * sw;  // exact (two bf16 values)
        } else {
          blo = xb[kb][j][0];
          bhi = xb[kb][j][1];
          const uint32_t sx = (uint32_t)__shfl((int)sx2[j], 16 * (kb / 2) + r16);
          s = bf16_bits_to_f32(kb & 1 ? sx >> 16 : sx & 0xFFFFu) * sw;  // exact
        }
        const i32x8 b = {(int)blo.x, (int)blo.y, (int)blo.z, (int)blo.w, (int)bhi.x, (int)bhi.y, (int)bhi.z, (int)bhi.w};
        const f32x4 pr = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 127, 0,
                                                                          127);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[j][e] = __builtin_fmaf(pr[e], s, acc[j][e]);
      }
    }
    // the chunk and the slice are read before the next ones overwrite them
    __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0)
    asm volatile("" ::: "memory");
  }

  // partial sums of the waves, added in wave order
  __syncthreads();
  f32x4* red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int j = 0; j < MF; ++j) red[(wave * MF + j) * 64 + lane] = acc[j];
  __syncthreads();
  for (int u = tid; u < MF * 64; u += 64 * nw) {
    f32x4 v = red[u];
    for (int k = 1; k < nw; ++k) {
      const f32x4 t = red[k * (MF * 64) + u];
      v = f32x4{v[0] + t[0], v[1] + t[1], v[2] + t[2], v[3] + t[3]};
    }
    // lane l of fragment j: token 16 j + l % 16, features n0 + 4 (l / 16) .. + 3
    const int j = u >> 6, l = u & 63, m = 16 * j + (l & 15);
    if (m >= M) continue;
    const u32x2 o = f16_out ? u32x2{pack_f16x2(v[0], v[1]), pack_f16x2(v[2], v[3])}
                            : u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    *reinterpret_cast<u32x2*>(p.out + (int64_t)m * p.out_stride + n0 + 4 * (l >> 4)) = o;
  }
}

template <int MF, int XI, bool F16_IN>
hipError_t launch_thin(const Fp8GemmParams& p, const ThinPlan& pl, const void* x, int64_t x_stride, bool f16_out,
                       hipStream_t stream) {
  auto kern = thin_linear_kernel<MF, XI, F16_IN>;
  const int lds = pl.lds;
  static std::atomic<int> lds_set{0};  // largest dynamic LDS size granted so far
  if (lds > lds_set.load(std::memory_order_relaxed)) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    lds_set.store(lds, std::memory_order_relaxed);
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.N / 16)), dim3((unsigned)(64 * pl.nw)), (size_t)lds, stream, p,
                     (const uint16_t*)x, x_stride, f16_out ? 1 : 0);
  return hipGetLastError();
}

}  // namespace

// Where the kernel is taken, from both sides measured (us per call, GPU time,
// weights from HBM, quantisation included; this kernel / the fastest of
// fp8_linear.hip; more in profiles/fp8_linear_kernels.md).  Every workgroup
// reads all the activations, so it loses its lead with M K (their bytes per
// workgroup) and with M N (their reads in all):
//   6,144 x 4,096:   M 1 7.5 / 16.5, 8 10.5 / 17.2, 16 12.1 / 17.3, 32 15.9 / 18.4
//   24,576 x 4,096:  M 1 21.1 / 30.6, 16 28.8 / 31.3, 24 35.4 / 33, 32 39.6 / 33
//   4,096 x 12,288:  M 1 12.2 / 20.7, 16 17.2 / 21.4, 24 21.5 / 21.9, 32 23.6 / 22.1
//   5,120 x 25,600:  M 1 30.3 / 41.8, 8 38.6 / 42.3, 12 42.0 / 42.5, 16 46.1 / 42.6
//   51,200 x 5,120:  M 1 45.9 / 55.5, 8 51.8 / 56.8, 12 55.7 / 57.5, 16 60.6 / 57.9
// With two workgroups on a CU a second token fragment doubles what the four
// waves do per chunk:
//   5,120 x 8,192:   M 16 18.5 / 20.1, 24 23.2 / 21.2
//   6,144 x 1,024:   M 16 6.3 / 6.8, 24 7.3 / 7.0 (one wave per workgroup)
// Few workgroups leave CUs idle, which a K split would use: worth it only for
// what one round of chunks holds.
//   512 x 8,192:     M 1 6.2 / 10.2, 16 10.9 / 11.1, 32 14.7 / 11.2
//   512 x 12,288:    M 1 8.2 / 11.6, 3 11.9 / 11.8, 16 13.8 / 12.1 (two rounds)
//   256 x 32,768:    M 1 14.3 / 15.2, 3 22.2 / 15.6 (four rounds)
// Its own quantisation repeats per workgroup and pays for one or two tokens
// (6,144 x 4,096, M = 2: 8.2 against 9.9 with a launch before; M = 4: 12.6
// against 9.9), up to four when every workgroup has a CU (4,096 x 4,096, M = 4:
// 7.6, five tokens with a launch before 7.9).
ThinPlan fp8_thin_plan(int64_t M, int64_t N, int Kc, int cus, int64_t lds_limit, bool raw_x) {
  ThinPlan pl;
  if (M < 1 || M > kThinMaxM || N % 128 != 0 || Kc < 1 || M * Kc > (1 << 11) || M * N > 600000) return pl;
  // Waves: the chunks in equal rounds, of at most four waves (two workgroups a
  // CU) or, when a CU has one workgroup at most, eight (12,288 columns: six
  // waves twice 11.4 us, four waves three times 13.4; 25,600 columns, 320
  // workgroups: four waves 27.3, five 33.2 with one workgroup a CU).
  const int chunks = (Kc + kThinKb - 1) / kThinKb;
  const bool one_wg = N / 16 <= cus;
  const int most = one_wg ? kThinMaxWaves : 4;
  const int rounds = (chunks + most - 1) / most;
  const int nw = (chunks + rounds - 1) / rounds;
  if (N / 16 <= cus / 2 && M * Kc * rounds * rounds > (1 << 10)) return pl;
  if (!one_wg && M > 16 && (chunks == 1 || M * Kc > 1280)) return pl;
  // The waves do not depend on who quantises, so neither do the sums: where
  // the slices do not fit beside the chunks (four tokens and eight waves), the
  // activations are quantised before.
  int xi = !raw_x || M > (one_wg ? 4 : 2) ? 0 : M <= 1 ? 2 : M <= 2 ? 4 : 8;
  if (thin_lds_bytes(nw, (int)M, xi) > lds_limit) xi = 0;
  if (thin_lds_bytes(nw, (int)M, xi) > lds_limit) return pl;
  pl.nw = nw;
  pl.mf = M <= 16 ? 1 : 2;
  pl.xi = xi;
  pl.lds = thin_lds_bytes(nw, (int)M, xi);
  return pl;
}

hipError_t launch_fp8_thin_linear(const Fp8GemmParams& p, const ThinPlan& pl, const void* x, int64_t x_stride,
                                  bool f16_in, bool f16_out, hipStream_t stream) {
  if (pl.mf == 0 || p.M < 1 || p.M > 16 * pl.mf || pl.nw < 1 || pl.nw > kThinMaxWaves || p.N % 16 != 0 ||
      (pl.xi > 0 && p.M * kThinKb > 4 * pl.xi) || pl.lds < thin_lds_bytes(pl.nw, (int)p.M, pl.xi))
    return hipErrorInvalidValue;
  switch (pl.xi > 0 ? 16 * pl.xi + (f16_in ? 1 : 0) : pl.mf) {
    case 1: return launch_thin<1, 0, false>(p, pl, nullptr, 0, f16_out, stream);
    case 2: return launch_thin<2, 0, false>(p, pl, nullptr, 0, f16_out, stream);
    case 32: return launch_thin<1, 2, false>(p, pl, x, x_stride, f16_out, stream);
    case 33: return launch_thin<1, 2, true>(p, pl, x, x_stride, f16_out, stream);
    case 64: return launch_thin<1, 4, false>(p, pl, x, x_stride, f16_out, stream);
    case 65: return launch_thin<1, 4, true>(p, pl, x, x_stride, f16_out, stream);
    case 128: return launch_thin<1, 8, false>(p, pl, x, x_stride, f16_out, stream);
    case 129: return launch_thin<1, 8, true>(p, pl, x, x_stride, f16_out, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace nvamd
