// Prompt-shaped projections on MFMA: y[rows][N] = x[rows][K] . W[N][K]^T for
// more rows than a decode batch, bf16/f16 in, f32 accumulation, with the fused
// epilogues (q/k/v, residual, SwiGLU) of the decode-shaped dense_rows_kernel.
//
// A workgroup of 8 waves owns BF features x BR rows and streams K in stages
// of two 32-wide k steps through NB LDS buffers: global_load_lds copies one
// MFMA operand fragment (16 rows x 32 k, 1 KiB) per wave instruction, in the
// lane order the MFMA takes it, so a fragment is read back with one
// conflict-free ds_read_b128 whatever the source order (packed or
// row-major). Each buffer is requested NB - 1 stages before its use, and one
// barrier a stage both publishes a buffer and frees the previous one.
//
// Waves 0-3 take the even k steps and waves 4-7 the odd ones (2 x 2 wave
// tiles of BF/2 x BR/2 each), so every SIMD has a second wave to issue MFMAs
// while the first waits for its fragments, and a fragment is still read from
// LDS by two waves only. The two halves' sums meet in LDS at the end, each
// half finishing half of the output fragments. A row's sum over K is the
// same whatever tile shape the launch takes.
//
// What bounds it: LDS traffic. A stage of the 64x64 tile reads 32 KB and
// writes 16 KB of LDS (384 cycles at 128 bytes a cycle) against 128 cycles
// of MFMAs per SIMD, and takes 0.19 us with every operand in L2; the fixed
// part of a launch (start, first loads, exchange, stores) is 3.4 us. Reading
// a stage's fragments into registers under the previous stage's MFMAs took
// the 1024 x 3072 product at 1000 rows from 16.8 to 14.7 us. Before this
// kernel such products ran the decode-shaped one 64 rows at a time: the
// seven calls of a Qwen3-0.6B layer's dense half at 1000 rows took 364 us.
#include <math.h>

#include <algorithm>

#include "dense_common.cuh"
#include "host_common.h"

#pragma clang fp contract(off)

namespace rlse {
namespace {

constexpr int kTWaves = 8;
constexpr int kFragBytes = 1024;

// Copies 16 bytes per lane from src to lds + 16 * lane (lds wave-uniform).
__device__ __forceinline__ void load_frag(const char* src, char* lds) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void*)src,
      (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

// Waits until at most N vector memory operations of this wave are in flight
// and its LDS reads are done, then for the workgroup.
template <int N>
__device__ __forceinline__ void wait_and_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <typename T, int EPI, int BF, int BR, int NB>
__global__ __launch_bounds__(64 * kTWaves) void dense_tile_kernel(DenseParams p, int ntiles,
                                                                  int nfb, int nrb, int band,
                                                                  int per) {
  constexpr int FT = BF / 32, RT = BR / 32;  // 16x16 fragments of a wave tile
  constexpr int NI = FT * RT;
  constexpr int NO = NI > 1 ? NI / 2 : 1;    // items a k half finishes (NI == 1: half 0)
  constexpr int FA = BF / 16 * 2, FB = BR / 16 * 2;  // fragments of a stage
  constexpr int L = (FA + FB) / kTWaves;             // of them per wave
  static_assert((FA + FB) % kTWaves == 0 && (NI == 1 || NI % 2 == 0), "tile shape");
  static_assert(4 * NI <= NB * (FA + FB), "the halves' exchange fits the buffers");
  __shared__ __align__(1024) char smem[NB][(FA + FB) * kFragBytes];

  // Workgroup b runs on XCD b % 8, and each XCD takes a contiguous run of
  // `per` tiles in an order that walks bands of `band` feature tiles row by
  // row: a run is a near-square block of the output, so the weights and rows
  // an XCD's L2 fetches are as few as they can be.
  const int wid = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (wid >= nfb * nrb) return;
  const int bd = wid / (band * nrb), in_band = wid - bd * band * nrb;
  const int width = min(band, nfb - bd * band);
  const int rb = in_band / width, fb = bd * band + in_band - rb * width;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave >> 2, wf = (wave >> 1) & 1, wr = wave & 1;
  const int fi = lane & 15, g = lane >> 4;
  const int K = p.K, S = K >> 5;
  const int last_rt = (p.rows - 1) >> 4;

  // This wave's fragments of a stage: number wave + 8i, a tile's two k steps
  // being neighbours, so the wave's k step within a stage is wave % 2.
  const char* src[L];
  int step[L];  // bytes from k step to k step
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int f = wave + kTWaves * i;
    if (f < FA) {
      const int tile = min(fb * (BF / 16) + (f >> 1), ntiles - 1);
      const int row = EPI == kEpiSiluMul
                          ? (fi < 8 ? tile * 8 + fi : p.n1 + tile * 8 + (fi - 8))
                          : tile * 16 + fi;
      src[i] = p.packed ? (const char*)p.w + ((size_t)tile * S * 64 + lane) * 16
                        : (const char*)p.w + (size_t)row * K * 2 + 16 * g;
      step[i] = p.packed ? kFragBytes : 64;
    } else {
      // Row tiles past the batch read its last one.
      const int rt = min(rb * (BR / 16) + ((f - FA) >> 1), last_rt);
      src[i] = p.xpacked ? (const char*)p.x + ((size_t)rt * S * 64 + lane) * 16
                         : (const char*)p.x + (size_t)min(16 * rt + fi, p.rows - 1) * K * 2 +
                               16 * g;
      step[i] = p.xpacked ? kFragBytes : 64;
    }
  }
  auto load_stage = [&](int st, int buf) __attribute__((always_inline)) {
    const int s = min(2 * st + (wave & 1), S - 1);  // an odd S's last step twice
#pragma unroll
    for (int i = 0; i < L; ++i)
      load_frag(src[i] + (uint32_t)s * (uint32_t)step[i], &smem[buf][(wave + kTWaves * i) * kFragBytes]);
  };

  // The output fragments this wave finishes, and their epilogue operands,
  // requested ahead of the main loop.
  auto item_of = [&](int o) { return NI > 1 ? kg * NO + o : 0; };
  auto feature = [&](int it) {
    return (fb * (BF / 16) + wf * FT + it / RT) * 16 + 4 * g;  // SwiGLU: of gate and up rows
  };
  auto row_of = [&](int it) { return rb * BR + (wr * RT + it % RT) * 16 + fi; };
  const bool finishes = NI > 1 || kg == 0;
  uint2 pre[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    const int it = item_of(o), n = feature(it), r = row_of(it);
    pre[o] = make_uint2(0, 0);
    if (finishes && n < ntiles * 16 && r < p.rows) {
      if constexpr (EPI == kEpiResidual)
        pre[o] = *reinterpret_cast<const uint2*>((const T*)p.out0 + (size_t)r * p.N + n);
      if constexpr (EPI == kEpiQkv)
        if (p.bias) pre[o] = *reinterpret_cast<const uint2*>((const T*)p.bias + n);
    }
  }

  f32x4_t acc[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int nst = (S + 1) >> 1;
#pragma unroll
  for (int b = 0; b < NB - 1; ++b)
    if (b < nst) load_stage(b, b);
  // One stage: its buffer published, the next one requested into the buffer
  // the previous stage has been read out of, its fragments on their way to
  // registers. The MFMAs of a stage run under the next one's LDS reads.
  int buf = 0;
  auto fetch = [&](int st, auto steady, u32x4_t (&a)[FT],
                   u32x4_t (&b)[RT]) __attribute__((always_inline)) {
    // Stage st has landed once only the NB - 2 requested after it are left.
    if (steady || st + NB - 2 < nst)
      wait_and_barrier<(NB - 2) * L>();
    else
      wait_and_barrier<0>();
    if (steady || st + NB - 1 < nst) load_stage(st + NB - 1, buf == 0 ? NB - 1 : buf - 1);
    const char* sm = smem[buf];
#pragma unroll
    for (int f = 0; f < FT; ++f)
      a[f] = *reinterpret_cast<const u32x4_t*>(sm + ((wf * FT + f) * 2 + kg) * kFragBytes +
                                               lane * 16);
#pragma unroll
    for (int r = 0; r < RT; ++r)
      b[r] = *reinterpret_cast<const u32x4_t*>(sm + (FA + (wr * RT + r) * 2 + kg) * kFragBytes +
                                               lane * 16);
    buf = buf + 1 == NB ? 0 : buf + 1;
    __builtin_amdgcn_sched_barrier(0);  // the reads are issued before the MFMAs they hide under
  };
  auto multiply = [&](const u32x4_t (&a)[FT],
                      const u32x4_t (&b)[RT]) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < FT; ++f)
#pragma unroll
      for (int r = 0; r < RT; ++r) acc[f * RT + r] = Mma16<T>::run(a[f], b[r], acc[f * RT + r]);
    __builtin_amdgcn_sched_barrier(0);
  };
  // The steady loop has no branches: a join would make the compiler wait for
  // every LDS read in flight before the MFMAs. The last stages follow it.
  u32x4_t a0[FT], b0[RT], a1[FT], b1[RT];
  fetch(0, std::false_type{}, a0, b0);
  int st = 1;
  for (; st + NB < nst; st += 2) {
    fetch(st, std::true_type{}, a1, b1);
    multiply(a0, b0);
    fetch(st + 1, std::true_type{}, a0, b0);
    multiply(a1, b1);
  }
  for (; st < nst; st += 2) {
    fetch(st, std::false_type{}, a1, b1);
    multiply(a0, b0);
    if (st + 1 < nst) fetch(st + 1, std::false_type{}, a0, b0);
    if (2 * st + kg < S) multiply(a1, b1);
  }
  // An odd stage count leaves its last stage, whose second k step may not exist.
  if ((nst & 1) && 2 * (nst - 1) + kg < S) multiply(a0, b0);

  // Exchange: each half hands the other the items it does not finish.
  wait_and_barrier<0>();
  f32x4_t* ex = reinterpret_cast<f32x4_t*>(&smem[0][0]) + (size_t)(wave & 3) * NI * 64 + lane;
#pragma unroll
  for (int i = 0; i < NI; ++i)
    if (NI > 1 ? (i / NO != kg) : kg == 1) ex[i * 64] = acc[i];
  __syncthreads();
  if (!finishes) return;

#pragma unroll
  for (int o = 0; o < NO; ++o) {
    f32x4_t mine = acc[o];
    if constexpr (NI > 1) mine = kg == 0 ? acc[o] : acc[NO + o];
    const int it = item_of(o);
    const f32x4_t other = ex[it * 64];
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = mine[e] + other[e];
    const int n = feature(it), r = row_of(it);
    const bool in = n < ntiles * 16 && r < p.rows;
    float pv[8];
    Packet<T>::unpack(make_uint4(pre[o].x, pre[o].y, 0, 0), pv);
    float out[4];
    if constexpr (EPI == kEpiSiluMul) {
      // Lane l < 32 holds four gate features, lane l + 32 the matching up
      // features of the same row.
      float up[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) up[e] = __shfl_xor(v[e], 32, 64);
      if (!in || lane >= 32) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        out[e] = silu_mul_rounded<T>(round_cvt<T>(v[e]), round_cvt<T>(up[e]));
      const int c = (n >> 4) * 8 + 4 * g;
      store4<T>((T*)p.out0 +
                    (p.opacked ? (((size_t)(r >> 4) * (p.n1 >> 5) + (c >> 5)) * 64 + (r & 15) +
                                  16 * ((c & 31) >> 3)) * 8 + (c & 7)
                               : (size_t)r * p.n1 + c),
                out);
    } else {
      if (!in) continue;
      if constexpr (EPI == kEpiResidual) {
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = pv[e] + round_cvt<T>(v[e]);
        store4<T>((T*)p.out0 + (size_t)r * p.N + n, out);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = round_cvt<T>(v[e]) + (p.bias ? pv[e] : 0.f);
        T* dst;
        if (n >= p.n2)
          dst = (T*)p.out2 + (size_t)r * (p.N - p.n2) + (n - p.n2);
        else if (n >= p.n1)
          dst = (T*)p.out1 + (size_t)r * (p.n2 - p.n1) + (n - p.n1);
        else
          dst = (T*)p.out0 + (size_t)r * p.n1 + n;
        store4<T>(dst, out);
      }
    }
  }
}

template <typename T, int EPI, int BF, int BR, int NB>
int run_tile(const DenseParams& p, hipStream_t s) {
  const int ntiles = EPI == kEpiSiluMul ? p.n1 / 8 : p.N / 16;
  const int nfb = (ntiles * 16 + BF - 1) / BF, nrb = (p.rows + BR - 1) / BR;
  const long long total = (long long)nfb * nrb;
  if (total > (1LL << 28)) return fail(RLSE_ERR_INVALID_VALUE, "dense: too many rows");
  const int per = (int)((total + 7) / 8);
  // A run of band x (per / band) tiles reads band * BF + (per / band) * BR
  // rows of the two operands: least at band = sqrt(per * BR / BF).
  const int square = (int)(sqrt((double)per * BR / BF) + 0.5);
  const int band = std::min(nfb, std::max(std::max(1, square), (per + nrb - 1) / nrb));
  hipLaunchKernelGGL((dense_tile_kernel<T, EPI, BF, BR, NB>), dim3(8 * per), dim3(64 * kTWaves), 0,
                     s, p, ntiles, nfb, nrb, band, per);
  return launch_status("dense_tile_kernel");
}

// The tile shape, by how many workgroups each makes of the output. A larger
// tile reads fewer bytes per product, a smaller one puts more compute units
// to work; measured over 65 to 2048 rows of Qwen3-0.6B's and Qwen2.5-0.5B's
// projections (us, 32x32 / 64x64 / 128x64):
//   up to 256 tiles of 32x32       1024 x 2048, 256 rows:  8.1 / 12.4 / 15.2
//   up to 320 tiles of 64x64       1024 x 2048, 1000 rows: 21.8 / 13.1 / 15.6
//   above that                     6144 x 1024, 1000 rows: 53.1 / 27.0 / 23.6
//                                  1024 x 2048, 1500 rows: 30.3 / 22.7 / 16.2
// 128x128 tiles (one workgroup per compute unit) were at best equal to
// 128x64 (4096 x 1024, 1000 rows: 15.0 against 14.9; 6144 x 1024: 31.2
// against 23.6) on these shapes, and deeper buffers changed nothing.
template <typename T, int EPI>
int pick_tile(const DenseParams& p, hipStream_t s) {
  const long long f = p.N, r = p.rows;
  auto tiles = [&](int bf, int br) { return ((f + bf - 1) / bf) * ((r + br - 1) / br); };
  if (tiles(32, 32) <= 256) return run_tile<T, EPI, 32, 32, 8>(p, s);
  if (tiles(64, 64) <= 320) return run_tile<T, EPI, 64, 64, 4>(p, s);
  return run_tile<T, EPI, 128, 64, 3>(p, s);
}

template <int EPI>
int by_type(int dtype, const DenseParams& p, hipStream_t s) {
  return dtype == RLSE_DTYPE_BF16 ? pick_tile<bf16, EPI>(p, s) : pick_tile<f16, EPI>(p, s);
}

}  // namespace

int launch_dense_tile(int epi, int dtype, const DenseParams& p, hipStream_t s) {
  switch (epi) {
    case kEpiQkv: return by_type<kEpiQkv>(dtype, p, s);
    case kEpiResidual: return by_type<kEpiResidual>(dtype, p, s);
    default: return by_type<kEpiSiluMul>(dtype, p, s);
  }
}

}  // namespace rlse
