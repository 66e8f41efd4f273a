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
// Waves 0-3 take the first half of K and waves 4-7 the second (2 x 2 wave
// tiles of BF/2 x BR/2 each), so every SIMD has a second wave to issue MFMAs
// while the first waits for its fragments, and a fragment is still read from
// LDS by two waves only. The halves' sums meet in LDS at the end, each half
// finishing half of the output fragments.
//
// Order of the sum: dense_rows_kernel's, so that a row has the same bits
// whatever rows share its call. There K is cut into slices, a slice into the
// k steps of four waves, each summed from zero, the four added in order and
// the slices in order. Here a half runs through its segments (one wave's
// steps there) one after the other: at a segment's end its accumulators are
// added to the running slice's sum, at a slice's end that to the finished
// slices' sum. With one slice the first half's result is segments 0 + 1 and
// the second hands over 2 and 3; with more, the second half takes the last
// one or two slices and hands over each.
//
// What bounds it: LDS traffic. A stage of the 64x64 tile reads 32 KB and
// writes 16 KB of LDS (384 cycles at 128 bytes a cycle) against 128 cycles
// of MFMAs per SIMD, and takes 0.19 us with every operand in L2; the fixed
// part of a launch (start, first loads, exchange, stores) is about 4 us. Us at
// 1000 rows, weights from memory: 1024 x 2048 11.3, 1024 x 3072 14.9, 6144 x
// 1024 25.7; summing each half as the steps come instead took 10.7, 14.2 and
// 23.8, and the decode-shaped kernel 64 rows at a time 65.9, 74.3 and 110.5.
// Measured and dropped: a stage's fragments read under the previous stage's
// MFMAs (1024 x 2048 11.7, 1024 x 3072 14.9: the segments' ends break the
// overlap, and the 128x64 tile has no registers for it).
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

// Waits for the wave's LDS reads. (The builtins, unlike inline asm, tell the
// compiler so: it adds no waits of its own where branches meet.)
__device__ __forceinline__ void wait_lds() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(15 | 7 << 4 | 3 << 14);
}

// Waits until at most N vector memory operations of this wave are in flight,
// then for the workgroup.
template <int N>
__device__ __forceinline__ void wait_loads_and_barrier() {
  static_assert(N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | 7 << 4 | 15 << 8 | (N >> 4) << 14);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// A launch's parameters, in two cache lines.
struct TileParams {
  const void *x, *w, *bias;
  void *out0, *out1, *out2;
  int rows, K, N, n1, n2;
  int ntiles, nfb, nrb, band, per;
  int steps, cut;    // a segment's k steps; the first half takes steps [0, cut)
  int slices, q, r;  // S / slices, S % slices
  int rem;           // (the second half's first slice x S) mod slices
  int second;        // slices of the second half
  int packed, xpacked, opacked;
};

template <typename T, int EPI, int BF, int BR, int NB, bool SLICED>
__global__ __launch_bounds__(64 * kTWaves, 4) void dense_tile_kernel(TileParams p) {
  constexpr int FT = BF / 32, RT = BR / 32;  // 16x16 fragments of a wave tile
  constexpr int NI = FT * RT;
  constexpr int NO = NI > 1 ? NI / 2 : 1;    // items a k half finishes (NI == 1: half 0)
  constexpr int FA = BF / 16 * 2, FB = BR / 16 * 2;  // fragments of a stage
  constexpr int L = (FA + FB) / kTWaves;             // of them per wave
  static_assert((FA + FB) % kTWaves == 0 && (NI == 1 || NI % 2 == 0), "tile shape");
  static_assert(12 * NO <= NB * (FA + FB), "the halves' exchange fits the buffers");
  __shared__ __align__(1024) char smem[NB][(FA + FB) * kFragBytes];

  const int ntiles = p.ntiles, nfb = p.nfb, nrb = p.nrb, band = p.band, per = p.per;
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

  const int cut = p.cut;
  const int nst = max(cut, S - cut), both = min(cut, S - cut);  // stages; those of both halves
  const int mine = kg ? S - cut : cut;

  // This wave's fragments of a stage: number wave + 8i, a tile's fragments of
  // the two halves being neighbours, so the wave copies for half wave % 2.
  const int load_base = wave & 1 ? cut : 0, load_last = wave & 1 ? S - 1 : cut - 1;
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
    const int s = min(load_base + st, load_last);  // the shorter half's last step again
#pragma unroll
    for (int i = 0; i < L; ++i)
      load_frag(src[i] + (uint32_t)s * (uint32_t)step[i],
                &smem[buf][(wave + kTWaves * i) * kFragBytes]);
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

  // acc: the running segment; cur: the running slice's finished segments (not
  // SLICED: the half's first segment); tot: the finished slices. Sums start
  // from -0, which leaves every addend as it is.
  f32x4_t acc[NI], cur[NI], tot[SLICED ? NI : 1];
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f}, none = {-0.f, -0.f, -0.f, -0.f};
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    acc[i] = zero;
    cur[i] = SLICED ? none : zero;
    if constexpr (SLICED) tot[i] = none;
  }
  int at = kg ? cut : 0, slice_end = S;  // ends of the running segment and slice
  int seg = 0;                           // the segment's number in its slice
  int left = 0;                          // steps to the segment's end
  int slices_left = kg ? p.second : p.slices - p.second;
  int rem = kg ? p.rem : 0;  // slice s ends at (s + 1) S / slices: the division's remainder
  auto next_slice = [&]() {
    rem += p.r;
    const bool carry = rem >= p.slices;
    rem -= carry ? p.slices : 0;
    slice_end = at + p.q + carry;
    seg = 0;
  };
  auto next_segment = [&]() {
    const int from = at;
    at = min(slice_end, from + p.steps);
    left = at - from;
  };
  if constexpr (SLICED) next_slice();
  next_segment();
  if (mine == 0) left = S + 1;
  // The running segment has ended: its sum joins its slice's, in order.
  auto end_segment = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      cur[i] = SLICED ? cur[i] + acc[i] : acc[i];
      acc[i] = zero;
    }
    if constexpr (SLICED) {
      ++seg;
      if (at == slice_end) {
        if (seg < 4)  // the slice's last segments are empty: zeros
#pragma unroll
          for (int i = 0; i < NI; ++i) cur[i] += zero;
        if (--slices_left > 0) {
#pragma unroll
          for (int i = 0; i < NI; ++i) {
            tot[i] += cur[i];
            cur[i] = none;
          }
        }
        next_slice();
      }
      next_segment();
    } else {
      left = S + 1;
    }
  };

#pragma unroll
  for (int b = 0; b < NB - 1; ++b)
    if (b < nst) load_stage(b, b);
  // One stage: its buffer published, the next one requested into the buffer
  // the previous stage has been read out of, its fragments on their way to
  // registers.
  int buf = 0;
  auto fetch = [&](int st, auto steady, u32x4_t (&a)[FT],
                   u32x4_t (&b)[RT]) __attribute__((always_inline)) {
    wait_lds();
    // Stage st has landed once only the NB - 2 requested after it are left.
    if (steady || st + NB - 2 < nst)
      wait_loads_and_barrier<(NB - 2) * L>();
    else
      wait_loads_and_barrier<0>();
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
    __builtin_amdgcn_sched_barrier(0);  // a segment's end runs under these reads
  };
  auto multiply = [&](const u32x4_t (&a)[FT],
                      const u32x4_t (&b)[RT]) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < FT; ++f)
#pragma unroll
      for (int r = 0; r < RT; ++r) acc[f * RT + r] = DenseMma<T>::run(a[f], b[r], acc[f * RT + r]);
    __builtin_amdgcn_sched_barrier(0);
  };
  // The stages whose prefetch and steps exist in both halves, then the rest.
  // Segments of many slices are short: their ends are looked for in every
  // stage, and added up while its fragments arrive. One slice's two are loops
  // of their own (the branch in the loop takes registers that the 128x64 tile
  // does not have).
  u32x4_t a[FT], b[RT];
  const int steady = min(nst - NB + 1, both);
  int st = 0;
  if constexpr (SLICED) {
    for (; st < steady; ++st) {
      fetch(st, std::true_type{}, a, b);
      if (left == 0) end_segment();
      multiply(a, b);
      --left;
    }
    for (; st < nst; ++st) {
      fetch(st, std::false_type{}, a, b);
      if (st < mine) {
        if (left == 0) end_segment();
        multiply(a, b);
        --left;
      }
    }
    end_segment();
  } else {
    while (st < steady) {
      const int end = min(steady, st + left);
      left -= end - st;
      do {
        fetch(st, std::true_type{}, a, b);
        multiply(a, b);
      } while (++st < end);
      if (left == 0) end_segment();
    }
    for (; st < nst; ++st) {
      fetch(st, std::false_type{}, a, b);
      if (st < mine) {
        multiply(a, b);
        if (--left == 0) end_segment();
      }
    }
  }

  // Exchange: the first half hands over its sum, the second its two addends
  // (-0 where it has one), of the items the other finishes.
  wait_lds();
  wait_loads_and_barrier<0>();
  if (kg == 0) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if constexpr (SLICED)
        cur[i] = tot[i] + cur[i];
      else
        cur[i] += acc[i];
    }
  }
  auto addend = [&](int i, int which) __attribute__((always_inline)) {
    if constexpr (SLICED)
      return which == 0 ? tot[i] : cur[i];
    else
      return which == 0 ? cur[i] : acc[i];
  };
  f32x4_t* ex = reinterpret_cast<f32x4_t*>(&smem[0][0]) + (wave & 3) * 3 * NO * 64 + lane;
  if (kg == 1) {
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      ex[(NO + o) * 64] = addend(o, 0);
      ex[(2 * NO + o) * 64] = addend(o, 1);
    }
  } else if (NI > 1) {
#pragma unroll
    for (int o = 0; o < NO; ++o) ex[o * 64] = cur[NI > 1 ? NO + o : 0];
  }
  __syncthreads();
  if (!finishes) return;
  f32x4_t sum[NO];
  if (kg == 0) {
    f32x4_t x0[NO], x1[NO];
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      x0[o] = ex[(NO + o) * 64];
      x1[o] = ex[(2 * NO + o) * 64];
    }
#pragma unroll
    for (int o = 0; o < NO; ++o) sum[o] = cur[o] + x0[o] + x1[o];
  } else {
#pragma unroll
    for (int o = 0; o < NO; ++o) sum[o] = ex[o * 64];
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      const int i = NI > 1 ? NO + o : 0;
      sum[o] = sum[o] + addend(i, 0) + addend(i, 1);
    }
  }

#pragma unroll
  for (int o = 0; o < NO; ++o) {
    const int it = item_of(o);
    const f32x4_t v = sum[o];
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

// A grid holds fewer than 2^32 threads: more tiles run as several launches.
constexpr long long kMaxTiles = (1LL << 32) / (64 * kTWaves) - 8;

template <typename T, int EPI, int BF, int BR, int NB>
int run_tile(const DenseParams& p, hipStream_t s) {
  const int ntiles = EPI == kEpiSiluMul ? p.n1 / 8 : p.N / 16;
  const int nfb = (int)((ntiles * 16LL + BF - 1) / BF);
  if (nfb > kMaxTiles) return fail(RLSE_ERR_INVALID_VALUE, "dense: too many features");
  const int S = p.K / 32, n = p.ksplit;
  const int second = n > 3 ? 2 : 1, first = n - second;  // slices of the halves
  TileParams t;
  t.w = p.w, t.bias = p.bias;
  t.K = p.K, t.N = p.N, t.n1 = p.n1, t.n2 = p.n2;
  t.ntiles = ntiles, t.nfb = nfb;
  t.steps = p.steps, t.cut = n > 1 ? first * S / n : std::min(2 * p.steps, S);
  t.slices = n, t.q = S / n, t.r = S % n, t.rem = first * (S % n) % n;
  t.second = second;
  t.packed = p.packed, t.xpacked = p.xpacked, t.opacked = p.opacked;
  const long long max_rows = kMaxTiles / nfb * BR;
  for (long long r0 = 0; r0 < p.rows; r0 += max_rows) {
    const int rows = (int)std::min<long long>(p.rows - r0, max_rows);
    const int nrb = (int)((rows + BR - 1LL) / BR);
    const int per = (int)(((long long)nfb * nrb + 7) / 8);
    // A run of band x (per / band) tiles reads band * BF + (per / band) * BR
    // rows of the two operands: least at band = sqrt(per * BR / BF).
    const int square = (int)(sqrt((double)per * BR / BF) + 0.5);
    t.band = std::min(nfb, std::max(std::max(1, square), (per + nrb - 1) / nrb));
    t.rows = rows, t.nrb = nrb, t.per = per;
    // (Whole 16-row tiles: packed rows are as far apart as row-major ones.)
    auto from = [&](const void* base, int features) {
      return base ? (void*)((T*)base + (size_t)r0 * features) : nullptr;
    };
    t.x = from(p.x, p.K);
    t.out0 = from(p.out0, EPI == kEpiResidual ? p.N : p.n1);
    t.out1 = from(p.out1, p.n2 - p.n1), t.out2 = from(p.out2, p.N - p.n2);
    if (n > 1)
      hipLaunchKernelGGL((dense_tile_kernel<T, EPI, BF, BR, NB, true>), dim3(8 * per),
                         dim3(64 * kTWaves), 0, s, t);
    else
      hipLaunchKernelGGL((dense_tile_kernel<T, EPI, BF, BR, NB, false>), dim3(8 * per),
                         dim3(64 * kTWaves), 0, s, t);
    const int rc = launch_status("dense_tile_kernel");
    if (rc) return rc;
  }
  return RLSE_OK;
}

// The tile shape, by how many workgroups each makes of the output. A larger
// tile reads fewer bytes per product, a smaller one puts more compute units
// to work; with several slices of K the segments' ends cost the largest most.
// Measured over 80 to 2000 rows of the projections of Qwen3-0.6B,
// Qwen2.5-0.5B and layers of 3584 and 4096 features (us, 32x32 / 64x64 / 128x64):
//   up to 256 tiles of 32x32    1024 x 2048, 256 rows: 8.6 / 10.6 / 17.3
//   (288 of them                1152 x 896, 256 rows: 7.9 / 7.0 / 12.4)
//   up to 384 tiles of 64x64    6144 x 1024, 256 rows: 18.2 / 10.8 / 11.2
//   (512                        4096 x 4096, 512 rows: 61.0 / 33.1 / 30.2)
//   slices, up to 640 of them   1152 x 896, 2000 rows: 27.9 / 14.8 / 19.6
//   (896                        3584 x 18944, 1000 rows: 491 / 257 / 187)
//   above                       6144 x 1024, 1000 rows: 64.1 / 28.7 / 25.2
// 128x128 tiles (one workgroup per compute unit) were at best equal to
// 128x64, and deeper buffers changed nothing.
template <typename T, int EPI>
int pick_tile(const DenseParams& p, hipStream_t s) {
  const long long f = p.N, r = p.rows;
  auto tiles = [&](int bf, int br) { return ((f + bf - 1) / bf) * ((r + br - 1) / br); };
  if (tiles(32, 32) <= 256) return run_tile<T, EPI, 32, 32, 8>(p, s);
  if (tiles(64, 64) <= (p.ksplit > 1 ? 640 : 384)) return run_tile<T, EPI, 64, 64, 4>(p, s);
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
