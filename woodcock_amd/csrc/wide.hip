// wide.hip -- many-row passes on the matrix cores: prompts through the drafter
// (python/woodcock/spec.py:129-141) and the backend operations over many rows
// (include/woodcock/ops.h:9-24).
//
// The few-row kernels stream every weight once per tile of at most 16 rows, so
// a prompt of L rows streams them L / 16 times.  Here a pass covers up to
// kWideRows rows with tiled GEMMs whose activations keep fp32 precision: an fp32
// value is the exact sum of three bf16 terms of 8 significant bits each (its
// mantissa cut in three), so x . w with a bf16 weight is three
// v_mfma_f32_16x16x32_bf16 products with fp32 accumulation and no rounding of
// the inputs.
#include "wide.h"

namespace wc {

typedef __bf16 wbf16x8 __attribute__((ext_vector_type(8)));
typedef float wf32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int wu32x4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ the three-term split

// x = hi + mid + lo exactly (|x| normal): each term is the top 16 bits of what
// the terms before it left.  An infinite x is its own hi term with nothing left.
__device__ __forceinline__ void wd_split1(float x, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  hi = __float_as_uint(x) & 0xffff0000u;
  const float h = __uint_as_float(hi);
  const float r = x == h ? 0.f : x - h;
  mid = __float_as_uint(r) & 0xffff0000u;
  lo = __float_as_uint(r - __uint_as_float(mid));
}

// 8 fp32 -> three 16-byte bf16 vectors
__device__ __forceinline__ void wd_split8(const float* x, uint4& hi, uint4& mid, uint4& lo) {
  uint32_t h[8], m[8], l[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) wd_split1(x[e], h[e], m[e], l[e]);
  auto pk = [](uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); };  // the top halves
  hi = make_uint4(pk(h[0], h[1]), pk(h[2], h[3]), pk(h[4], h[5]), pk(h[6], h[7]));
  mid = make_uint4(pk(m[0], m[1]), pk(m[2], m[3]), pk(m[4], m[5]), pk(m[6], m[7]));
  lo = make_uint4(pk(l[0], l[1]), pk(l[2], l[3]), pk(l[4], l[5]), pk(l[6], l[7]));
}

// Split activations ("planes") as the GEMM reads them: row tile m / 16, 32-wide
// k step k / 32, term p, then the 16-byte fragment of MFMA lane
// (m % 16) + 16 ((k % 32) / 8): one row tile's k step is 3 KB in a run.
__device__ __forceinline__ int64_t wd_index(int m, int k, int steps, int p) {
  return ((static_cast<int64_t>(m >> 4) * steps + (k >> 5)) * 3 + p) * 512 + ((m & 15) + 16 * ((k & 31) >> 3)) * 8 +
         (k & 7);
}

// ------------------------------------------------------------------ activations -> planes

constexpr int kWidePrepThreads = 512;

// Block (row tile, k part, segment): 16 rows, each normalised over its whole
// segment (every part sums the squares itself: the rows come from L2), the
// part's share of the k steps written as planes.  A wave writes one whole
// fragment kilobyte per term and reads 16 rows x 128 bytes.
template <bool BF16>
__device__ __forceinline__ void wide_prep_rows(const WidePrepArgs& a, const WidePrepArgs::Seg& sg, int step0,
                                               float* s_ss) {
  constexpr int NW = kWidePrepThreads / kWave;
  const int t = threadIdx.x, lane = t % kWave, wave = t / kWave;
  const int mt = blockIdx.x, m = mt * 16 + lane % 16, g = lane / 16;
  const bool live = m < a.M;
  const int mr = min(m, a.M - 1);
  int64_t row = sg.row_idx ? static_cast<int64_t>(sg.row_idx[mr]) + sg.row_add : mr;
  if (sg.max_row > 0) row = row < 0 ? 0 : row >= sg.max_row ? sg.max_row - 1 : row;
  const int steps = sg.K / 32;
  const char* base = static_cast<const char*>(sg.x) + row * sg.ld * (BF16 ? 2 : 4);
  auto load = [&](int s, float* v) {
    const int k = s * 32 + g * 8;
    if constexpr (BF16) {
      const uint4 q = *reinterpret_cast<const uint4*>(base + k * 2);
      v[0] = bf16_lo(q.x); v[1] = bf16_hi(q.x); v[2] = bf16_lo(q.y); v[3] = bf16_hi(q.y);
      v[4] = bf16_lo(q.z); v[5] = bf16_hi(q.z); v[6] = bf16_lo(q.w); v[7] = bf16_hi(q.w);
    } else {
      const float4 u = *reinterpret_cast<const float4*>(base + k * 4);
      const float4 w = *reinterpret_cast<const float4*>(base + k * 4 + 16);
      v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w; v[4] = w.x; v[5] = w.y; v[6] = w.z; v[7] = w.w;
    }
  };
  float inv = 1.f;
  if (sg.gain) {
    float ss = 0.f;
#pragma unroll 4
    for (int s = wave; s < steps; s += NW) {
      float v[8];
      load(s, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
    }
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (g == 0) s_ss[wave * 16 + lane] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) tot += s_ss[w * 16 + lane % 16];
    inv = 1.f / sqrtf(tot / static_cast<float>(sg.K) + a.eps);
  }
  const int parts = gridDim.y, per = (steps + parts - 1) / parts;
  const int sb = blockIdx.y * per, se = min(steps, sb + per);
#pragma unroll 2
  for (int s = sb + wave; s < se; s += NW) {
    float v[8];
    load(s, v);
    if (sg.gain) {
      const uint4 q = *reinterpret_cast<const uint4*>(sg.gain + s * 32 + g * 8);
      const float gv[8] = {bf16_lo(q.x), bf16_hi(q.x), bf16_lo(q.y), bf16_hi(q.y),
                           bf16_lo(q.z), bf16_hi(q.z), bf16_lo(q.w), bf16_hi(q.w)};
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = v[e] * gv[e] * inv;
    }
    if (!live)
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = 0.f;
    uint4 hi, mid, lo;
    wd_split8(v, hi, mid, lo);
    uint4* dst = reinterpret_cast<uint4*>(a.xa) + (static_cast<int64_t>(mt) * a.steps + step0 + s) * 192 + lane;
    dst[0] = hi;
    dst[64] = mid;
    dst[128] = lo;
  }
}

__global__ __launch_bounds__(kWidePrepThreads) void k_wide_prep(WidePrepArgs a) {
  __shared__ float s_ss[kWidePrepThreads / kWave * 16];
  const int z = blockIdx.z;
  // the segments by constant index: a run-time index would put the array in scratch memory
  int step0 = 0;
  WidePrepArgs::Seg sg = a.seg[0];
  if (z == 1) {
    sg = a.seg[1];
    step0 = a.seg[0].K / 32;
  } else if (z == 2) {
    sg = a.seg[2];
    step0 = (a.seg[0].K + a.seg[1].K) / 32;
  }
  if (sg.bf16)
    wide_prep_rows<true>(a, sg, step0, s_ss);
  else
    wide_prep_rows<false>(a, sg, step0, s_ss);
}

// ------------------------------------------------------------------ the GEMM

// k steps whose leading-term products share an accumulator chain before they
// are folded into the running sum (see k_wide_gemm)
constexpr int kWideFlush = 8;

// 16 bytes per lane straight into LDS: lane l's to dst + l
__device__ __forceinline__ void wd_load_lds(const void* src, wu32x4* dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}
// This wave's LDS reads and all but its last N loads into LDS are done, then the
// block's waves meet.  (A fence would wait for every load into LDS.)
template <int N>
__device__ __forceinline__ void wd_stage_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | (N >> 4) << 14);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// N consecutive fragments (a kilobyte apart) from LDS address `at`, complete on
// return.  Written out because the compiler, reading an array that loads into
// LDS fill, waits for all of those loads.
template <int N>
__device__ __forceinline__ void wd_read_lds(uint32_t at, wu32x4 (&r)[N]) {
  static_assert(N == 1 || N == 2 || N == 3 || N == 4 || N == 6, "fragments per read");
  if constexpr (N == 1)
    asm volatile(
                 "ds_read_b128 %0, %1 offset:0\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(r[0])
                 : "v"(at)
                 : "memory");
  else if constexpr (N == 2)
    asm volatile(
                 "ds_read_b128 %0, %2 offset:0\n\t"
                 "ds_read_b128 %1, %2 offset:1024\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(r[0]), "=&v"(r[1])
                 : "v"(at)
                 : "memory");
  else if constexpr (N == 3)
    asm volatile(
                 "ds_read_b128 %0, %3 offset:0\n\t"
                 "ds_read_b128 %1, %3 offset:1024\n\t"
                 "ds_read_b128 %2, %3 offset:2048\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2])
                 : "v"(at)
                 : "memory");
  else if constexpr (N == 4)
    asm volatile(
                 "ds_read_b128 %0, %4 offset:0\n\t"
                 "ds_read_b128 %1, %4 offset:1024\n\t"
                 "ds_read_b128 %2, %4 offset:2048\n\t"
                 "ds_read_b128 %3, %4 offset:3072\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
                 : "v"(at)
                 : "memory");
  else if constexpr (N == 6)
    asm volatile(
                 "ds_read_b128 %0, %6 offset:0\n\t"
                 "ds_read_b128 %1, %6 offset:1024\n\t"
                 "ds_read_b128 %2, %6 offset:2048\n\t"
                 "ds_read_b128 %3, %6 offset:3072\n\t"
                 "ds_read_b128 %4, %6 offset:4096\n\t"
                 "ds_read_b128 %5, %6 offset:5120\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5])
                 : "v"(at)
                 : "memory");
}
__device__ __forceinline__ uint32_t wd_lds_address(const wu32x4* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) wu32x4*)p));
}

// Block tile BM rows x BN weight rows; WK groups of WM x WN waves, group g on
// the k steps s = g (mod WK) of 32, a wave on (BM / WM) x (BN / WN) of its
// group's product.  A stage is WK k steps of both operands, loaded straight
// into LDS in fragment order (one kilobyte per 16 x 32 tile, lane by lane: the
// reads are conflict-free 16-byte ones); NS stages rotate, so a load has NS - 1
// stages of products to land, with one barrier per stage.  The weights are the
// MFMA's A operand and the rows its B operand, so a lane ends with four
// consecutive output columns of one row.  Blocks go to the XCDs in runs of
// consecutive tiles, rows fastest: an XCD's blocks share their weight tiles in
// its L2.
//
// Accuracy: one accumulator chain over all of K rounds at every MFMA at the
// size of the running sum (8.7e-7 relative off 64 bits on a fuse of K 6144,
// against 1.3e-7 for the few-row kernels' short chains).  So the leading
// terms' products of kWideFlush steps are summed on their own and folded into
// the running sum, the fold's own rounding error going to the accumulator of
// the small terms (1.1e-7).
template <int BM, int BN, int WM, int WN, int WK, int NS, int WPE, int EPI>
__global__ __launch_bounds__(WM* WN* WK* kWave) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void k_wide_gemm(
    WideArgs a, int mblocks) {
  constexpr int GW = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16;
  constexpr int ACH = BM / 16 * 3, WCH = BN / 16;  // kilobytes per k step
  constexpr int AR = ACH / GW, WR = WCH / GW, PL = AR + WR;
  constexpr int SV = WK * (ACH + WCH) * 64;        // 16-byte vectors per stage
  static_assert(ACH % GW == 0 && WCH % GW == 0, "whole kilobytes per wave");
  static_assert((NS == 2 || NS == 4) && kWideFlush % NS == 0, "folds fall on the last stage of a round");
  static_assert(WK == 1 || (WK - 1) * BM * BN * 4 <= SV * 16, "the groups' sums fit a stage");
  // one array per stage, so that the reads of a stage wait for its own loads only
  __shared__ wu32x4 s_0[SV], s_1[SV], s_2[NS > 2 ? SV : 1], s_3[NS > 2 ? SV : 1];
  const int t = threadIdx.x, lane = t % kWave;
  const int wv = __builtin_amdgcn_readfirstlane(t / kWave), grp = wv / GW, wave = wv % GW;
  int blk;
  {
    const int nb = gridDim.x, q = nb / 8, r = nb % 8, x = blockIdx.x % 8, i = blockIdx.x / 8;
    blk = x < r ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
  }
  const int m0 = (blk % mblocks) * BM, cb = blk / mblocks;
  constexpr bool pair = EPI == kWideSiluPair;

  // chunk c of the rows' planes: row tile c / 3, term c % 3 (tiles past the last re-read it)
  const int mt_last = (a.M + 15) / 16 - 1;
  const wu32x4* ap[AR];
#pragma unroll
  for (int i = 0; i < AR; ++i) {
    const int c = wave * AR + i, mt = min(m0 / 16 + c / 3, mt_last);
    ap[i] = reinterpret_cast<const wu32x4*>(a.xa) + (static_cast<int64_t>(mt) * a.steps * 3 + c % 3) * 64 + lane;
  }
  const uint16_t *wp0[WR], *wp1[WR];
#pragma unroll
  for (int i = 0; i < WR; ++i) {
    const int j = wave * WR + i;  // the block's weight tile; the pair alternates gate and up tiles
    int n = (pair ? cb * (BN / 2) + (j >> 1) * 16 : cb * BN + j * 16) + lane % 16;
    n = min(n, a.N - 1);
    int seg = pair ? (j & 1) : 0, s0 = 0;
    if constexpr (!pair) {
      if (a.n_seg > 1 && n >= a.seg_start[1]) {
        seg = 1;
        s0 = a.seg_start[1];
      }
      if (a.n_seg > 2 && n >= a.seg_start[2]) {
        seg = 2;
        s0 = a.seg_start[2];
      }
    }
    const int64_t off = (n - s0) * a.ldw + 8 * (lane / 16);
    wp0[i] = (seg == 0 ? a.w[0][0] : seg == 1 ? a.w[1][0] : a.w[2][0]) + off;
    wp1[i] = (seg == 0 ? a.w[0][1] : seg == 1 ? a.w[1][1] : a.w[2][1]) + off;
  }

  // hi: the leading terms' sums since the last fold into tot; lo: the two
  // small terms' sums over all of K
  wf32x4 hi[TN][TM], lo[TN][TM], tot[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) hi[j][i] = lo[j][i] = tot[j][i] = wf32x4{0.f, 0.f, 0.f, 0.f};
  auto fold = [&]() {
    mfma_settle();
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const wf32x4 u = tot[j][i] + hi[j][i];
        lo[j][i] += hi[j][i] - (u - tot[j][i]);
        tot[j][i] = u;
        hi[j][i] = wf32x4{0.f, 0.f, 0.f, 0.f};
      }
  };
  const int wm = wave / WN, wn = wave % WN;
  const int stages = (a.steps + WK - 1) / WK;
  // stage st (past the last: the last again, so that every stage has the same loads in flight)
  auto fetch = [&](wu32x4* d, int st) {
    const int s = min(min(st, stages - 1) * WK + grp, a.steps - 1);
    d += grp * (ACH + WCH) * 64;
#pragma unroll
    for (int i = 0; i < AR; ++i) wd_load_lds(ap[i] + static_cast<int64_t>(s) * 192, d + (wave * AR + i) * 64);
    const bool first = s < a.steps0;
    const int64_t k = static_cast<int64_t>(first ? s : s - a.steps0) * 32;
#pragma unroll
    for (int i = 0; i < WR; ++i) wd_load_lds((first ? wp0[i] : wp1[i]) + k, d + (ACH + wave * WR + i) * 64);
  };
  auto multiply = [&](const wu32x4* d, int st) {
    if (WK > 1 && st * WK + grp >= a.steps) return;  // the last stage may hold fewer steps
    const uint32_t at = wd_lds_address(d) + (grp * (ACH + WCH) * 64 + lane) * 16;
    wu32x4 wf[TN];
    wd_read_lds<TN>(at + (ACH + wn * TN) * 1024, wf);
    constexpr int IG = TM % 2 == 0 && TM * TN < 16 ? 2 : 1;  // row tiles per read (what the registers hold)
#pragma unroll
    for (int i0 = 0; i0 < TM; i0 += IG) {
      wu32x4 xf[3 * IG];
      wd_read_lds<3 * IG>(at + (wm * TM + i0) * 3072, xf);
#pragma unroll
      for (int p = 2; p >= 0; --p)
#pragma unroll
        for (int i = 0; i < IG; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            wf32x4& c = p ? lo[j][i0 + i] : hi[j][i0 + i];
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(wbf16x8, wf[j]),
                                                        __builtin_bit_cast(wbf16x8, xf[3 * i + p]), c, 0, 0, 0);
          }
    }
  };
  // stage st has landed in cur for every wave, and every wave is done with the
  // stage before it, whose buffer takes stage st + NS - 1
  auto stage = [&](wu32x4* cur, wu32x4* prev, int st) {
    wd_stage_barrier<(NS - 2) * PL>();
    fetch(prev, st + NS - 1);
    multiply(cur, st);
  };
  fetch(s_0, 0);
  if constexpr (NS > 2) {
    fetch(s_1, 1);
    fetch(s_2, 2);
  }
  for (int st = 0; st < stages; st += NS) {
    if constexpr (NS == 2) {
      stage(s_0, s_1, st);
      if (st + 1 < stages) stage(s_1, s_0, st + 1);
    } else {
      stage(s_0, s_3, st);
      if (st + 1 < stages) stage(s_1, s_0, st + 1);
      if (st + 2 < stages) stage(s_2, s_1, st + 2);
      if (st + 3 < stages) stage(s_3, s_2, st + 3);
    }
    if ((st + NS) % kWideFlush == 0) fold();
  }
  wd_stage_barrier<0>();  // the loads past the last stage land before the buffers are used again
  mfma_settle();
  fold();
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) tot[j][i] += lo[j][i];

  if constexpr (WK > 1) {  // the groups' sums through LDS, added in group order
    float4* sum = reinterpret_cast<float4*>(s_0);
    __syncthreads();
    if (grp > 0) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
          sum[((grp - 1) * GW + wave) * TN * TM * 64 + (j * TM + i) * 64 + lane] =
              float4{tot[j][i][0], tot[j][i][1], tot[j][i][2], tot[j][i][3]};
    }
    __syncthreads();
    if (grp > 0) return;
#pragma unroll
    for (int g = 0; g < WK - 1; ++g)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const float4 v = sum[(g * GW + wave) * TN * TM * 64 + (j * TM + i) * 64 + lane];
          tot[j][i] += wf32x4{v.x, v.y, v.z, v.w};
        }
  }

  // lane: row l % 16 of its row tile, columns 4 (l / 16) .. + 3 of its weight tile
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + (wm * TM + i) * 16 + lane % 16;
    if constexpr (pair) {
      const int steps_out = a.N / 32;
#pragma unroll
      for (int j = 0; j < TN; j += 2) {
        const int n = cb * (BN / 2) + (wn * TN + j) / 2 * 16 + 4 * (lane / 16);
        if (m >= (a.M + 15) / 16 * 16 || n >= a.N) continue;  // whole row tiles: the next GEMM reads them
        uint32_t h[4], md[4], l[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float gv = tot[j][i][e], uv = tot[j + 1][i][e];
          wd_split1(m < a.M ? gv / (1.f + expf(-gv)) * uv : 0.f, h[e], md[e], l[e]);
        }
        auto pk = [](uint32_t u, uint32_t v) { return __builtin_amdgcn_perm(v, u, 0x07060302u); };
        uint16_t* dst = a.planes + wd_index(m, n, steps_out, 0);
        *reinterpret_cast<uint2*>(dst) = make_uint2(pk(h[0], h[1]), pk(h[2], h[3]));
        *reinterpret_cast<uint2*>(dst + 512) = make_uint2(pk(md[0], md[1]), pk(md[2], md[3]));
        *reinterpret_cast<uint2*>(dst + 1024) = make_uint2(pk(l[0], l[1]), pk(l[2], l[3]));
      }
    } else {
      if (m >= a.M) continue;
      const float* rp = nullptr;
      if constexpr (EPI == kWideResidual)
        rp = a.res + (a.res_row ? static_cast<int64_t>(a.res_row[m] + a.res_add) : m) * a.ldres;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = cb * BN + (wn * TN + j) * 16 + 4 * (lane / 16);
        if (n >= a.N) continue;  // N is a multiple of 8
        float4 v{tot[j][i][0], tot[j][i][1], tot[j][i][2], tot[j][i][3]};
        if constexpr (EPI == kWideResidual) {
          const float4 q = *reinterpret_cast<const float4*>(rp + n);
          v.x += q.x;
          v.y += q.y;
          v.z += q.z;
          v.w += q.w;
        }
        *reinterpret_cast<float4*>(a.y + m * a.ldy + n) = v;
      }
    }
  }
}

// ------------------------------------------------------------------ linear

// The same product straight from fp32 rows and row-major weights, for callers
// without a workspace for planes: a block splits what it stages.  Block tile BM
// x BN, WK groups of WM x WN waves on alternate k steps; two LDS buffers in
// fragment order, the next step's values in registers while the current one is
// multiplied.  fp32 weights (WF) are split as the rows are: six products per
// pair of fragments, everything down to 2^-24 of the leading one.  Sums as in
// k_wide_gemm.
struct WideLinArgs {
  const float* x;
  const void* w;
  int M, N, K;
  float* y;
  int accumulate;
  int vec;  // rows of y keep 16-byte vectors whole
};

template <int BM, int BN, int WM, int WN, int WK, int WPE, bool WF>
__global__ __launch_bounds__(WM* WN* WK* kWave) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void k_wide_linear(
    WideLinArgs a, int mblocks) {
  constexpr int GW = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16;
  constexpr int AR = BM / 16 / GW, WR = BN / 16 / GW, WP = WF ? 3 : 1;
  constexpr int ACH = BM / 16 * 3, WCH = BN / 16 * WP, SV = WK * (ACH + WCH) * 64;
  static_assert(AR * GW * 16 == BM && WR * GW * 16 == BN, "whole tiles per wave");
  static_assert(WK == 1 || (WK - 1) * BM * BN * 4 <= 2 * SV * 16, "the groups' sums fit the buffers");
  __shared__ wu32x4 s_buf[2 * SV];
  const int t = threadIdx.x, lane = t % kWave;
  const int wv = __builtin_amdgcn_readfirstlane(t / kWave), grp = wv / GW, wave = wv % GW;
  int blk;
  {
    const int nb = gridDim.x, q = nb / 8, r = nb % 8, x = blockIdx.x % 8, i = blockIdx.x / 8;
    blk = x < r ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
  }
  const int m0 = (blk % mblocks) * BM, n0 = blk / mblocks * BN;
  const int steps = a.K / 32, stages = (steps + WK - 1) / WK;
  const int wm = wave / WN, wn = wave % WN;

  // this lane's 8 values of a fragment: row l % 16, k 8 (l / 16) .. + 7 (rows past the last re-read it)
  const float* xp[AR];
#pragma unroll
  for (int i = 0; i < AR; ++i)
    xp[i] = a.x + static_cast<int64_t>(min(m0 + (wave * AR + i) * 16 + lane % 16, a.M - 1)) * a.K + 8 * (lane / 16);
  const char* wp[WR];
#pragma unroll
  for (int i = 0; i < WR; ++i)
    wp[i] = static_cast<const char*>(a.w) +
            (static_cast<int64_t>(min(n0 + (wave * WR + i) * 16 + lane % 16, a.N - 1)) * a.K + 8 * (lane / 16)) *
                (WF ? 4 : 2);
  wu32x4 rx[AR][2], rw[WR][WF ? 2 : 1];
  auto fetch = [&](int st) {
    const int64_t k = static_cast<int64_t>(min(st * WK + grp, steps - 1)) * 32;
#pragma unroll
    for (int i = 0; i < AR; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) rx[i][h] = *reinterpret_cast<const wu32x4*>(xp[i] + k + 4 * h);
#pragma unroll
    for (int i = 0; i < WR; ++i)
#pragma unroll
      for (int h = 0; h < (WF ? 2 : 1); ++h)
        rw[i][h] = *reinterpret_cast<const wu32x4*>(wp[i] + k * (WF ? 4 : 2) + 16 * h);
  };
  auto split = [&](const wu32x4* r, wu32x4* d) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = __uint_as_float(r[e / 4][e % 4]);
    uint4 h, m, l;
    wd_split8(v, h, m, l);
    d[0] = __builtin_bit_cast(wu32x4, h);
    d[64] = __builtin_bit_cast(wu32x4, m);
    d[128] = __builtin_bit_cast(wu32x4, l);
  };
  auto put = [&](int b) {
    wu32x4* d = s_buf + b * SV + grp * (ACH + WCH) * 64 + lane;
#pragma unroll
    for (int i = 0; i < AR; ++i) split(rx[i], d + (wave * AR + i) * 192);
#pragma unroll
    for (int i = 0; i < WR; ++i) {
      if constexpr (WF)
        split(rw[i], d + (ACH + (wave * WR + i) * 3) * 64);
      else
        d[(ACH + wave * WR + i) * 64] = rw[i][0];
    }
  };

  wf32x4 hi[TN][TM], lo[TN][TM], tot[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) hi[j][i] = lo[j][i] = tot[j][i] = wf32x4{0.f, 0.f, 0.f, 0.f};
  fetch(0);
  put(0);
  lds_barrier();
  for (int st = 0; st < stages; ++st) {
    if (st + 1 < stages) fetch(st + 1);
    if (WK == 1 || st * WK + grp < steps) {
      const wu32x4* d = s_buf + (st & 1) * SV + grp * (ACH + WCH) * 64 + lane;
      wbf16x8 wf[TN][WP];
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < WP; ++q) wf[j][q] = __builtin_bit_cast(wbf16x8, d[(ACH + (wn * TN + j) * WP + q) * 64]);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        wbf16x8 xf[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) xf[p] = __builtin_bit_cast(wbf16x8, d[((wm * TM + i) * 3 + p) * 64]);
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
          for (int q = (WP - 1 < 2 - p ? WP - 1 : 2 - p); q >= 0; --q)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
              wf32x4& c = p + q ? lo[j][i] : hi[j][i];
              c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j][q], xf[p], c, 0, 0, 0);
            }
      }
    }
    if ((st + 1) % kWideFlush == 0 || st + 1 == stages) {
      mfma_settle();
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const wf32x4 u = tot[j][i] + hi[j][i];
          lo[j][i] += hi[j][i] - (u - tot[j][i]);
          tot[j][i] = u;
          hi[j][i] = wf32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (st + 1 < stages) put((st + 1) & 1);
    lds_barrier();
  }
  mfma_settle();
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) tot[j][i] += lo[j][i];
  if constexpr (WK > 1) {
    float4* sum = reinterpret_cast<float4*>(s_buf);
    if (grp > 0) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
          sum[((grp - 1) * GW + wave) * TN * TM * 64 + (j * TM + i) * 64 + lane] =
              float4{tot[j][i][0], tot[j][i][1], tot[j][i][2], tot[j][i][3]};
    }
    __syncthreads();
    if (grp > 0) return;
#pragma unroll
    for (int g = 0; g < WK - 1; ++g)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const float4 v = sum[(g * GW + wave) * TN * TM * 64 + (j * TM + i) * 64 + lane];
          tot[j][i] += wf32x4{v.x, v.y, v.z, v.w};
        }
  }

  // An infinite input meets zero terms of the other operand, which leaves NaN
  // where the product is infinite: a wave with such a sum takes plain fp32 sums
  // of its tile instead.
  bool odd = false;
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) odd = odd || !(fabsf(tot[j][i][e]) <= 3.402823466e38f);
  if (__ballot(odd) != 0) {
    for (int c = lane; c < TM * 16 * TN * 16; c += kWave) {
      const int m = m0 + wm * TM * 16 + c / (TN * 16), n = n0 + wn * TN * 16 + c % (TN * 16);
      if (m >= a.M || n >= a.N) continue;
      const float* xr = a.x + static_cast<int64_t>(m) * a.K;
      float v = 0.f;
      for (int k = 0; k < a.K; ++k) {
        const int64_t at = static_cast<int64_t>(n) * a.K + k;
        v = fmaf(xr[k], WF ? static_cast<const float*>(a.w)[at] : bf16_to_float(static_cast<const uint16_t*>(a.w)[at]), v);
      }
      float* yp = a.y + static_cast<int64_t>(m) * a.N + n;
      *yp = a.accumulate ? *yp + v : v;
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + (wm * TM + i) * 16 + lane % 16;
    if (m >= a.M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + (wn * TN + j) * 16 + 4 * (lane / 16);
      float* yp = a.y + static_cast<int64_t>(m) * a.N + n;
      if (a.vec && n < a.N) {
        float4 v{tot[j][i][0], tot[j][i][1], tot[j][i][2], tot[j][i][3]};
        if (a.accumulate) {
          const float4 q = *reinterpret_cast<const float4*>(yp);
          v.x += q.x;
          v.y += q.y;
          v.z += q.z;
          v.w += q.w;
        }
        *reinterpret_cast<float4*>(yp) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < a.N) yp[e] = a.accumulate ? yp[e] + tot[j][i][e] : tot[j][i][e];
      }
    }
  }
}

// ------------------------------------------------------------------ q / k norm, RoPE, append

// One wave per head vector of 128: lane j holds dims j and j + 64, a RoPE pair.
template <typename KT>
__global__ __launch_bounds__(256) void k_wide_qkv(WideQkvArgs a) {
  constexpr int D = 128;
  const int lane = threadIdx.x % kWave, h = blockIdx.y * 4 + threadIdx.x / kWave, r = blockIdx.x;
  const int nh = a.H + 2 * a.Hk;
  if (h >= nh) return;
  const float* src = a.qkv + (static_cast<int64_t>(r) * nh + h) * D;
  float x1 = src[lane], x2 = src[lane + 64];
  const int offset = *a.offset_dev + a.offset_add, slot = offset + r;
  if (h < a.H + a.Hk) {
    const uint16_t* g = h < a.H ? a.q_gain : a.k_gain;
    const float g1 = bf16_to_float(g[lane]), g2 = bf16_to_float(g[lane + 64]);
    const int pos = min(max(a.positions ? a.positions[r] : slot, 0), a.rope_max - 1);
    const float c = a.rope_cos[static_cast<int64_t>(pos) * 64 + lane], s = a.rope_sin[static_cast<int64_t>(pos) * 64 + lane];
    const float ss = wave_sum_dpp(fmaf(x2, x2, x1 * x1));
    const float inv = 1.f / sqrtf(ss / static_cast<float>(D) + a.eps);
    const float u = x1 * inv * g1, v = x2 * inv * g2;
    x1 = u * c - v * s;
    x2 = v * c + u * s;
    if (h < a.H) {
      float* q = a.q + (static_cast<int64_t>(r) * a.H + h) * D;
      q[lane] = x1;
      q[lane + 64] = x2;
      return;
    }
  }
  if (slot < 0 || slot >= a.cap) return;
  const bool is_k = h < a.H + a.Hk;
  KT* dst = static_cast<KT*>(is_k ? a.kc : a.vc) + (static_cast<int64_t>(is_k ? h - a.H : h - a.H - a.Hk) * a.cap + slot) * D;
  if constexpr (sizeof(KT) == 2) {
    dst[lane] = float_to_bf16(x1);
    dst[lane + 64] = float_to_bf16(x2);
  } else {
    dst[lane] = x1;
    dst[lane + 64] = x2;
  }
}

// out = RMSNorm(x) per row, one block each (a pass's final norm)
__global__ __launch_bounds__(256) void k_wide_norm(const float* __restrict__ x, float* __restrict__ y, int K,
                                                   const uint16_t* __restrict__ gain, float eps) {
  __shared__ float red[4];
  const float* xr = x + static_cast<int64_t>(blockIdx.x) * K;
  float* yr = y + static_cast<int64_t>(blockIdx.x) * K;
  float ss = 0.f;
  for (int k = threadIdx.x * 4; k < K; k += 1024) {
    const float4 v = *reinterpret_cast<const float4*>(xr + k);
    ss = fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, ss))));
  }
  ss = wave_sum_dpp(ss);
  if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = ss;
  __syncthreads();
  const float inv = 1.f / sqrtf((red[0] + red[1] + red[2] + red[3]) / static_cast<float>(K) + eps);
  for (int k = threadIdx.x * 4; k < K; k += 1024) {
    const float4 v = *reinterpret_cast<const float4*>(xr + k);
    const uint2 g = *reinterpret_cast<const uint2*>(gain + k);
    *reinterpret_cast<float4*>(yr + k) = float4{v.x * bf16_lo(g.x) * inv, v.y * bf16_hi(g.x) * inv,
                                                v.z * bf16_lo(g.y) * inv, v.w * bf16_hi(g.y) * inv};
  }
}

// ------------------------------------------------------------------ many-row attention

// Flash attention over 64 query vectors per block (rows x GQA group of one kv
// head, 16 per wave) and chunks of CH keys.  KP = 1: bf16 keys / values; KP =
// 3: fp32 ones, split into three terms as they are staged.  S^T = K Q^T puts
// one query vector in each lane (keys 16 kt + 4 g + e), so P^T feeds O^T = V^T
// P^T from the registers with V^T read by transposing LDS reads.  Every product
// keeps the terms down to 2^-24 of the leading one: 3 MFMAs per tile for KP =
// 1, 6 for KP = 3.
template <int KP, int CH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_wide_attn(WideAttnArgs a) {
  constexpr int D = 128, LDK = D + 8, LDV = D + 16, KT = CH / 16, NL = CH / 16;
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  __shared__ __attribute__((aligned(16))) uint16_t s_k[KP][CH * LDK], s_v[KP][CH * LDV];
  const int kh = blockIdx.y, z = gridDim.x - 1 - blockIdx.x;  // the longest key ranges first
  const int rep = a.H / a.Hk, QV = a.rows * rep;
  const int t = threadIdx.x, lane = t % kWave, wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int kl = lane % 16, gq = lane / 16, dg = gq * 8;
  const int vq = z * 64 + wave * 16 + kl, vqc = min(vq, QV - 1), row = vqc / rep;
  const float* qsrc = a.q + static_cast<int64_t>(row) * a.ld_q + (kh * rep + vqc % rep) * D + dg;

  // key range of the block: causal limits from its first and last rows
  const int r0 = min(z * 64, QV - 1) / rep, r1 = min(z * 64 + 63, QV - 1) / rep;
  const bool causal = a.mask == nullptr && a.offset_dev != nullptr;
  const int offset = causal ? *a.offset_dev + a.offset_add : 0;
  int kb = 0, ke = a.keys;
  if (causal) {
    ke = min(ke, offset + r1 + 1);
    if (a.window > 0) kb = max(0, offset + r0 - a.window + 1) / CH * CH;
  }
  const int S = gridDim.z, split = blockIdx.z;
  if (S > 1 && ke > kb) {  // whole chunks per split
    const int per = ((ke - kb + S - 1) / S + CH - 1) / CH * CH;
    kb += split * per;
    ke = min(ke, kb + per);
  }
  const int lim = causal ? offset + row : 0x3fffffff;
  const int wlo = causal && a.window > 0 ? offset + row - a.window : -1;

  wbf16x8 qf[4][3];
#pragma unroll
  for (int st = 0; st < 4; ++st) {
    const float4 u = *reinterpret_cast<const float4*>(qsrc + st * 32), w = *reinterpret_cast<const float4*>(qsrc + st * 32 + 4);
    const float sc = a.scale * 1.4426950408889634f;
    const float x[8] = {u.x * sc, u.y * sc, u.z * sc, u.w * sc, w.x * sc, w.y * sc, w.z * sc, w.w * sc};
    uint4 h, m, l;
    wd_split8(x, h, m, l);
    qf[st][0] = __builtin_bit_cast(wbf16x8, h);
    qf[st][1] = __builtin_bit_cast(wbf16x8, m);
    qf[st][2] = __builtin_bit_cast(wbf16x8, l);
  }

  // chunk loads: thread t holds 8 dims 8 (t % 16) .. of keys t / 16 + 16 i (rows past the last re-read it)
  constexpr int RV = KP == 1 ? 1 : 2;  // 16-byte vectors per 8 dims
  wu32x4 rk[NL][RV], rv[NL][RV];
  constexpr int ES = KP == 1 ? 2 : 4;
  const char* kbase = static_cast<const char*>(a.k) + (kh * a.ld_head + (t % 16) * 8) * ES;
  const char* vbase = static_cast<const char*>(a.v) + (kh * a.ld_head + (t % 16) * 8) * ES;
  auto fetch = [&](int c0) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int64_t at = static_cast<int64_t>(min(c0 + t / 16 + 16 * i, a.keys - 1)) * a.ld_key * ES;
#pragma unroll
      for (int x = 0; x < RV; ++x) {
        rk[i][x] = *reinterpret_cast<const wu32x4*>(kbase + at + 16 * x);
        rv[i][x] = *reinterpret_cast<const wu32x4*>(vbase + at + 16 * x);
      }
    }
  };
  auto put = [&](const wu32x4* r, bool live, uint16_t* p0, int plane) {
    if constexpr (KP == 1) {
      *reinterpret_cast<wu32x4*>(p0) = live ? r[0] : wu32x4{0, 0, 0, 0};
    } else {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = live ? __uint_as_float(r[e / 4][e % 4]) : 0.f;
      uint4 h, m, l;
      wd_split8(x, h, m, l);
      *reinterpret_cast<uint4*>(p0) = h;
      *reinterpret_cast<uint4*>(p0 + plane) = m;
      *reinterpret_cast<uint4*>(p0 + 2 * plane) = l;
    }
  };

  float m_r = -INFINITY;
  double l_r = 0.0;
  wf32x4 o[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) o[dt] = wf32x4{0.f, 0.f, 0.f, 0.f};
  const int vr0 = 4 * gq + kl / 4, vc0 = 4 * (kl % 4);
  // the mask bytes of the lane's keys, four to a word: one load where the rows keep words whole
  const uint8_t* mrow = a.mask ? a.mask + row * a.mask_ld : nullptr;
  const bool mvec = a.mask_ld % 4 == 0 && a.keys % 4 == 0 && (reinterpret_cast<uintptr_t>(a.mask) & 3) == 0;
  uint32_t mk[KT];
  auto fetch_mask = [&](int c0) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      const int key = c0 + kt * 16 + 4 * gq;
      if (mvec) {
        mk[kt] = *reinterpret_cast<const uint32_t*>(mrow + min(key, a.keys - 4));
      } else {
        mk[kt] = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) mk[kt] |= static_cast<uint32_t>(mrow[min(key + e, a.keys - 1)]) << (8 * e);
      }
    }
  };

  if (kb < ke) {
    fetch(kb);
    if (mrow) fetch_mask(kb);
  }
  for (int c0 = kb; c0 < ke; c0 += CH) {
    const int n = min(CH, ke - c0);
    lds_barrier();
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int key = t / 16 + 16 * i;
      // rows past the range: zeros (what lies there may be anything, and P is 0 for them)
      put(rk[i], key < n, &s_k[0][key * LDK + (t % 16) * 8], CH * LDK);
      put(rv[i], key < n, &s_v[0][key * LDV + (t % 16) * 8], CH * LDV);
    }
    lds_barrier();
    // bit 4 kt + e: key c0 + 16 kt + 4 g + e is visible to the lane's row
    uint32_t vis = 0;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = kt * 16 + 4 * gq + e, key = c0 + j;
        const bool on = mrow ? (mk[kt] >> (8 * e) & 0xffu) != 0 : key <= lim && key > wlo;
        vis |= (j < n && on ? 1u : 0u) << (4 * kt + e);
      }
    if (c0 + CH < ke) {
      fetch(c0 + CH);
      if (mrow) fetch_mask(c0 + CH);
    }
    if (__ballot(vis != 0) == 0) continue;  // nothing for the wave's rows in this chunk

    wf32x4 sacc[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) sacc[kt] = wf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
      for (int kp = KP - 1; kp >= 0; --kp) {
        wbf16x8 kf[KT];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
          kf[kt] = __builtin_bit_cast(wbf16x8, *reinterpret_cast<const wu32x4*>(&s_k[kp][(kt * 16 + kl) * LDK + st * 32 + dg]));
#pragma unroll
        for (int qp = 2 - kp; qp >= 0; --qp)
#pragma unroll
          for (int kt = 0; kt < KT; ++kt)
            sacc[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kt], qf[st][qp], sacc[kt], 0, 0, 0);
      }
    mfma_settle();
    float mx = -INFINITY;
    float sv[KT][4];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sv[kt][e] = vis >> (4 * kt + e) & 1u ? sacc[kt][e] : -INFINITY;
        mx = fmaxf(mx, sv[kt][e]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m_r, mx);
    const float mb = m_new == -INFINITY ? 0.f : m_new;  // nothing visible yet: exp2(-inf) = 0 below
    const float alpha = __builtin_amdgcn_exp2f(m_r - mb);
    float p[KT][4], rs = 0.f;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p[kt][e] = __builtin_amdgcn_exp2f(sv[kt][e] - mb);
        rs += p[kt][e];
      }
    l_r = l_r * alpha + rs;  // this lane's keys; the row's four lanes are added at the end
    m_r = m_new;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int e = 0; e < 4; ++e) o[dt][e] *= alpha;
#pragma unroll
    for (int kk = 0; kk < CH / 32; ++kk) {
      const float px[8] = {p[2 * kk][0], p[2 * kk][1], p[2 * kk][2], p[2 * kk][3],
                           p[2 * kk + 1][0], p[2 * kk + 1][1], p[2 * kk + 1][2], p[2 * kk + 1][3]};
      uint4 ph[3];
      wd_split8(px, ph[0], ph[1], ph[2]);
#pragma unroll
      for (int vp = KP - 1; vp >= 0; --vp) {
        wbf16x8 vf[8];
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
          uint16_t* src = &s_v[vp][(kk * 32 + vr0) * LDV + dt * 16 + vc0];
          const s16x4 a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(src));
          const s16x4 a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(src + 16 * LDV));
          vf[dt] = __builtin_bit_cast(wbf16x8, s16x8{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]});
        }
#pragma unroll
        for (int pp = 2 - vp; pp >= 0; --pp)
#pragma unroll
          for (int dt = 0; dt < 8; ++dt)
            o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt], __builtin_bit_cast(wbf16x8, ph[pp]), o[dt], 0, 0, 0);
      }
    }
  }
  mfma_settle();
  l_r += __shfl_xor(l_r, 16);
  l_r += __shfl_xor(l_r, 32);
  if (vq >= QV) return;
  const float l = static_cast<float>(l_r);
  if (S > 1) {  // (m, l) and the unnormalised output of this split, for k_wide_merge
    float* part = a.partial + ((static_cast<int64_t>(kh) * S + split) * QV + vq) * (D + 2);
    if (gq == 0) {
      part[0] = m_r;
      part[1] = l;
    }
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      float2* pp = reinterpret_cast<float2*>(part + 2 + dt * 16 + 4 * gq);
      pp[0] = make_float2(o[dt][0], o[dt][1]);
      pp[1] = make_float2(o[dt][2], o[dt][3]);
    }
    return;
  }
  const int h = kh * rep + vq % rep;
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) {
    const float y[4] = {o[dt][0] / l, o[dt][1] / l, o[dt][2] / l, o[dt][3] / l};
    const int k = h * D + dt * 16 + 4 * gq;
    if (a.out) *reinterpret_cast<float4*>(a.out + static_cast<int64_t>(row) * a.H * D + k) = float4{y[0], y[1], y[2], y[3]};
    if (a.planes) {
      uint32_t hb[4], mb[4], lb[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) wd_split1(y[e], hb[e], mb[e], lb[e]);
      auto pk = [](uint32_t u, uint32_t v) { return __builtin_amdgcn_perm(v, u, 0x07060302u); };
      uint16_t* dst = a.planes + wd_index(row, k, a.H * D / 32, 0);
      *reinterpret_cast<uint2*>(dst) = make_uint2(pk(hb[0], hb[1]), pk(hb[2], hb[3]));
      *reinterpret_cast<uint2*>(dst + 512) = make_uint2(pk(mb[0], mb[1]), pk(mb[2], mb[3]));
      *reinterpret_cast<uint2*>(dst + 1024) = make_uint2(pk(lb[0], lb[1]), pk(lb[2], lb[3]));
    }
  }
}

// The splits of one query vector (block x) of a kv head (block y), thread =
// output dim; m in base 2.
__global__ __launch_bounds__(128) void k_wide_merge(WideAttnArgs a, int S) {
  constexpr int D = 128;
  const int v = blockIdx.x, kh = blockIdx.y, t = threadIdx.x, rep = a.H / a.Hk, QV = a.rows * rep;
  const float* part = a.partial + (static_cast<int64_t>(kh) * S * QV + v) * (D + 2);
  const int64_t ld = static_cast<int64_t>(QV) * (D + 2);
  float M = -INFINITY;
  for (int s = 0; s < S; ++s) M = fmaxf(M, part[s * ld]);
  float l = 0.f, o = 0.f;
#pragma unroll 8
  for (int s = 0; s < S; ++s) {
    const float m = part[s * ld], w = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - M);
    l = fmaf(part[s * ld + 1], w, l);
    o = fmaf(part[s * ld + 2 + t], w, o);
  }
  const float y = o / l;
  const int row = v / rep, k = (kh * rep + v % rep) * D + t;
  if (a.out) a.out[static_cast<int64_t>(row) * a.H * D + k] = y;
  if (a.planes) {
    uint32_t h, m, lo;
    wd_split1(y, h, m, lo);
    uint16_t* dst = a.planes + wd_index(row, k, a.H * D / 32, 0);
    dst[0] = static_cast<uint16_t>(h >> 16);
    dst[512] = static_cast<uint16_t>(m >> 16);
    dst[1024] = static_cast<uint16_t>(lo >> 16);
  }
}

// ------------------------------------------------------------------ launchers

__global__ void k_wide_advance(int32_t* dst, const int32_t* src, int add) { *dst = *src + add; }

int launch_wide_prep(const WidePrepArgs& a, hipStream_t s) {
  const unsigned tiles = static_cast<unsigned>((a.M + 15) / 16);
  // enough blocks for the CUs: every part re-reads its rows for the norm, so no more than that
  const unsigned parts = std::max(1u, std::min(8u, 512 / (tiles * a.n_seg)));
  hipLaunchKernelGGL(k_wide_prep, dim3(tiles, parts, a.n_seg), dim3(kWidePrepThreads), 0, s, a);
  WC_LAUNCHED();
  return WC_OK;
}

template <int BM, int BN, int WM, int WN, int WK, int NS, int WPE>
static void wide_gemm_t(const WideArgs& a, int epi, hipStream_t s) {
  const int mb = (a.M + BM - 1) / BM, cols = epi == kWideSiluPair ? BN / 2 : BN, nb = (a.N + cols - 1) / cols;
  const dim3 grid(mb * nb), block(WM * WN * WK * kWave);
  if (epi == kWideStore)
    hipLaunchKernelGGL((k_wide_gemm<BM, BN, WM, WN, WK, NS, WPE, kWideStore>), grid, block, 0, s, a, mb);
  else if (epi == kWideResidual)
    hipLaunchKernelGGL((k_wide_gemm<BM, BN, WM, WN, WK, NS, WPE, kWideResidual>), grid, block, 0, s, a, mb);
  else
    hipLaunchKernelGGL((k_wide_gemm<BM, BN, WM, WN, WK, NS, WPE, kWideSiluPair>), grid, block, 0, s, a, mb);
}

// Tile choice: the least steps x rounds x (time of a k step of one block), a
// round being one block per CU.  Step times in us, measured over the
// projections of the Qwen3-1.7B and -4B drafters at 24..1024 rows (one round /
// several): a small tile costs less per step, a large one covers more of the
// output per round.  Against 128 x 128 for everything (us, the 1.7B / 4B fuse):
// 24 rows 150 -> 23 / 209 -> 42 (32 x 32), 160 rows 154 -> 36 / 211 -> 53 (32 x
// 64), 333 rows 155 -> 50 / 211 -> 66 (64 x 64), 1024 rows 169 -> 99 (64 x 128) /
// 221 -> 175 (128 x 128 with eight waves); its own four-wave form, two blocks
// per CU, stays the best above one round (1024 rows of the 4B gate / up pair:
// 298 against 329 us, 1.0 PFLOP/s of MFMA work).
struct WideTile {
  int bm, bn;
  float one, more;
};
constexpr WideTile kWideTiles[] = {{32, 32, .165f, .165f}, {32, 64, .215f, .215f}, {64, 64, .28f, .28f},
                                   {64, 128, .48f, .48f},  {128, 128, .64f, .79f}, {128, 128, .80f, .70f}};

int launch_wide_gemm(const WideArgs& a, int epi, hipStream_t s) {
  int cus = 0;
  if (int rc = device_cus(&cus)) return rc;
  int best = 0;
  float best_t = 0.f;
  for (int i = 0; i < 6; ++i) {
    const WideTile& t = kWideTiles[i];
    const int bn = epi == kWideSiluPair ? t.bn / 2 : t.bn;
    const int blocks = (a.M + t.bm - 1) / t.bm * ((a.N + bn - 1) / bn), rounds = (blocks + cus - 1) / cus;
    const float us = rounds > 1 ? rounds * t.more : t.one;
    if (i == 0 || us < best_t) {
      best = i;
      best_t = us;
    }
  }
  switch (best) {
    case 0: wide_gemm_t<32, 32, 2, 1, 4, 4, 2>(a, epi, s); break;
    case 1: wide_gemm_t<32, 64, 2, 1, 2, 4, 2>(a, epi, s); break;
    case 2: wide_gemm_t<64, 64, 2, 2, 2, 4, 2>(a, epi, s); break;
    case 3: wide_gemm_t<64, 128, 2, 2, 1, 4, 2>(a, epi, s); break;
    case 4: wide_gemm_t<128, 128, 4, 2, 1, 4, 2>(a, epi, s); break;
    default: wide_gemm_t<128, 128, 2, 2, 1, 2, 2>(a, epi, s); break;
  }
  WC_LAUNCHED();
  return WC_OK;
}

template <int BM, int BN, int WM, int WN, int WK, int WPE>
static void wide_linear_t(const WideLinArgs& a, bool wf, hipStream_t s) {
  const int mb = (a.M + BM - 1) / BM, nb = (a.N + BN - 1) / BN;
  const dim3 grid(mb * nb), block(WM * WN * WK * kWave);
  if (wf)
    hipLaunchKernelGGL((k_wide_linear<BM, BN, WM, WN, WK, WPE, true>), grid, block, 0, s, a, mb);
  else
    hipLaunchKernelGGL((k_wide_linear<BM, BN, WM, WN, WK, WPE, false>), grid, block, 0, s, a, mb);
}

int launch_wide_linear(const float* x, int L, int in, const void* W, int w_dtype, int out, float* y, int accumulate,
                       hipStream_t s) {
  int cus = 0;
  if (int rc = device_cus(&cus)) return rc;
  const WideLinArgs a{x, W, L, out, in, y, accumulate, out % 4 == 0 && aligned(y, 16)};
  const bool wf = w_dtype == WC_F32;
  // as launch_wide_gemm: the least rounds x step time, bf16 / fp32 weights (us,
  // in 2048: 16 rows 2048 outputs 17 / 24 with 32 x 32, 160 rows 23 / 36 with 32 x
  // 64, 384 rows 36 / 53 with 64 x 64, 384 rows 6144 outputs 69 / 110 with 64 x
  // 128; 128 x 128 was never the best)
  constexpr WideTile kTiles[2][4] = {
      {{32, 32, .26f, .265f}, {32, 64, .34f, .345f}, {64, 64, .54f, .555f}, {64, 128, .80f, .54f}},
      {{32, 32, .38f, .386f}, {32, 64, .53f, .53f}, {64, 64, .78f, .78f}, {64, 128, 1.25f, .86f}}};
  int best = 0;
  float best_t = 0.f;
  for (int i = 0; i < 4; ++i) {
    const WideTile& t = kTiles[wf][i];
    const int64_t blocks = static_cast<int64_t>((L + t.bm - 1) / t.bm) * ((out + t.bn - 1) / t.bn);
    const int64_t rounds = (blocks + cus - 1) / cus;
    const float us = rounds > 1 ? rounds * t.more : t.one;
    if (i == 0 || us < best_t) {
      best = i;
      best_t = us;
    }
  }
  switch (best) {
    case 0: wide_linear_t<32, 32, 2, 1, 4, 2>(a, wf, s); break;
    case 1: wide_linear_t<32, 64, 2, 1, 4, 2>(a, wf, s); break;
    case 2: wide_linear_t<64, 64, 2, 2, 2, 2>(a, wf, s); break;
    default: wide_linear_t<64, 128, 2, 2, 1, 2>(a, wf, s); break;
  }
  WC_LAUNCHED();
  return WC_OK;
}

int launch_wide_qkv(const WideQkvArgs& a, int kv_dtype, hipStream_t s) {
  const dim3 grid(a.rows, (a.H + 2 * a.Hk + 3) / 4);
  if (kv_dtype == WC_BF16)
    hipLaunchKernelGGL(k_wide_qkv<uint16_t>, grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(k_wide_qkv<float>, grid, dim3(256), 0, s, a);
  WC_LAUNCHED();
  return WC_OK;
}

int launch_wide_norm(const float* x, float* y, int rows, int K, const uint16_t* gain, float eps, hipStream_t s) {
  hipLaunchKernelGGL(k_wide_norm, dim3(rows), dim3(256), 0, s, x, y, K, gain, eps);
  WC_LAUNCHED();
  return WC_OK;
}

int launch_wide_advance(int32_t* dst, const int32_t* src, int add, hipStream_t s) {
  hipLaunchKernelGGL(k_wide_advance, dim3(1), dim3(1), 0, s, dst, src, add);
  WC_LAUNCHED();
  return WC_OK;
}

int launch_wide_attn(const WideAttnArgs& a, int kv_dtype, hipStream_t s) {
  const int qv = a.rows * (a.H / a.Hk), groups = (qv + 63) / 64;
  // One block walks its keys chunk by chunk (~1.5 us each), so a grid that
  // leaves CUs idle splits them, down to two chunks each.
  int splits = 1;
  if (a.partial) {
    const int chunk = kv_dtype == WC_BF16 ? 64 : 32;
    const size_t fit = a.partial_floats / (static_cast<size_t>(a.Hk) * qv * 130);
    splits = std::min(256 / (groups * a.Hk), a.keys / (2 * chunk));
    splits = std::max(1, std::min(std::min(splits, 32), static_cast<int>(std::min<size_t>(fit, 32))));
  }
  const dim3 grid(groups, a.Hk, splits);
  if (kv_dtype == WC_BF16)
    hipLaunchKernelGGL((k_wide_attn<1, 64>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((k_wide_attn<3, 32>), grid, dim3(256), 0, s, a);
  WC_LAUNCHED();
  if (splits > 1) {
    hipLaunchKernelGGL(k_wide_merge, dim3(qv, a.Hk), dim3(128), 0, s, a, splits);
    WC_LAUNCHED();
  }
  return WC_OK;
}

}  // namespace wc
