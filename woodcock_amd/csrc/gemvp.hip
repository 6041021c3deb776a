// gemvp.hip -- the gate / up pair of 2..16 input rows on the matrix cores, one
// block per CU with every weight of the block in flight.
//
//   y[m][n] = SiLU(g) * u,  (g, u) = inv[m] * sum_k (gate, up)[n][k] * (x[m][k] * gain[k])
//
// What bounds it: the two matrices' bytes (50 MB for a 2048 x 6144 pair).  A
// half tile is 8 features: rows 0..7 of the A operand of
// v_mfma_f32_16x16x32_bf16 are their gate rows, rows 8..15 their up rows, so a
// block's work comes in 8-feature steps and the matrices divide evenly over the
// CUs (16-feature blocks left half of the CUs with twice the others' work: 384
// blocks for 6144 features, and the launch lasted as long as those CUs took).
// Wave w of eight owns a contiguous eighth of the k steps for all of the
// block's NT half tiles: it requests its own slice of the M input rows and of
// the gain, then the weights of up to SL half tiles at once, and splits
// x * gain into three bf16 terms (exact to ~2^-25) while the weights arrive;
// the terms stay in registers for every half tile.  Nothing is staged and no
// barrier is met before the partial tiles are summed in wave order in LDS.
// At 5 rows of a 2048 x 6144 pair: 13.4 us (3.7 TB/s), against 15.2 us on
// 16-feature blocks of four waves (k_gemvf); sixteen waves here: 15.9 us.
#include "gemv.h"

namespace wc {

typedef __bf16 gpbf16x8 __attribute__((ext_vector_type(8)));
typedef float gpf32x4 __attribute__((ext_vector_type(4)));

constexpr int kGpWaves = 8;
constexpr int kGpMaxTiles = 5;  // half tiles per block, at most

// 8 fp32 -> three bf16 terms, each the rounding of what the previous ones left
__device__ __forceinline__ void gp_split3(const float* x, gpbf16x8 (&p)[3]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const __bf16 hi = static_cast<__bf16>(x[e]);
    const float r1 = x[e] - static_cast<float>(hi);
    const __bf16 mid = static_cast<__bf16>(r1);
    p[0][e] = hi;
    p[1][e] = mid;
    p[2][e] = static_cast<__bf16>(r1 - static_cast<float>(mid));
  }
}

// PER: k steps of a wave, at least K / 32 / 8 (steps past a wave's share read
// its last step's addresses and count as zeros).
template <int NT, int PER, bool FRAG>
__global__ __launch_bounds__(kGpWaves * kWave) void k_gemv_pair(GemvArgs a) {
  constexpr int SL = PER > 8 || (PER > 4 && NT > 3) ? (NT < 2 ? NT : 2) : (NT < 3 ? NT : 3);  // half tiles in flight
  __shared__ float s_c[kGpWaves][NT][4][kWave];
  __shared__ float s_ss[kGpWaves][kWave];
  __shared__ float s_inv[16];
  const int t = threadIdx.x, lane = t % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int lm = lane % 16, kg = lane / 16;
  const int K = a.in[0].K, S = K / 32, per = (S + kGpWaves - 1) / kGpWaves;
  const int i0 = min(S, wave * per), i1 = min(S, i0 + per), ilast = max(i1 - 1, 0);
  const int tiles = (a.N + 7) / 8, h0 = blockIdx.x * NT;

  // the wave's slice of the input rows (columns past the launch's rows repeat
  // the last one and are never read back) and of the gain
  const float* xr = static_cast<const float*>(a.in[0].x) +
                    static_cast<int64_t>(in_row(a.in[0], min(lm, a.M - 1))) * a.in[0].ld + kg * 8;
  const uint16_t* gr = a.in[0].gain + kg * 8;
  float4 xa[PER], xb[PER];
  uint4 gn[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int k = min(i0 + u, ilast) * 32;
    xa[u] = *reinterpret_cast<const float4*>(xr + k);
    xb[u] = *reinterpret_cast<const float4*>(xr + k + 4);
    gn[u] = *reinterpret_cast<const uint4*>(gr + k);
  }
  // lane l of half tile h: gate (l % 16 < 8) or up row 8 h + l % 8 at k group l / 16
  const uint16_t* wbase = lm < 8 ? a.w[0][0] : a.w[1][0];
  uint4 w[SL][PER];
  auto issue = [&](int slot, int j) {
    const int h = min(h0 + j, tiles - 1);
    const uint16_t* p;
    if constexpr (FRAG)
      p = wbase + (static_cast<int64_t>(h / 2) * S * 64 + (h % 2) * 8 + lm % 8 + 16 * kg) * 8;
    else
      p = wbase + static_cast<int64_t>(min(8 * h + lm % 8, a.N - 1)) * a.ldw[0] + kg * 8;
#pragma unroll
    for (int u = 0; u < PER; ++u)
      w[slot][u] = *reinterpret_cast<const uint4*>(p + static_cast<int64_t>(min(i0 + u, ilast)) * (FRAG ? 512 : 32));
  };
#pragma unroll
  for (int j = 0; j < SL; ++j) issue(j, j);
  const int m_live = a.m_dev ? min(max(*a.m_dev, 0), a.M) : a.M;

  gpbf16x8 xs[PER][3];
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const bool on = i0 + u < i1;
    float x[8] = {xa[u].x, xa[u].y, xa[u].z, xa[u].w, xb[u].x, xb[u].y, xb[u].z, xb[u].w};
    const float g[8] = {bf16_lo(gn[u].x), bf16_hi(gn[u].x), bf16_lo(gn[u].y), bf16_hi(gn[u].y),
                        bf16_lo(gn[u].z), bf16_hi(gn[u].z), bf16_lo(gn[u].w), bf16_hi(gn[u].w)};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[e] = on ? x[e] : 0.f;
      ss = fmaf(x[e], x[e], ss);
      x[e] = on ? x[e] * g[e] : 0.f;
    }
    gp_split3(x, xs[u]);
  }
  s_ss[wave][lane] = ss;

  // the leading terms and the two small ones in chains of their own: fewer
  // roundings at the sum's size, and two chains in flight
  gpf32x4 acc[NT], acl[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    acc[j] = acl[j] = gpf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      // a repeated step: zero weights too (an infinite one times the zero input would be NaN)
      const uint32_t on = i0 + u < i1 ? 0xffffffffu : 0u;
      uint4 q = w[j % SL][u];
      q = make_uint4(q.x & on, q.y & on, q.z & on, q.w & on);
      const gpbf16x8 qb = __builtin_bit_cast(gpbf16x8, q);
      acl[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qb, xs[u][2], acl[j], 0, 0, 0);
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qb, xs[u][0], acc[j], 0, 0, 0);
      acl[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qb, xs[u][1], acl[j], 0, 0, 0);
    }
    if (j + SL < NT) issue(j % SL, j + SL);
  }
  mfma_settle();
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) s_c[wave][j][e][lane] = acc[j][e] + acl[j][e];
  __syncthreads();
  if (t < 16) {
    float tot = 0.f;
#pragma unroll
    for (int v = 0; v < kGpWaves; ++v)
#pragma unroll
      for (int q = 0; q < 4; ++q) tot += s_ss[v][q * 16 + t];
    s_inv[t] = 1.f / sqrtf(tot / static_cast<float>(K) + a.eps);
  }
  __syncthreads();
  // outputs (feature r of the block, input row m), features fastest: tile row
  // i, column m is element i % 4 of lane 16 (i / 4) + m
  for (int idx = t; idx < NT * 8 * a.M; idx += kGpWaves * kWave) {
    const int r = idx % (NT * 8), m = idx / (NT * 8), n = h0 * 8 + r;
    if (m >= m_live || n >= a.N) continue;
    const int j = r / 8, i = r % 8, cl = (i / 4) * 16 + m, ce = i % 4;
    float g = 0.f, u = 0.f;
#pragma unroll
    for (int v = 0; v < kGpWaves; ++v) {
      g += s_c[v][j][ce][cl];
      u += s_c[v][j][ce][cl + 32];
    }
    store_out<true>(a, m, n, g * s_inv[m], u * s_inv[m], 0.f);
  }
  if (a.adv_dst && blockIdx.x == 0 && t == 0) *a.adv_dst = *a.adv_src + a.adv_add + m_live;
}

template <int NT, bool FRAG>
static void launch_pair_t(const GemvArgs& a, int per, int grid, hipStream_t s) {
  if (per <= 4)
    hipLaunchKernelGGL((k_gemv_pair<NT, 4, FRAG>), dim3(grid), dim3(kGpWaves * kWave), 0, s, a);
  else if (per <= 8)
    hipLaunchKernelGGL((k_gemv_pair<NT, 8, FRAG>), dim3(grid), dim3(kGpWaves * kWave), 0, s, a);
  else
    hipLaunchKernelGGL((k_gemv_pair<NT, 10, FRAG>), dim3(grid), dim3(kGpWaves * kWave), 0, s, a);
}

// False when the launch does not fit the kernel: 2..16 fp32 input rows, one
// normed segment of at most 2560 (ten k steps a wave: what the registers hold),
// at least a half tile for every one of 256 CUs (fewer blocks would leave CUs
// without work where k_gemvf's smaller loads do not matter) and at most
// kGpMaxTiles each (beyond, 16-feature blocks divide evenly enough: at 5 half
// tiles per CU they are 2.5 per CU, at 6 already 3).
bool launch_gemv_pair(const GemvArgs& a, hipStream_t s) {
  constexpr int kCus = 256;
  const int tiles = (a.N + 7) / 8, per = (a.in[0].K / 32 + kGpWaves - 1) / kGpWaves;
  const int nt = (tiles + kCus - 1) / kCus;
  if (a.n_in != 1 || a.M < 2 || a.M > kMaxM || a.in[0].K % 32 != 0 || !a.in[0].gain || a.fin_gain || a.xn_out ||
      a.epi == kEpiArgmax || per > 10 || tiles < kCus || nt > kGpMaxTiles)
    return false;
  const int grid = (tiles + nt - 1) / nt;
#define WC_GP(NT)                                                                        \
  case NT:                                                                               \
    a.wfrag ? launch_pair_t<NT, true>(a, per, grid, s) : launch_pair_t<NT, false>(a, per, grid, s); \
    return true;
  switch (nt) {
    WC_GP(1)
    WC_GP(2)
    WC_GP(3)
    WC_GP(4)
    WC_GP(5)
  }
#undef WC_GP
  return false;
}

}  // namespace wc
