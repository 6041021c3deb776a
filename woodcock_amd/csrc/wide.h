// wide.h -- many-row passes on the matrix cores (wide.hip): the arguments and
// launchers of the GEMM over split activations and of what surrounds it.
#pragma once
#include "wc_common.h"

namespace wc {

// Split activations ("planes"): an fp32 row as three bf16 terms whose sum it is
// exactly, in the order the GEMM's MFMA fragments read them (wd_index in
// wide.hip): 6 bytes per element, rows padded to whole tiles of 16.
inline size_t wide_plane_bytes(size_t rows, size_t k) { return (rows + 15) / 16 * 16 * k * 6; }

// ------------------------------------------------------------------ activations -> planes
constexpr int kWidePrepSegs = 3;
struct WidePrepArgs {
  struct Seg {
    const void* x;           // fp32 or bf16 rows
    int64_t ld;
    int bf16;
    const int32_t* row_idx;  // optional gather: row r reads row_idx[r] + row_add, clamped into [0, max_row) if > 0
    int row_add, max_row;
    const uint16_t* gain;    // RMSNorm gain, or NULL: the rows as they are
    int K;
  } seg[kWidePrepSegs];
  int n_seg;
  int M;       // live rows (the last tile's rows past them are zeros)
  float eps;
  uint16_t* xa;
  int steps;   // k steps of all segments together
};

int launch_wide_prep(const WidePrepArgs& a, hipStream_t s);

// ------------------------------------------------------------------ the GEMM

enum WideEpi { kWideStore = 0, kWideResidual = 1, kWideSiluPair = 2 };

struct WideArgs {
  const uint16_t* xa;        // planes of the input rows
  int steps;                 // K / 32
  int steps0;                // k steps of the first weight segment along K (steps: only one)
  const uint16_t* w[3][2];   // bf16 weights [output segment][k segment], row-major, row stride ldw
  int64_t ldw;
  int seg_start[4];          // first weight row of each output segment
  int n_seg;
  int M, N;                  // rows; weight rows (SiLU pair: rows of gate, which w[1] = up mirrors)
  float* y;                  // [M][ldy]
  int64_t ldy;
  const float* res;          // residual [M][ldres], rows gathered through res_row when given
  int64_t ldres;
  const int32_t* res_row;
  int res_add;
  uint16_t* planes;          // SiLU pair: the outputs as planes of N / 32 steps
};

int launch_wide_gemm(const WideArgs& a, int epi, hipStream_t s);

// y [L][out] (+)= x [L][in] . W [out][in]^T on the matrix cores: fp32 x, bf16 or
// fp32 W, in a multiple of 32, x and W 16-byte aligned
int launch_wide_linear(const float* x, int L, int in, const void* W, int w_dtype, int out, float* y, int accumulate,
                       hipStream_t s);

// ------------------------------------------------------------------ q / k norm, RoPE, append (head_dim 128)

struct WideQkvArgs {
  const float* qkv;  // [rows][(H + 2 Hk) D]
  int H, Hk, rows;
  const uint16_t *q_gain, *k_gain;
  float eps;
  const float *rope_cos, *rope_sin;
  int rope_max;
  const int32_t* positions;  // [rows] or NULL: offset + row
  const int32_t* offset_dev;
  int offset_add;
  float* q;  // [rows][H D] normalised and rotated
  void *kc, *vc;
  int cap;
};

int launch_wide_qkv(const WideQkvArgs& a, int kv_dtype, hipStream_t s);

// y = RMSNorm(x) of `rows` rows of K (a multiple of 8)
int launch_wide_norm(const float* x, float* y, int rows, int K, const uint16_t* gain, float eps, hipStream_t s);
// *dst = *src + add
int launch_wide_advance(int32_t* dst, const int32_t* src, int add, hipStream_t s);

// ------------------------------------------------------------------ attention (head_dim 128)

struct WideAttnArgs {
  const float* q;  // [rows][H D]
  int64_t ld_q;
  int H, Hk, rows;
  const void *k, *v;           // key t of kv head h at h * ld_head + t * ld_key elements
  int64_t ld_head, ld_key;
  int keys;                    // rows that exist (cache capacity, or T)
  const int32_t* offset_dev;   // causal: row r sees keys <= *offset_dev + offset_add + r
  int offset_add;
  int window;
  const uint8_t* mask;         // [rows][mask_ld], or NULL: causal with offset_dev, everything without
  int64_t mask_ld;
  float scale;
  float* partial;              // optional scratch of `partial_floats`: few blocks over many keys split them
  size_t partial_floats;
  float* out;                  // [rows][H D], or NULL
  uint16_t* planes;            // the output as planes of H D / 32 steps, or NULL
};

int launch_wide_attn(const WideAttnArgs& a, int kv_dtype, hipStream_t s);

}  // namespace wc
