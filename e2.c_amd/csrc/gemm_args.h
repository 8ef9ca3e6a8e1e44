// gemm_args.h — what the int8 GEMM kernels share: their arguments, the epilogue kinds and the LDS
// swizzle of a 128-byte K slice.
#pragma once

#include "common.h"

namespace e2mi {

enum { EPI_F32 = 0, EPI_I8Q = 1, EPI_GEGLU = 2, EPI_GELUMUL = 3, EPI_QKV = 4 };

struct GemmArgs {
    const int8_t *A;
    const float *as;
    const int8_t *W;
    const float *ws;
    const float *bias;
    float *Y;        // EPI_F32 output, EPI_GEGLU optional f32 g
    int8_t *Yq;      // EPI_I8Q / EPI_GEGLU quantized output
    float *ys;       // ... and its per-128 scales [M][ldys]
    int32_t *accd;   // optional int32 accumulator dump [nb][M][N] (parity tests)
    const float *mul;  // EPI_GELUMUL: the multiplier of gelu(y) [M][ldmul]
    int ldmul;
    int lda, ldw, ldy, ldyq, ldys;
    int M, N, K;
    float lo, hi;
    // EPI_QKV: q/k gammas [256], RoPE tables [positions][256], each row's position (packed
    // batches) or none (row % qS), f16 outputs q [M][qH*256], k [M][qKV*256] and V^T
    // [M/qS][qKV][256][qS], optional f32 copies q, k, v [M][heads*256]
    const float *q_gamma, *k_gamma, *cs, *sn;
    const int32_t *pos;
    uint16_t *q16, *k16, *vt16;
    float *q32, *k32, *v32;
    int qH, qKV, qS;
    float eps;
    // a device row count (a multiple of 256, past M where M is below 256), which the kernels but the
    // per-token ones take as their own first argument, or null: M rows
    const int *rows;
};

// The norm_add that makes a GEMM's activations, run in the GEMM's own workgroups (gemm_s.hip; the
// engine at few rows): x' = (rmsnorm(y) * gamma_a + x) * post_scale -> x_out (another buffer than x),
// then rmsnorm(x') * gamma_n (without gamma_n: x' itself) quantized per 128. Rows of K columns.
// Set for the GEMMs that the thread launches while a NormInScope lives; they take no quantized
// activations then.
struct NormIn {
    const float *y = nullptr, *x = nullptr, *gamma_a = nullptr, *gamma_n = nullptr;
    float *x_out = nullptr;
    float post_scale = 1.f, eps = 0.f;
};
const NormIn &norm_in();
class NormInScope {
  public:
    explicit NormInScope(const NormIn &n);
    ~NormInScope();
    NormInScope(const NormInScope &) = delete;
    NormInScope &operator=(const NormInScope &) = delete;
};

// gemm_s.hip: the kernels for few rows, and which one (0: none) takes an M x N x K GEMM with the
// epilogue `epi` (tok: per-token activation scales); launch_gemm_small runs it, its tiles of the first
// `few` rows before those of the rest (DeviceRows::few), and returns 1, or returns 0 for the caller's kernels
// and -1 on error
enum { GEMM_SK = 1, GEMM_S32 = 2, GEMM_S64 = 3, GEMM_RING = 5 };  // (4 is forward_signature's)
int gemm_small_route(int M, int N, int K, int epi, bool tok);
int launch_gemm_small(hipStream_t s, const GemmArgs &p, int epi, int few, bool tok);

#if defined(__HIPCC__)
// LDS tiles hold 128-byte K slices of consecutive rows with no padding. The LDS has 64 banks of 4
// bytes and serves a ds_read_b128 16 lanes at a time; a 128-byte row spans 32 banks, so rows of
// equal parity share a bank half. The 16-byte chunk c of row r sits at slot c ^ ((r >> 1) & 7):
// the 16 consecutive rows read by one 16-lane group then cover all 64 banks once. Each
// 1-KB direct-to-LDS load fills 8 rows of a tile: lane l writes slot l, so it fetches row l/8's
// chunk (l % 8) ^ ((row >> 1) & 7).
__device__ inline int swzk(int r) { return (r >> 1) & 7; }
__device__ inline int swz(int r, int c) { return r * 128 + ((c ^ swzk(r)) << 4); }
#endif

}  // namespace e2mi
