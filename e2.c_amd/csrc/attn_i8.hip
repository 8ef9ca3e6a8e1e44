// attn_i8.hip — the int8 attention variant on gfx950 int8 MFMA (v_mfma_i32_32x32x32_i8), for
// packed batches of all-valid sequences.
//
// Reference semantics (text.c:638-700 attb_i8, selected by dispatch.c's attention rule for long
// sequences): per query head h (kv head h / (H / KV)) of a sequence of S rows,
//   Q rows quantized per 128 of D (the activation quantizer), K quantized per key row and V^T per
//   dim over the sequence's keys (the weight quantizer, e2_q8w_from_f32), both with scale
//   amax * RN(1/127) and bytes rne(x * RN(127 / amax));
//   scores[i][j] = fold over D's two 128-blocks b of fma((float)acc_b, RN(qs[i][b] * ks[j]), .);
//   p = softmax(scores[i]) (max, exp, sum, then p = e * RN(1 / sum));
//   P quantized per 128-key block of the row (the activation quantizer on p);
//   ctx[i][d] = fold over key blocks b of fma((float)acc_b, RN(ps[i][b] * vs[d]), .).
// The context is then quantized per (row, 128 dims) for the O-projection GEMM, as in attn.hip.
//
// Kernels:
//   k_i8_prep      one wave per (row, q head | k head): Q per 128, K per row (float4 per lane); and
//                  per (sequence, kv head, 64-row chunk): column maxima of V
//   k_i8_vquant    per (sequence, kv head, 32-row chunk): V^T bytes (thread d writes 32 bytes of
//                  row d of V^T [KV][D][M]) and the per-dim scales
//   k_attn_i8      a workgroup is (sequence, head, 32 queries). Pass 1 walks the key tiles for each
//                  query's softmax max and sum (online); pass 2 walks them again per 128-key block:
//                  the block's probabilities, their quantization with the block's scale, then
//                  O^T += V^T P^T on int8 MFMA with int32 accumulators folded into f32 once per
//                  block. S^T = K Q^T as in attn.hip: K tile rows are permuted so a lane's 16
//                  logits are 16 consecutive keys of its query, exactly its P^T operand bytes.
#include <algorithm>

#include "common.h"

namespace e2mi {

constexpr int kI8D = 256;                           // head dim
constexpr int kI8Tile = 8192;                       // K [32 keys][256] or V^T [64 d][128 keys]
constexpr int kI8Buf = kI8Tile + 256;               // + the tile's key scales (64 loaded, 32 used)

// ---------------------------------------------------------------- Q and K quantization
struct I8PrepArgs {
    const float *q32, *k32, *v32;  // [M][H*D], [M][KV*D], [M][KV*D]
    int8_t *q8;                    // [M][H*D]
    float *qs;                     // [M][H*2]
    int8_t *k8;                    // [M][KV*D]
    float *ks;                     // [M][KV]
    int8_t *vt8;                   // [KV][D][2 M]: sequence b's keys at columns 2 start[b] + j
    float *vpart;                  // [B][KV][nch][D] column maxima of 64-row chunks
    float *vs;                     // [B][KV][D]
    const int32_t *seq_start, *seq_len;
    int M, H, KV, nch;
    int nbk;      // B KV
    uint32_t nv;  // V's workgroups of the first launch (nbk nch)
};

// V's part of the launch: workgroup c B KV + (b, kv) takes the column maxima of rows [64 c, 64 c + 64)
// of the sequence, thread = dim
__device__ inline void i8_vmax(const I8PrepArgs &a, uint32_t blk) {
    const int bk = blk % (uint32_t)a.nbk, c = blk / (uint32_t)a.nbk, b = bk / a.KV, kv = bk % a.KV, d = threadIdx.x;
    const int L = a.seq_len[b], r0 = 64 * c;
    if (r0 >= L) return;
    const int r1 = min(L, r0 + 64);
    const size_t st = (size_t)a.KV * kI8D;
    const float *src = a.v32 + ((size_t)a.seq_start[b] + r0) * st + kv * kI8D + d;
    float m8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int r = r0;
    for (; r + 8 <= r1; r += 8, src += 8 * st)
#pragma unroll
        for (int e = 0; e < 8; e++) m8[e] = fmaxf(m8[e], fabsf(src[e * st]));
    for (; r < r1; r++, src += st) m8[0] = fmaxf(m8[0], fabsf(*src));
    float am = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) am = fmaxf(am, m8[e]);
    a.vpart[((size_t)bk * a.nch + c) * kI8D + d] = am;
}

__global__ __launch_bounds__(256) void k_i8_prep(I8PrepArgs a) {
    const uint32_t blk = blockIdx.x + gridDim.x * blockIdx.y;  // (one row of the grid but for very many workgroups)
    if (blk < a.nv) return i8_vmax(a, blk);
    const int lane = threadIdx.x & 63;
    const long item = (long)(blk - a.nv) * 4 + (threadIdx.x >> 6);
    const int per = a.H + a.KV;
    if (item >= (long)a.M * per) return;
    const int row = (int)(item / per), j = (int)(item % per);
    if (j < a.H) {
        // Q: lanes 0-31 hold block 0 (d < 128), lanes 32-63 block 1
        const float4 x = *(const float4 *)(a.q32 + (size_t)row * a.H * kI8D + j * kI8D + 4 * lane);
        const float am = group_max<32>(fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))));
        const QScale s = qscale(am);
        *(uint32_t *)(a.q8 + (size_t)row * a.H * kI8D + j * kI8D + 4 * lane) = pack4_magic(x.x, x.y, x.z, x.w, s.inv);
        if ((lane & 31) == 0) a.qs[(size_t)row * a.H * 2 + j * 2 + (lane >> 5)] = s.sc;
    } else {
        // K: one scale per key row over all of D (the weight quantizer)
        const int kv = j - a.H;
        const float4 x = *(const float4 *)(a.k32 + (size_t)row * a.KV * kI8D + kv * kI8D + 4 * lane);
        const float am = group_max<64>(fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))));
        const QScale s = qscale(am);
        *(uint32_t *)(a.k8 + (size_t)row * a.KV * kI8D + kv * kI8D + 4 * lane) = pack4_magic(x.x, x.y, x.z, x.w, s.inv);
        if (lane == 0) a.ks[(size_t)row * a.KV + kv] = s.sc;
    }
}

// ---------------------------------------------------------------- V^T quantization
// grid (B * KV, ceil(max_len / 32)): thread d reduces its column's chunk maxima, then quantizes rows
// [32 c, 32 c + 32) of the sequence into 32 bytes of V^T row d
__global__ __launch_bounds__(256) void k_i8_vquant(I8PrepArgs a) {
    const int b = blockIdx.x / a.KV, kv = blockIdx.x % a.KV, c = blockIdx.y, d = threadIdx.x;
    const int L = a.seq_len[b], r0 = 32 * c;
    if (r0 >= L) return;
    const int nc = (L + 63) / 64;
    const float *part = a.vpart + (size_t)blockIdx.x * a.nch * kI8D + d;
    float am = 0.f;
    for (int i = 0; i < nc; i++) am = fmaxf(am, part[(size_t)i * kI8D]);
    const QScale s = qscale(am);
    if (c == 0) a.vs[(size_t)blockIdx.x * kI8D + d] = s.sc;
    const int n = min(32, L - r0);
    const size_t row0 = (size_t)a.seq_start[b] + r0;
    const float *src = a.v32 + row0 * a.KV * kI8D + kv * kI8D + d;
    uint32_t w[8];
#pragma unroll
    for (int g = 0; g < 8; g++) {
        float x[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int r = 4 * g + e;
            x[e] = r < n ? src[(size_t)r * a.KV * kI8D] : 0.f;
        }
        w[g] = pack4_magic(x[0], x[1], x[2], x[3], s.inv);
    }
    // sequence b's keys start at column 2 start[b] (16-byte aligned; its columns end before the
    // next sequence's, which starts at least L rows later): whole 16-byte chunks are its own
    int8_t *dst = a.vt8 + ((size_t)kv * kI8D + d) * 2 * a.M + 2 * (size_t)a.seq_start[b] + r0;
#pragma unroll
    for (int g = 0; g < 2; g++)
        if (16 * g < n) *(uint4 *)(dst + 16 * g) = make_uint4(w[4 * g], w[4 * g + 1], w[4 * g + 2], w[4 * g + 3]);
}

// ---------------------------------------------------------------- attention
struct AttnI8Args {
    const int8_t *q8;
    const float *qs;
    const int8_t *k8;
    const float *ks;
    const int8_t *vt8;
    const float *vs;
    int8_t *cq;            // [M][H*D] int8 context
    float *cs;             // [M][H*D/128]
    float *c32;            // optional [M][H*D] f32 context
    const int32_t *seq_start, *seq_len;
    const int32_t *work;   // optional: b | h << 16 | query block << 24 per workgroup, negative idle
    int M, H, KV;
};

// A block is 32 queries, four waves each on a key tile of its own. Pass 1 takes four tiles at once:
// wave w the scores of tile w; the tiles' maxima and partial sums are exchanged through LDS and folded
// in tile order by every wave. Pass 2 quantizes a 128-key block's four tiles in the four waves,
// exchanges the bytes, and each wave computes 64 of the 256 dims over the block. A wave's K tiles and
// V^T pieces (8 KB each: [32 keys][256], [64 dims][128 keys]) share a ring of two buffers, loaded a
// step ahead. KEEP (no sequence longer than 512 keys): a wave keeps its four tiles' scores in
// registers for pass 2, else they are computed again.
// What bounds it is the chain of a block: load, scores, exchange, probabilities, exchange, context. A
// workgroup of four waves that walk the tiles together, 32 queries each, has one wave on a SIMD and
// a chain four times as long; here two workgroups share a CU. us per call with the quantization (about
// 16), such workgroups -> these: 3 heads, 1 x 100 tokens 26.8 -> 16.4, 12 x 64-512 70.8 -> 36.4, 64 x 64-512 125.2
// -> 98.1; 4 heads, 2 x 1024-2048 217.7 -> 102.4, 16 x 1024-2048 661.7 -> 447.7. KEEP against computing the scores
// again: 36.4 | 41.0 and 98.1 | 111.9. Blocks of 64 queries on eight waves: 36.6, 103.8, 93.9 and 451.4.
constexpr int kI8Keep = 512;
constexpr int kI8P = 0, kI8M = 4096, kI8L = kI8M + 1024, kI8X = kI8L + 2048;  // bytes, maxima, partial sums
constexpr int kI8V = 8 * kI8Buf, kI8S = kI8V + kI8D * 4, kAttnI8Lds = kI8S + kI8X;

// WALK: a workgroup runs its entry's blocks one after the other (a kernel of its own: the loop costs the others
// 40 registers and 1-3 %).
template <bool KEEP, bool WALK>
__global__ __launch_bounds__(256, 2) void k_attn_i8(AttnI8Args a, int n_work, int nwg) {
    extern __shared__ __align__(16) unsigned char smem[];
    int q0 = blockIdx.x * 32, h = blockIdx.y, b = blockIdx.z;
    if (WALK || a.work) {  // work entry i's nwg workgroups on one XCD (i % 8)
        const int i = (blockIdx.x / (8 * nwg)) * 8 + (blockIdx.x & 7);
        const int item = i < n_work ? a.work[i] : -1;
        if (item < 0) return;
        b = item & 0xffff;
        h = (item >> 16) & 0xf;  // (one part: work_entry(b, h, 0, 1, query block))
        q0 = (item >> 24) * 128 + ((blockIdx.x >> 3) % nwg) * 32;
    }
    for (const int q1 = q0 + (WALK ? 128 : 32); q0 < min(a.seq_len[b], q1); q0 += 32) {
        int tid = threadIdx.x;
        if constexpr (WALK) asm volatile("" : "+v"(tid), "+s"(b));  // (nothing of a block is kept in registers for the next)
        const int Sk = a.seq_len[b];
        const int lane = tid & 63, half = lane >> 5, ql = lane & 31;
        const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int HD = a.H * kI8D, kvh = h / (a.H / a.KV);
        const size_t row0 = (size_t)a.seq_start[b];
        const int qi = q0 + ql, qc = min(qi, Sk - 1);  // this lane's query
        // Q^T operand (B of S^T = K Q^T): the query's d = 32 kk + 16 half .. + 16
        v4i qf[8];
        {
            const int8_t *qp = a.q8 + (row0 + qc) * HD + h * kI8D + 16 * half;
#pragma unroll
            for (int kk = 0; kk < 8; kk++) qf[kk] = *(const v4i *)(qp + 32 * kk);
        }
        const float qs0 = a.qs[(row0 + qc) * a.H * 2 + h * 2], qs1 = a.qs[(row0 + qc) * a.H * 2 + h * 2 + 1];
        float *vs_l = (float *)(smem + kI8V);
        vs_l[tid] = a.vs[((size_t)b * a.KV + kvh) * kI8D + tid];
        // the loads above complete here, under a wait the compiler sees: otherwise its wait would sit
        // inside a loop and also cover the tile loads in flight
        __builtin_amdgcn_s_waitcnt(0x0F70);

        const int ntiles = (Sk + 31) / 32, nblk = (ntiles + 3) / 4;
        const uint32_t rowB = (uint32_t)a.KV * kI8D, vpitch = 2u * (uint32_t)a.M;
        const v4u rK = rsrc_words(a.k8 + row0 * rowB + kvh * kI8D, (uint32_t)Sk * rowB);
        const v4u rKS = rsrc_words(a.ks + row0 * a.KV + kvh, (uint32_t)Sk * a.KV * 4);
        const v4u rV = rsrc_words(a.vt8 + (size_t)kvh * kI8D * 2 * a.M, (uint32_t)((size_t)kI8D * 2 * a.M));
        const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const lds_void *)smem);
        // K: load i fills physical rows rho = 4 i + lane / 16, 16-byte position lane % 16 holding chunk
        // (lane % 16) ^ (rho % 16), of key 16 ((rho / 4) % 2) + 4 (rho / 8) + rho % 4 = 16 (i % 2) + 4 (i / 2) + lane / 16;
        // keys past the sequence are out of the buffer's range and read as 0
        auto issue_k = [&](int g, int buf) __attribute__((always_inline)) {
            const int k0 = (4 * g + w) * 32;
            const uint32_t base = lds0 + (uint32_t)((2 * w + buf) * kI8Buf);
#pragma unroll
            for (int i = 0; i < 8; i++)
                dma16(rK, base + i * 1024, (uint32_t)(k0 + 16 * (i & 1) + 4 * (i >> 1) + (lane >> 4)) * rowB +
                      (uint32_t)(((lane & 15) ^ ((4 * i + (lane >> 4)) & 15)) << 4), 0u);
            dma4(rKS, base + kI8Tile, (uint32_t)(k0 + lane) * a.KV * 4, 0u);
        };
        // V^T: load i fills rows d = 8 i + lane / 8 of the wave's 64, position lane % 8 holding keys
        // 16 c .. + 15 of the block, c = (lane % 8) ^ (lane / 8)
        auto issue_v = [&](int g, int buf) __attribute__((always_inline)) {
            const uint32_t base = lds0 + (uint32_t)((2 * w + buf) * kI8Buf);
#pragma unroll
            for (int i = 0; i < 8; i++)
                dma16(rV, base + i * 1024, (uint32_t)(64 * w + 8 * i + (lane >> 3)) * vpitch +
                      (uint32_t)(2 * row0 + 128 * g + (((lane & 7) ^ (lane >> 3)) << 4)), 0u);
        };
        // the ring's stream: pass 1's K tiles, then KEEP ? V^T blocks : K tiles and V^T of each block in turn
        auto issue = [&](int n) __attribute__((always_inline)) {
            if (n < nblk) return issue_k(n, n & 1);
            const int m = n - nblk;
            if (KEEP ? m >= nblk : m >= 2 * nblk) return;
            if (KEEP) issue_v(m, n & 1);
            else if (m & 1) issue_v(m >> 1, n & 1);
            else issue_k(m >> 1, n & 1);
        };
        // every wave is past its reads of step n's buffer and its loads of step n + 1 have arrived; step n + 2's
        // go into the buffer of step n
        auto step_done = [&](int n) __attribute__((always_inline)) {
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            issue(n + 2);
        };
        auto sync = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
        unsigned char *const pq8 = smem + kI8S + kI8P;
        float *ml = (float *)(smem + kI8S + kI8M), *pl = (float *)(smem + kI8S + kI8L);

        // one K tile: S^T (8 MFMAs, two 128-d blocks), folded like the reference's GEMM, keys past the
        // sequence at -inf. s[r] is key 16 half + r of the tile (K row ql, chunk 2 kk + half).
        auto scores = [&](const unsigned char *sb, int k0, float (&s)[16]) __attribute__((always_inline)) {
            v16i acc0 = (v16i){}, acc1 = (v16i){};
#pragma unroll
            for (int kk = 0; kk < 8; kk++) {
                const v4i kf = *(const v4i *)(sb + ql * 256 + (((2 * kk + half) ^ (ql & 15)) << 4));
                if (kk < 4) acc0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf, qf[kk], acc0, 0, 0, 0);
                else acc1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf, qf[kk], acc1, 0, 0, 0);
            }
            const float *ksl = (const float *)(sb + kI8Tile) + 16 * half;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const float4 k4 = *(const float4 *)(ksl + 4 * g);
                const float kv4[4] = {k4.x, k4.y, k4.z, k4.w};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int r = 4 * g + e;
                    const float f = __builtin_fmaf((float)acc0[r], __fmul_rn(qs0, kv4[e]), 0.f);
                    const float x = __builtin_fmaf((float)acc1[r], __fmul_rn(qs1, kv4[e]), f);
                    s[r] = (k0 + 16 * half + r < Sk) ? x : -INFINITY;
                }
            }
        };

        issue(0);
        issue(1);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        float keep[KEEP ? 4 : 1][16];
        float mrun = -INFINITY, mfold = -INFINITY, lrun = 0.f, mt[4];
        int nprev = 0;
        // the partial sums of the group before (its tiles' maxima in mt), in tile order
        auto fold = [&](int g) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < 4; t++) {
                if (t < nprev) {
                    const float mnew = fmaxf(mfold, mt[t]);
                    if (mnew > -INFINITY) {
                        lrun = (mfold == -INFINITY ? 0.f : lrun * __expf(mfold - mnew)) + pl[(g & 1) * 256 + t * 64 + lane];
                        mfold = mnew;
                    }
                }
            }
        };
        auto pass1 = [&](int g, float (&s)[16]) __attribute__((always_inline)) {
            const int nt = min(4, ntiles - 4 * g);
            float mloc = -INFINITY;
            if (w < nt) {
                scores(smem + (2 * w + (g & 1)) * kI8Buf, (4 * g + w) * 32, s);
#pragma unroll
                for (int r = 0; r < 16; r++) mloc = fmaxf(mloc, s[r]);
                mloc = fmaxf(mloc, xor_lane<32>(mloc));
                if (half == 0) ml[(g & 1) * 128 + w * 32 + ql] = mloc;
            }
            step_done(g);
            fold(g - 1);
            float mine = mrun;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                if (t < nt) {
                    mt[t] = ml[(g & 1) * 128 + t * 32 + ql];
                    mrun = fmaxf(mrun, mt[t]);
                    if (t == w) mine = mrun;
                }
            }
            nprev = nt;
            if (w < nt) {
                float ps = 0.f;
#pragma unroll
                for (int r = 0; r < 16; r++) ps += s[r] == -INFINITY ? 0.f : __expf(s[r] - mine);
                pl[(g & 1) * 256 + w * 64 + lane] = ps;
            }
        };
        if constexpr (KEEP) {
#pragma unroll
            for (int g = 0; g < 4; g++)
                if (g < nblk) pass1(g, keep[g]);
        } else {
            for (int g = 0; g < nblk; g++) pass1(g, keep[0]);
        }
        sync();
        fold(nblk - 1);
        const float ltot = lrun + xor_lane<32>(lrun);
        const float inv_l = ltot > 0.f ? __fdiv_rn(1.0f, ltot) : 0.f;

        float of[2][16];
#pragma unroll
        for (int dt = 0; dt < 2; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) of[dt][r] = 0.f;
        auto pass2 = [&](int g, float (&s)[16]) __attribute__((always_inline)) {
            const int nt = min(4, ntiles - 4 * g), nv = KEEP ? nblk + g : nblk + 2 * g + 1;  // this block's V^T step
            float pv[16], am = 0.f;
#pragma unroll
            for (int r = 0; r < 16; r++) pv[r] = 0.f;
            if (w < nt) {
                if (!KEEP) scores(smem + (2 * w + ((nv - 1) & 1)) * kI8Buf, (4 * g + w) * 32, s);
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const float e = s[r] == -INFINITY ? 0.f : __expf(s[r] - mrun);
                    pv[r] = __fmul_rn(e, inv_l);
                    am = fmaxf(am, pv[r]);
                }
            }
            am = fmaxf(am, xor_lane<32>(am));
            if (half == 0) ml[w * 32 + ql] = am;
            if (KEEP && g == 0) sync();  // (step nblk - 1 was done in pass 1)
            else step_done(nv - 1);
#pragma unroll
            for (int t = 0; t < 4; t++) am = fmaxf(am, ml[t * 32 + ql]);
            const QScale ps = qscale(am);
            v4i mine;
#pragma unroll
            for (int q = 0; q < 4; q++)
                mine[q] = (int)pack4_magic(pv[4 * q], pv[4 * q + 1], pv[4 * q + 2], pv[4 * q + 3], ps.inv);
            *(v4i *)(pq8 + w * 1024 + lane * 16) = mine;
            sync();
            v16i acc[2] = {(v16i){}, (v16i){}};
            const unsigned char *vb = smem + (2 * w + (nv & 1)) * kI8Buf;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                if (t < nt) {
                    const v4i pq = *(const v4i *)(pq8 + t * 1024 + lane * 16);
#pragma unroll
                    for (int dt = 0; dt < 2; dt++) {
                        const v4i vf = *(const v4i *)(vb + (32 * dt + ql) * 128 + (((2 * t + half) ^ (ql & 7)) << 4));
                        acc[dt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf, pq, acc[dt], 0, 0, 0);
                    }
                }
            }
            // d = 64 w + 32 dt + 8 (r / 4) + 4 half + r % 4
#pragma unroll
            for (int dt = 0; dt < 2; dt++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float4 v4 = *(const float4 *)(vs_l + 64 * w + 32 * dt + 8 * q + 4 * half);
                    const float vv[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        of[dt][4 * q + e] = __builtin_fmaf((float)acc[dt][4 * q + e], __fmul_rn(ps.sc, vv[e]), of[dt][4 * q + e]);
                }
            if (!KEEP) step_done(nv);
        };
        if constexpr (KEEP) {
#pragma unroll
            for (int g = 0; g < 4; g++)
                if (g < nblk) pass2(g, keep[g]);
        } else {
            for (int g = 0; g < nblk; g++) pass2(g, keep[0]);
        }

        // a 128-dim block is two waves'
        float am = 0.f;
#pragma unroll
        for (int dt = 0; dt < 2; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) am = fmaxf(am, fabsf(of[dt][r]));
        am = fmaxf(am, xor_lane<32>(am));
        if (half == 0) ml[128 + w * 32 + ql] = am;
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        am = fmaxf(am, ml[128 + (w ^ 1) * 32 + ql]);
        const QScale qs = qscale(am);
        const size_t orow = row0 + qi;
        if (qi < Sk) {  // rows past the sequence belong to the next one
#pragma unroll
            for (int dt = 0; dt < 2; dt++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int d = 64 * w + 32 * dt + 8 * q + 4 * half;
                    *(uint32_t *)(a.cq + orow * HD + h * kI8D + d) =
                        pack4_magic(of[dt][4 * q], of[dt][4 * q + 1], of[dt][4 * q + 2], of[dt][4 * q + 3], qs.inv);
                    if (a.c32)
                        *(float4 *)(a.c32 + orow * HD + h * kI8D + d) =
                            make_float4(of[dt][4 * q], of[dt][4 * q + 1], of[dt][4 * q + 2], of[dt][4 * q + 3]);
                }
            if (half == 0 && !(w & 1)) a.cs[orow * (HD / kQBlock) + h * 2 + (w >> 1)] = qs.sc;
        }
        if constexpr (!WALK) return;
    }
}

static size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

template <bool KEEP, bool WALK>
static int launch_attn_i8(hipStream_t s, const AttnI8Args &a, int B, int max_len, int n_work, int nwg) {
    static bool attr = false;
    if (!attr) {
        if (check_hip(hipFuncSetAttribute((const void *)k_attn_i8<KEEP, WALK>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                          kAttnI8Lds), "attention_i8 lds attribute"))
            return -1;
        attr = true;
    }
    const dim3 grid = a.work ? dim3((n_work + 7) / 8 * 8 * nwg) : dim3((max_len + 31) / 32, a.H, B);
    hipLaunchKernelGGL((k_attn_i8<KEEP, WALK>), grid, dim3(256), kAttnI8Lds, s, a, n_work, nwg);
    return check_hip(hipGetLastError(), "attention_i8 launch");
}
// A work entry has four blocks of 32 queries, fewer where no sequence is that long, each a workgroup's: one
// whose block lies past its sequence costs 1-2 us of a CU's slot (300 x 1-66, 3 heads: 71.2 us with four
// workgroups an entry, 43.3 with three). From three entries a CU of sequences of at most 128, one
// workgroup walks an entry's blocks instead (four | one: 3 heads, 300 x 1-128 86.8 | 65.8; 15 heads, 64 x 8-100
// 83.9 | 60.9, 128 x 100-128 220.5 | 216.8; with fewer, 3 heads, 128 x 100-128 50.8 | 55.2).
static int launch_attn_i8(hipStream_t s, const AttnI8Args &a, int B, int max_len, int n_work) {
    if (a.work && max_len <= 128 && n_work >= 3 * num_cus()) return launch_attn_i8<true, true>(s, a, B, max_len, n_work, 1);
    const int nwg = std::min(4, (max_len + 31) / 32);
    return max_len <= kI8Keep ? launch_attn_i8<true, false>(s, a, B, max_len, n_work, nwg)
                              : launch_attn_i8<false, false>(s, a, B, max_len, n_work, nwg);
}

struct I8Ws {
    size_t q8, qs, k8, ks, vt8, vpart, vs, total;
};
static I8Ws i8_ws(int M, int B, int max_len, int H, int KV) {
    I8Ws w;
    const int nch = (max_len + 63) / 64;
    w.q8 = 0;
    w.qs = w.q8 + al256((size_t)M * H * kI8D);
    w.k8 = w.qs + al256((size_t)M * H * 2 * 4);
    w.ks = w.k8 + al256((size_t)M * KV * kI8D);
    w.vt8 = w.ks + al256((size_t)M * KV * 4);
    w.vpart = w.vt8 + al256((size_t)KV * kI8D * 2 * M);
    w.vs = w.vpart + al256((size_t)B * KV * nch * kI8D * 4);
    w.total = w.vs + al256((size_t)B * KV * kI8D * 4);
    return w;
}

}  // namespace e2mi

using namespace e2mi;

extern "C" size_t e2mi_attention_i8_workspace_bytes(int M, int B, int max_len, int H, int KV) {
    if (M <= 0 || B <= 0 || max_len <= 0 || H <= 0 || KV <= 0) return 0;
    return i8_ws(M, B, max_len, H, KV).total;
}

extern "C" int e2mi_attention_i8_packed(e2mi_stream stream, const float *q32, const float *k32,
                                        const float *v32, int M, const int32_t *seq_start,
                                        const int32_t *seq_len, int B, int max_len, int H, int KV,
                                        int D, void *workspace, int8_t *ctx_q, float *ctx_s,
                                        float *ctx32, const int32_t *work, int n_work) {
    if (D != kI8D || B <= 0 || M <= 0 || max_len <= 0 || H <= 0 || KV <= 0 || H % KV || M % 16) {
        set_error("attention_i8_packed: needs head_dim 256, H %% KV == 0 and M %% 16 == 0 "
                  "(B=%d M=%d H=%d KV=%d D=%d)", B, M, H, KV, D);
        return -1;
    }
    if (!q32 || !k32 || !v32 || !seq_start || !seq_len || !workspace || !ctx_q || !ctx_s ||
        !aligned16(q32) || !aligned16(k32) || !aligned16(v32) || ((uintptr_t)workspace & 255) ||
        ((uintptr_t)ctx_q & 3) || (ctx32 && !aligned16(ctx32))) {
        set_error("attention_i8_packed: null or misaligned pointer");
        return -1;
    }
    if ((size_t)kI8D * 2 * M >= 0x7fffffffu || (size_t)M * KV * kI8D >= 0x7fffffffu) {
        set_error("attention_i8_packed: too many rows");
        return -1;
    }
    // a work entry holds the head in 4 bits (b | h << 16 | part << 20 | parts - 1 << 22 | qb << 24,
    // the f16 kernels' encoding)
    if (work && (n_work <= 0 || B > 0xffff || H > 0xf || (max_len + 127) / 128 > 127)) {
        set_error("attention_i8_packed: work list needs n_work > 0, B < 65536, H < 16, max_len < 16257");
        return -1;
    }
    const I8Ws wo = i8_ws(M, B, max_len, H, KV);
    unsigned char *ws = (unsigned char *)workspace;
    I8PrepArgs p = {q32, k32, v32, (int8_t *)(ws + wo.q8), (float *)(ws + wo.qs), (int8_t *)(ws + wo.k8),
                    (float *)(ws + wo.ks), (int8_t *)(ws + wo.vt8), (float *)(ws + wo.vpart),
                    (float *)(ws + wo.vs), seq_start, seq_len, M, H, KV, (max_len + 63) / 64, B * KV, (uint32_t)B * KV * ((max_len + 63) / 64)};
    hipStream_t s = (hipStream_t)stream;
    // a dimension of a grid takes 2^32 threads: 2^20 workgroups a row where one row would not do
    const long items = (long)M * (H + KV), prep = p.nv + (items + 3) / 4, row = prep < (1L << 24) ? prep : 1L << 20;
    hipLaunchKernelGGL(k_i8_prep, dim3((unsigned)row, (unsigned)((prep + row - 1) / row)), dim3(256), 0, s, p);
    hipLaunchKernelGGL(k_i8_vquant, dim3(B * KV, (max_len + 31) / 32), dim3(256), 0, s, p);
    const AttnI8Args a = {p.q8, p.qs, p.k8, p.ks, p.vt8, p.vs, ctx_q, ctx_s, ctx32, seq_start, seq_len, work, M, H, KV};
    return launch_attn_i8(s, a, B, max_len, n_work);
}
