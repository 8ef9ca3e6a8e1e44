// gemm_s.hip — the int8 GEMMs at row counts that leave most of the chip idle in gemm.hip's 128- and
// 256-row tiles (a query, a paragraph, a few documents): the same values, bit for bit, with the same
// epilogues, in tiles of 32 or 64 rows.
#include <algorithm>

#include "common.h"
#include "gemm_args.h"
#include "rowmath.h"

namespace e2mi {

bool gemm_fold_fast();

namespace {

// how the int32 products become f32: per 128-block in the reference's order, by the activation scale
// only with the weight scale once at the end (e2mi_gemm_set_fold), or once over the whole K (per-token
// activation scales)
enum { FOLD_EXACT = 0, FOLD_FAST = 1, FOLD_TOK = 2 };

// f16 of an f32 value that is already rounded (the register barrier keeps the compiler from folding
// the multiply that produced x into the conversion)
__device__ inline uint32_t f16_rn(float x) {
    asm volatile("" : "+v"(x));
    return __builtin_bit_cast(uint16_t, (_Float16)x);
}

// tile `pid` of the N-major tile list (all row tiles of one column tile, then the next) cut into one
// contiguous chunk per XCD, so a column tile's weight rows are fetched into one XCD's L2
__device__ inline int xcd_tile(int bid, int tiles) {
    const int per = (tiles + 7) / 8, t = (bid & 7) * per + (bid >> 3);
    return (bid >> 3) < per && t < tiles ? t : -1;
}

// The workgroup's BM x BN tile: the first `tiles` (tiles_m row tiles) dealt to the XCDs, then, in a forward
// planned on the device, those of the rows past the expected count, in the order of the grid, if there are such
// rows (dealt by the capacity, the expected rows would crowd some XCDs: q|k|v 768 -> 1280, 2304 of 4096 rows, 22.9
// against 13.8 us).
template <int BM, int BN>
__device__ inline bool tile_of(const int *rows, int M, int tiles_m, int tiles, int &m0, int &n0) {
    const int first = (tiles + 7) & ~7;
    if ((int)blockIdx.x < first) {
        const int t = xcd_tile(blockIdx.x, tiles);
        m0 = (t % tiles_m) * BM, n0 = (t / tiles_m) * BN;
        return t >= 0;
    }
    const int t = blockIdx.x - first, rest_m = (M + BM - 1) / BM - tiles_m;
    m0 = (tiles_m + t % rest_m) * BM, n0 = (t / rest_m) * BN;
    return m0 < *rows;
}

template <int NW, int RU, int CU>
struct Small {
    static constexpr int R = RU == 2 ? 4 : 3;              // blocks of W in flight per wave
    static constexpr int BN = 16 * CU * NW, BM = 16 * RU;  // tile columns and rows
    static constexpr int CPW = 16 * CU;                    // columns of a wave
    static constexpr int FP = BN + 4;                  // staging pitch, floats
    static constexpr int lds(int nb) {
        return nb * RU * 2048 + NW * R * CU * 2048 + nb * 256 + BN * 4 + BM * 4;
    }
};

// An NW-wave workgroup computes BM = 16 RU rows x 16 NW columns, each wave 16 columns of all rows by
// v_mfma_i32_16x16x64_i8. What bounds these calls is the chain launch -> operand latency -> fold ->
// store, not bytes or operations, so every load a wave can hold is issued at once: the tile's rows
// for the whole K (shared, one barrier) and the first R of the wave's own 2-KB weight blocks, the
// rest as their slots are read. Weight blocks are private to a wave: no barrier in the K loop, only
// its own load counts. The folded tile goes through LDS once, so that a row is held by 32 or 64
// lanes in the epilogue.
//
// NC > 0: the activations are made here from the norm_add before the GEMM (NormIn, rows of 256 NC), each
// column tile's workgroup norming the tile's rows again: 2 x 4 K bytes a row more to load, under the
// weight loads, against a row kernel's launch (3.3-3.9 us at 32-256 rows). The row kernel's steps
// (rowops.hip, ROW_ADDNORM / ROW_ADDSCALE) with k_gemm_an's byte packing: the same bits.
template <int EPI, int NW, int RU, int CU, int FOLD, int NC = 0>
__global__ __launch_bounds__(NW * 64, 1) void k_gemm_s(const int *rows, GemmArgs p, int tiles_m, int tiles, NormIn ni) {
    using S = Small<NW, RU, CU>;
    constexpr int R = S::R, CPW = S::CPW, BN = S::BN, BM = S::BM, FP = S::FP, NT = NW * 64;
    extern __shared__ __align__(16) unsigned char smem[];
    int m0, n0;
    if (!tile_of<BM, BN>(rows, p.M, tiles_m, tiles, m0, n0)) return;
    const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, c = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = p.K / kQBlock, nsb = FOLD == FOLD_TOK ? 1 : nb;

    const v4u rA = rsrc_words(p.A, (uint32_t)((size_t)p.M * p.lda));
    const v4u rW = rsrc_words(p.W, (uint32_t)((size_t)p.N * p.ldw));
    const v4u rS = rsrc_words(p.as, (uint32_t)((size_t)p.M * nsb * 4));
    const v4u rV = rsrc_words(p.ws, (uint32_t)((size_t)p.N * 4));
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const lds_void *)smem);
    const uint32_t oW = nb * RU * 2048, oS = oW + NW * R * CU * 2048, oV = oS + nb * 256, oI = oV + BN * 4;

    // load j of a 16-row slice fills its rows 8 j .. + 7: lane l fetches row l / 8's chunk
    // (l % 8) ^ swzk(row), which depends on j's parity. Rows past M (N) read as zero.
    const uint32_t ch[2] = {(uint32_t)((lane & 7) ^ (lane >> 4)) << 4, (uint32_t)((lane & 7) ^ (4 + (lane >> 4))) << 4};
    const uint32_t lr = (uint32_t)lane >> 3;
    constexpr int NR = BM / NW, ND = NC > 0 ? NC : 1;  // rows a wave norms, float4 chunks per lane of a row
    float4 ny[NR][ND], nx[NR][ND], ga[ND], gn[ND];
    if constexpr (NC > 0) {
#pragma unroll
        for (int j = 0; j < NR; j++)
#pragma unroll
            for (int i = 0; i < NC; i++) {
                const size_t o = (size_t)min(m0 + wave * NR + j, p.M - 1) * (256 * NC) + 4 * (lane + 64 * i);
                ny[j][i] = ld4(ni.y + o);
                nx[j][i] = ld4(ni.x + o);
            }
#pragma unroll
        for (int i = 0; i < NC; i++) {
            ga[i] = ld4(ni.gamma_a + 4 * (lane + 64 * i));
            gn[i] = ni.gamma_n ? ld4(ni.gamma_n + 4 * (lane + 64 * i)) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    } else {
        for (int i = wave; i < nb * RU * 2; i += NW) {
            const int b = i / (RU * 2), j = i % (RU * 2);
            dma16(rA, lds0 + (uint32_t)i * 1024u, (uint32_t)(m0 + 8 * j + lr) * (uint32_t)p.lda + ((j & 1) ? ch[1] : ch[0]),
                  (uint32_t)b * kQBlock);
        }
        for (int b = wave; b < nsb; b += NW)
            dma4(rS, lds0 + oS + (uint32_t)b * 256u, (uint32_t)(m0 + lane) * (uint32_t)nsb * 4u, (uint32_t)b * 4u);
    }
    if (wave < BN / 64) dma4(rV, lds0 + oV + wave * 256u, (uint32_t)(n0 + wave * 64 + lane) * 4u, 0);
    const uint32_t ring = oW + wave * R * CU * 2048;
    auto issue_w = [&](int b) {
        const uint32_t st = lds0 + ring + (uint32_t)(b % R) * (CU * 2048u);
#pragma unroll
        for (int j = 0; j < 2 * CU; j++)
            dma16(rW, st + j * 1024u, (uint32_t)(n0 + wave * CPW + 8 * j + lr) * (uint32_t)p.ldw + ch[j & 1],
                  (uint32_t)b * kQBlock);
    };
    const int ahead = min(nb, R);
    for (int b = 0; b < ahead; b++) issue_w(b);
    // wait until at most n of this wave's weight blocks are in flight
    auto wait_items = [&](int n) {
        if (n >= 4) vm_wait<8 * CU>();
        else if (n == 3) vm_wait<6 * CU>();
        else if (n == 2) vm_wait<4 * CU>();
        else if (n == 1) vm_wait<2 * CU>();
        else vm_wait<0>();
    };
    if (rows && m0 >= *rows) {  // planned on the device: no row here (the loads land before the LDS is released)
        vm_wait<0>();
        return;
    }
    // the epilogue's own operands: loaded once no weight block is left to wait for, so that they arrive
    // under the last products and the staging
    constexpr int RPW = BM / NW;  // QKV: rows of a wave
    const int hd = n0 >> 8, i0 = hh * 64 + c;
    const bool qk = hd < p.qH + p.qKV, isq = hd < p.qH;
    float cv[RPW][2], sv[RPW][2], gm[4];
    int pos[RPW];
    constexpr int QB = EPI == EPI_GEGLU ? BN / 256 : BN / 128, HW = NT / 32, QI = BM * QB / HW;
    float4 mu[QI];
    if constexpr (EPI == EPI_QKV) {
#pragma unroll
        for (int j = 0; j < RPW; j++) {
            const int m = min(m0 + wave * RPW + j, p.M - 1);
            pos[j] = p.pos ? p.pos[m] : m % p.qS;
        }
    }
    auto load_epi = [&]() {
        if constexpr (EPI == EPI_QKV) {
            const float *gam = isq ? p.q_gamma : p.k_gamma;
            gm[0] = gam[i0], gm[1] = gam[i0 + 32], gm[2] = gam[i0 + 128], gm[3] = gam[i0 + 160];
#pragma unroll
            for (int j = 0; j < RPW; j++) {
                const size_t e = (size_t)pos[j] * 256 + i0;
                cv[j][0] = p.cs[e], cv[j][1] = p.cs[e + 32];
                sv[j][0] = p.sn[e], sv[j][1] = p.sn[e + 32];
            }
        }
        if constexpr (EPI == EPI_GELUMUL) {
#pragma unroll
            for (int k = 0; k < QI; k++) {
                const int it = k * HW + (tid >> 5);
                mu[k] = ld4(p.mul + (size_t)min(m0 + it / QB, p.M - 1) * p.ldmul + n0 + (it % QB) * 128 + 4 * c);
            }
        }
    };
    if constexpr (NC > 0) {
#pragma unroll
        for (int j = 0; j < NR; j++) {
            const int r = wave * NR + j, m = m0 + r;
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < NC; i++) ss += sumsq4(ny[j][i]);
            float inv = rms_inv(group_sum<64>(ss), 256 * NC, ni.eps);
            ss = 0.f;
#pragma unroll
            for (int i = 0; i < NC; i++) {
                const float4 y = scale4(ny[j][i], inv, ga[i]), x = nx[j][i];
                const float4 v = make_float4(__fmul_rn(y.x + x.x, ni.post_scale), __fmul_rn(y.y + x.y, ni.post_scale),
                                             __fmul_rn(y.z + x.z, ni.post_scale), __fmul_rn(y.w + x.w, ni.post_scale));
                ny[j][i] = v;
                if (n0 == 0 && m < p.M) st4(ni.x_out + (size_t)m * (256 * NC) + 4 * (lane + 64 * i), v);
                ss += sumsq4(v);
            }
            if (ni.gamma_n) {
                inv = rms_inv(group_sum<64>(ss), 256 * NC, ni.eps);
#pragma unroll
                for (int i = 0; i < NC; i++) ny[j][i] = scale4(ny[j][i], inv, gn[i]);
            }
#pragma unroll
            for (int i = 0; i < NC; i++) {  // chunk l + 64 i: block 2 i + l / 32, its bytes 4 (l % 32) .. + 3
                const float4 v = ny[j][i];
                const QScale q = qscale(group_max<32>(amax4(v)));
                const int blk = 2 * i + hh;
                *(uint32_t *)(smem + blk * (RU * 2048) + (r >> 4) * 2048 + swz(r & 15, c >> 2) + (c & 3) * 4) =
                    pack4_magic(v.x, v.y, v.z, v.w, q.inv);
                if (c == 0) *(float *)(smem + oS + blk * 256 + r * 4) = q.sc;
            }
        }
        wait_items(ahead);
        lds_barrier();
    } else {
        wait_items(ahead);
        asm volatile("s_barrier" ::: "memory");  // every wave's part of A and the scales has landed
    }

    float f[RU][CU][4];
#pragma unroll
    for (int r = 0; r < RU; r++)
#pragma unroll
        for (int u = 0; u < CU; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) f[r][u][i] = 0.f;
    const int cl = lane & 15, rq = lane >> 4;  // operand row / output column, K chunk / output row quad
    float ws[CU];
#pragma unroll
    for (int u = 0; u < CU; u++) ws[u] = *(const float *)(smem + oV + (wave * CPW + 16 * u + cl) * 4);
    uint32_t fo[2];  // this lane's chunk of K half h in a 16-row slice
#pragma unroll
    for (int h = 0; h < 2; h++) fo[h] = (uint32_t)swz(cl, 4 * h + rq);
    v4i wf[CU][2], af[RU][2];
    auto read_frags = [&](int b) {
        const unsigned char *sw = smem + ring + (b % R) * (CU * 2048), *sa = smem + b * RU * 2048;
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int u = 0; u < CU; u++) wf[u][h] = *(const v4i *)(sw + u * 2048 + fo[h]);
#pragma unroll
            for (int r = 0; r < RU; r++) af[r][h] = *(const v4i *)(sa + r * 2048 + fo[h]);
        }
    };
    const v4i zero = {};
    // block b's products, from fragments read earlier; then its slot takes block b + R and block
    // b + 1's fragments are read, under the fold of block b - 1
    auto mul = [&](int b, v4i (&acc)[RU][CU]) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int r = 0; r < RU; r++)
#pragma unroll
                for (int u = 0; u < CU; u++)
                    acc[r][u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                        af[r][h], wf[u][h], h == 0 && (FOLD != FOLD_TOK || b == 0) ? zero : acc[r][u], 0, 0, 0);
        if (b + R < nb) issue_w(b + R);
        if (b + 1 < nb) {
            wait_items(min(nb - 1, b + R) - (b + 1));
            read_frags(b + 1);
        }
    };
    auto fold = [&](int b, const v4i (&acc)[RU][CU]) {
        const float *sb = (const float *)(smem + oS + b * 256);
#pragma unroll
        for (int r = 0; r < RU; r++) {
            const float4 a4 = *(const float4 *)(sb + r * 16 + rq * 4);
            const float av[4] = {a4.x, a4.y, a4.z, a4.w};
#pragma unroll
            for (int u = 0; u < CU; u++)
#pragma unroll
                for (int i = 0; i < 4; i++)  // the reference's order (FOLD_FAST: ws once, below)
                    f[r][u][i] = __builtin_fmaf((float)acc[r][u][i], FOLD == FOLD_FAST ? av[i] : __fmul_rn(av[i], ws[u]),
                                                f[r][u][i]);
        }
    };
    wait_items(ahead - 1);
    read_frags(0);
    v4i acc0[RU][CU], acc1[RU][CU];
    mul(0, acc0);
    int b = 1;
    if constexpr (FOLD == FOLD_TOK) {
        for (; b < nb; b++) mul(b, acc0);
        fold(0, acc0);
    } else {
        for (; b + 2 < nb; b += 2) {
            mul(b, acc1);
            fold(b - 1, acc0);
            mul(b + 1, acc0);
            fold(b, acc1);
        }
        load_epi();
        if (b + 1 < nb) {
            mul(b, acc1);
            fold(b - 1, acc0);
            mul(b + 1, acc0);
            fold(b, acc1);
            fold(b + 1, acc0);
        } else if (b < nb) {
            mul(b, acc1);
            fold(b - 1, acc0);
            fold(b, acc1);
        } else {
            fold(0, acc0);
        }
    }

    // the folded values with the optional bias and clamp (as in gemm.hip: both or none)
    const bool post = p.bias != nullptr || p.lo > -1e30f || p.hi < 1e30f;
#pragma unroll
    for (int u = 0; u < CU; u++) {
        const int n = n0 + wave * CPW + 16 * u + cl;
        const float bias = post && p.bias ? p.bias[min(n, p.N - 1)] : 0.f;
#pragma unroll
        for (int r = 0; r < RU; r++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float v = f[r][u][i];
                if constexpr (FOLD == FOLD_FAST) v = __fmul_rn(v, ws[u]);
                if (post) v = fminf(fmaxf(v + bias, p.lo), p.hi);
                f[r][u][i] = v;
            }
    }
    // register i of row unit r holds row 16 r + 4 rq + i
    if constexpr (EPI == EPI_F32) {
#pragma unroll
        for (int r = 0; r < RU; r++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int m = m0 + 16 * r + 4 * rq + i;
#pragma unroll
                for (int u = 0; u < CU; u++) {
                    const int n = n0 + wave * CPW + 16 * u + cl;
                    if (m < p.M && n < p.N) p.Y[(size_t)m * p.ldy + n] = f[r][u][i];
                }
            }
        return;
    }
    float *stg = (float *)smem;
    lds_barrier();  // every wave is past its last fragment read
#pragma unroll
    for (int r = 0; r < RU; r++)
#pragma unroll
        for (int u = 0; u < CU; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) stg[(16 * r + 4 * rq + i) * FP + wave * CPW + 16 * u + cl] = f[r][u][i];
    lds_barrier();

    if constexpr (EPI == EPI_I8Q || EPI == EPI_GELUMUL || EPI == EPI_GEGLU) {
        // a half-wave per (row, 128 output columns), lane c its columns 4 c .. + 3
        constexpr bool GG = EPI == EPI_GEGLU;
        const int o0 = GG ? n0 / 2 : n0;
#pragma unroll
        for (int k = 0; k < QI; k++) {
            const int it = k * HW + (tid >> 5), row = it / QB, qb = it % QB, m = m0 + row;
            const int oc = o0 + qb * 128 + 4 * c;
            float v[4];
            if constexpr (GG) {
                const float *g = stg + row * FP + qb * 256 + (c >> 3) * 64 + (c & 7) * 4;
                const float4 x = ld4(g), u = ld4(g + 32);
                v[0] = gelu_tanh(x.x) * u.x;
                v[1] = gelu_tanh(x.y) * u.y;
                v[2] = gelu_tanh(x.z) * u.z;
                v[3] = gelu_tanh(x.w) * u.w;
            } else {
                const float4 x = ld4(stg + row * FP + qb * 128 + 4 * c);
                v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w;
                if constexpr (EPI == EPI_GELUMUL) {
                    const float4 u = mu[k];
                    v[0] = gelu_tanh(v[0]) * u.x;
                    v[1] = gelu_tanh(v[1]) * u.y;
                    v[2] = gelu_tanh(v[2]) * u.z;
                    v[3] = gelu_tanh(v[3]) * u.w;
                }
            }
            const QScale s = qscale(group_max<32>(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])))));
            if (m < p.M) {
                *(uint32_t *)(p.Yq + (size_t)m * p.ldyq + oc) = pack4_magic(v[0], v[1], v[2], v[3], s.inv);
                if (c == 0) p.ys[(size_t)m * p.ldys + (oc >> 7)] = s.sc;
                if (EPI != EPI_I8Q && p.Y) st4(p.Y + (size_t)m * p.ldy + oc, make_float4(v[0], v[1], v[2], v[3]));
            }
        }
    }

    if constexpr (EPI == EPI_QKV) {
        // one head: W's rows in rotate-half pair order, so column wn * 128 + 32 t + c is dimension
        // (t >> 1) * 128 + wn * 64 + (t & 1) * 32 + c. A wave per row, lane (wn = hh, c) its four
        // columns t: the sum of squares over t, then over the lanes 16, 8, 4, 2, 1 apart, then both
        // wn, is the addition tree of p_epilogue_qkv (gemm.hip), so both kernels give the same bits.
        static_assert(EPI != EPI_QKV || BN == 256, "a tile is one head of 256");
        const int nqk = p.qH + p.qKV;
        float *inv_s = (float *)(smem + oI);
        float x[RPW][4];
#pragma unroll
        for (int j = 0; j < RPW; j++)
#pragma unroll
            for (int k = 0; k < 4; k++) x[j][k] = stg[(wave * RPW + j) * FP + hh * 128 + 32 * k + c];
#pragma unroll
        for (int j = 0; j < RPW; j++) {
            float a = __fmul_rn(x[j][0], x[j][0]);
#pragma unroll
            for (int k = 1; k < 4; k++) a = a + __fmul_rn(x[j][k], x[j][k]);
            a = group_sum<32>(a);
            a = a + xor_lane<32>(a);
            const float inv = __fdiv_rn(1.0f, __fsqrt_rn(__fdiv_rn(a, 256.0f) + p.eps));
            const int m = m0 + wave * RPW + j;
            if (qk) {
                const int hq = isq ? hd : hd - p.qH, ld = (isq ? p.qH : p.qKV) * 256;
                uint32_t lo16[2], hi16[2];
                float *o32 = isq ? p.q32 : p.k32;
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const float u = __fmul_rn(__fmul_rn(x[j][k], inv), gm[k]);
                    const float w = __fmul_rn(__fmul_rn(x[j][k + 2], inv), gm[k + 2]);
                    const float lo = __fmul_rn(u, cv[j][k]) - __fmul_rn(w, sv[j][k]);
                    const float hi = __fmul_rn(w, cv[j][k]) + __fmul_rn(u, sv[j][k]);
                    lo16[k] = f16_rn(lo);
                    hi16[k] = f16_rn(hi);
                    if (o32 && m < p.M) {
                        float *o = o32 + (size_t)m * ld + hq * 256 + i0 + 32 * k;
                        o[0] = lo;
                        o[128] = hi;
                    }
                }
                // the halves swapped so that each store writes 64 consecutive dimensions
                const auto sl = __builtin_amdgcn_permlane32_swap(lo16[0], lo16[1], false, false);
                const auto sh = __builtin_amdgcn_permlane32_swap(hi16[0], hi16[1], false, false);
                if (m < p.M) {
                    uint16_t *o = (isq ? p.q16 : p.k16) + (size_t)m * ld + hq * 256 + lane;
                    o[0] = (uint16_t)sl[0];
                    o[64] = (uint16_t)sl[1];
                    o[128] = (uint16_t)sh[0];
                    o[192] = (uint16_t)sh[1];
                }
            } else {
                if (lane == 0) inv_s[wave * RPW + j] = inv;
                if (p.v32 && m < p.M) {
                    float *o = p.v32 + (size_t)m * p.qKV * 256 + (hd - nqk) * 256 + i0;
                    o[0] = __fmul_rn(x[j][0], inv), o[32] = __fmul_rn(x[j][1], inv);
                    o[128] = __fmul_rn(x[j][2], inv), o[160] = __fmul_rn(x[j][3], inv);
                }
            }
        }
        if (!qk) {
            // V^T: a thread per (dimension, 16 rows), 8 rows a 16-byte store where 8 consecutive rows
            // are 8 aligned positions of one sequence
            lds_barrier();
            const int vh = hd - nqk, Sq = p.qS, d = tid & 255;
            const float *col = stg + ((d & ~0xC0) | (d & 0x40) << 1 | (d & 0x80) >> 1);
            const bool fast = Sq % 8 == 0 && ((uintptr_t)p.vt16 & 15) == 0;
            for (int r8 = (tid >> 8) * 8; r8 < BM; r8 += NT / 32) {
                uint32_t h[8];
#pragma unroll
                for (int k = 0; k < 8; k++) h[k] = f16_rn(__fmul_rn(col[(r8 + k) * FP], inv_s[r8 + k]));
                const int m = m0 + r8;
                if (fast && m + 8 <= p.M) {
                    uint16_t *dst = p.vt16 + ((size_t)((m / Sq) * p.qKV + vh) * 256 + d) * Sq + m % Sq;
                    *(uint4 *)dst = make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16);
                } else {
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        const int mm = m + k;
                        if (mm < p.M)
                            p.vt16[((size_t)((mm / Sq) * p.qKV + vh) * 256 + d) * Sq + mm % Sq] = (uint16_t)h[k];
                    }
                }
            }
        }
    }
}

// 32 x 32 output tiles, the K blocks dealt to the 8 waves: each wave loads its blocks' A and W (8 KB
// a block, all in flight at once), multiplies them and leaves the exact int32 block products in the
// block's weight slot; after one barrier the 512 threads fold the blocks in the reference's order.
// One operand latency whatever K is, and N / 32 workgroups per 32 rows. (Built and not kept: the norm_add
// of the finished rows in the workgroup that an atomic count finds last. The exchange past the XCDs'
// caches made it 11.9 us at 512 x 512, 256 rows, against 5.0 + 3.9 us for this kernel and the row
// kernel.)
template <int FOLD>
__global__ __launch_bounds__(512, 1) void k_gemm_sk(const int *rows, GemmArgs p, int tiles_m, int tiles) {
    extern __shared__ __align__(16) unsigned char smem[];
    int m0, n0;
    if (!tile_of<32, 32>(rows, p.M, tiles_m, tiles, m0, n0)) return;
    const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, c = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = p.K / kQBlock, nsb = FOLD == FOLD_TOK ? 1 : nb;
    const v4u rA = rsrc_words(p.A, (uint32_t)((size_t)p.M * p.lda));
    const v4u rW = rsrc_words(p.W, (uint32_t)((size_t)p.N * p.ldw));
    const v4u rS = rsrc_words(p.as, (uint32_t)((size_t)p.M * nsb * 4));
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const lds_void *)smem);
    const uint32_t oS = nb * 8192;  // slot b: A at b * 8192, W (then the products) 4 KB on; scales from oS
    const uint32_t ch[2] = {(uint32_t)((lane & 7) ^ (lane >> 4)) << 4, (uint32_t)((lane & 7) ^ (4 + (lane >> 4))) << 4};
    const uint32_t lr = (uint32_t)lane >> 3;
    for (int b = wave; b < nb; b += 8) {
        const uint32_t st = lds0 + (uint32_t)b * 8192u, ko = (uint32_t)b * kQBlock;
#pragma unroll
        for (int j = 0; j < 4; j++)
            dma16(rW, st + 4096u + j * 1024u, (uint32_t)(n0 + 8 * j + lr) * (uint32_t)p.ldw + ch[j & 1], ko);
#pragma unroll
        for (int j = 0; j < 4; j++)
            dma16(rA, st + j * 1024u, (uint32_t)(m0 + 8 * j + lr) * (uint32_t)p.lda + ch[j & 1], ko);
        if (FOLD != FOLD_TOK || b == 0)
            dma4(rS, lds0 + oS + (uint32_t)b * 256u, (uint32_t)(m0 + lane) * (uint32_t)nsb * 4u, (uint32_t)b * 4u);
    }
    const int row = tid >> 4, n = n0 + 2 * (tid & 15), m = m0 + row;
    const float ws0 = p.ws[min(n, p.N - 1)], ws1 = p.ws[min(n + 1, p.N - 1)];
    const bool post = p.bias != nullptr || p.lo > -1e30f || p.hi < 1e30f;
    float b0 = 0.f, b1 = 0.f;
    if (p.bias) b0 = p.bias[min(n, p.N - 1)], b1 = p.bias[min(n + 1, p.N - 1)];
    if (rows && m0 >= *rows) {  // planned on the device: no row here (the loads land before the LDS is released)
        vm_wait<0>();
        return;
    }
    vm_wait<0>();
    for (int b = wave; b < nb; b += 8) {
        unsigned char *sa = smem + b * 8192;
        v16i acc = {};
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            const int o = swz(c, kk * 2 + hh);
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(*(const v4i *)(sa + o), *(const v4i *)(sa + 4096 + o), acc, 0, 0, 0);
        }
        int *out = (int *)(sa + 4096);
#pragma unroll
        for (int i = 0; i < 16; i++) out[(8 * (i >> 2) + 4 * hh + (i & 3)) * 32 + c] = acc[i];
    }
    lds_barrier();
    float f0 = 0.f, f1 = 0.f;
    if constexpr (FOLD == FOLD_TOK) {
        int2 sum = make_int2(0, 0);
#pragma unroll 4
        for (int b = 0; b < nb; b++) {
            const int2 v = *(const int2 *)(smem + b * 8192 + 4096 + tid * 8);
            sum.x += v.x;
            sum.y += v.y;
        }
        const float a = *(const float *)(smem + oS + row * 4);
        f0 = __builtin_fmaf((float)sum.x, __fmul_rn(a, ws0), 0.f);
        f1 = __builtin_fmaf((float)sum.y, __fmul_rn(a, ws1), 0.f);
    } else {
#pragma unroll 4
        for (int b = 0; b < nb; b++) {
            const int2 v = *(const int2 *)(smem + b * 8192 + 4096 + tid * 8);
            const float a = *(const float *)(smem + oS + b * 256 + row * 4);
            f0 = __builtin_fmaf((float)v.x, FOLD == FOLD_FAST ? a : __fmul_rn(a, ws0), f0);
            f1 = __builtin_fmaf((float)v.y, FOLD == FOLD_FAST ? a : __fmul_rn(a, ws1), f1);
        }
    }
    if constexpr (FOLD == FOLD_FAST) f0 = __fmul_rn(f0, ws0), f1 = __fmul_rn(f1, ws1);
    if (post) {
        f0 = fminf(fmaxf(f0 + b0, p.lo), p.hi);
        f1 = fminf(fmaxf(f1 + b1, p.lo), p.hi);
    }
    if (m < p.M) {
        float *y = p.Y + (size_t)m * p.ldy + n;
        if (n + 1 < p.N && ((uintptr_t)y & 7) == 0) *(float2 *)y = make_float2(f0, f1);
        else {
            if (n < p.N) y[0] = f0;
            if (n + 1 < p.N) y[1] = f1;
        }
    }
}

// 64 x 128 output tiles between the tiles above and gemm.hip's: A and W stream through an LDS ring of
// three 128-wide K blocks (24 KB each), loaded two ahead by all eight waves with one barrier a block, so
// two workgroups share a CU up to 30 blocks and one holds up to 350 (the activation scales of the whole K
// stay in LDS, 256 bytes a block). A wave computes 32 x 32 outputs (4 v_mfma_i32_32x32x32_i8 and 8
// LDS reads a block; k_gemm_s's 64 x 16 read the whole A tile in every wave) and folds a block's products
// while the next block's fragments arrive. What bounds it is that chain, 0.5 us a block for one workgroup a
// CU (gemm.hip's 128 x 128 tiles with one wave a SIMD: 1.05). 3072 -> 768, 2520 rows: 31.3 -> 19.1 us
// (620 TOP/s); 2048 -> 512, 4096 rows: 22.9 -> 15.0. A ring of six blocks, one workgroup a CU, measured
// 19.7 and 15.5, and 33.9 against 26.4 at 3072 -> 768, 4096 rows.
constexpr int kRing = 3;  // K blocks
template <int FOLD>
__global__ __launch_bounds__(512, 4) void k_gemm_ring(const int *rows, GemmArgs p, int tiles_m, int tiles) {
    extern __shared__ __align__(16) unsigned char smem[];
    int m0, n0;
    if (!tile_of<64, 128>(rows, p.M, tiles_m, tiles, m0, n0)) return;
    const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, c = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
    const int nb = p.K / kQBlock;
    const v4u rA = rsrc_words(p.A, (uint32_t)((size_t)p.M * p.lda));
    const v4u rW = rsrc_words(p.W, (uint32_t)((size_t)p.N * p.ldw));
    const v4u rS = rsrc_words(p.as, (uint32_t)((size_t)p.M * nb * 4));
    const v4u rV = rsrc_words(p.ws, (uint32_t)((size_t)p.N * 4));
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const lds_void *)smem);
    constexpr int R = kRing;
    constexpr uint32_t kSlot = 24 * 1024, oS = R * kSlot;  // slot: A 8 KB, W 16 KB; then the scales
    const uint32_t oV = oS + (uint32_t)nb * 256u;
    if (rows && m0 >= *rows) return;  // planned on the device: no row here
    for (int b = wave; b < nb; b += 8)
        dma4(rS, lds0 + oS + (uint32_t)b * 256u, (uint32_t)(m0 + lane) * (uint32_t)nb * 4u, (uint32_t)b * 4u);
    if (wave < 2) dma4(rV, lds0 + oV + wave * 256u, (uint32_t)(n0 + wave * 64 + lane) * 4u, 0);
    // load j of a tile fills its rows 8 j .. + 7; every wave loads one of A's and two of W's a block
    const uint32_t lr = (uint32_t)lane >> 3, x = (uint32_t)(lane & 7);
    const uint32_t chA = (x ^ (((wave & 1) << 2) + (lane >> 4))) << 4, ch0 = (x ^ (lane >> 4)) << 4, ch1 = (x ^ (4 + (lane >> 4))) << 4;
    const uint32_t vA = (uint32_t)(m0 + 8 * wave + lr) * (uint32_t)p.lda + chA;
    const uint32_t vW0 = (uint32_t)(n0 + 16 * wave + lr) * (uint32_t)p.ldw + ch0;
    const uint32_t vW1 = (uint32_t)(n0 + 16 * wave + 8 + lr) * (uint32_t)p.ldw + ch1;
    auto issue = [&](int b) {
        const uint32_t st = lds0 + (uint32_t)(b % R) * kSlot, ko = (uint32_t)b * kQBlock;
        dma16(rA, st + wave * 1024u, vA, ko);
        dma16(rW, st + 8192u + wave * 2048u, vW0, ko);
        dma16(rW, st + 8192u + wave * 2048u + 1024u, vW1, ko);
    };
    for (int b = 0; b < min(nb, R - 1); b++) issue(b);
    // this wave's part of every block but the last n has landed and its own fragment reads are done; past
    // the barrier that holds for every wave
    auto sync = [&](int n) {
        if (n >= 1) asm volatile("s_waitcnt vmcnt(3) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    static_assert(R == 3, "sync leaves one block in flight");
    uint32_t fo[4];
#pragma unroll
    for (int k = 0; k < 4; k++) fo[k] = (uint32_t)swz(c, 2 * k + hh);
    float f[16], ws = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) f[i] = 0.f;
    v4i af[4], wf[4];
    auto fetch = [&](int b) {  // block b's fragments; its ring predecessor's slot takes block b + R - 1
        sync(min(nb - 1, b + R - 2) - b);
        if (b + R - 1 < nb) issue(b + R - 1);
        const unsigned char *st = smem + (uint32_t)(b % R) * kSlot;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            af[k] = *(const v4i *)(st + wm * 4096 + fo[k]);
            wf[k] = *(const v4i *)(st + 8192 + wn * 4096 + fo[k]);
        }
    };
    auto mul = [&](v16i &acc) {
        acc = (v16i){};
#pragma unroll
        for (int k = 0; k < 4; k++) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[k], wf[k], acc, 0, 0, 0);
    };
    auto fold = [&](int b, const v16i &acc) {
        const float *sb = (const float *)(smem + oS + b * 256) + wm * 32 + 4 * hh;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const float4 a4 = ld4(sb + 8 * g);
            const float av[4] = {a4.x, a4.y, a4.z, a4.w};
#pragma unroll
            for (int i = 0; i < 4; i++)  // the reference's order (FOLD_FAST: ws once, below)
                f[4 * g + i] = __builtin_fmaf((float)acc[4 * g + i], FOLD == FOLD_FAST ? av[i] : __fmul_rn(av[i], ws), f[4 * g + i]);
        }
    };
    v16i acc0, acc1;
    fetch(0);
    ws = *(const float *)(smem + oV + (wn * 32 + c) * 4);
    mul(acc0);
    int b = 1;
    for (; b + 1 < nb; b += 2) {
        fetch(b);
        fold(b - 1, acc0);
        mul(acc1);
        fetch(b + 1);
        fold(b, acc1);
        mul(acc0);
    }
    if (b < nb) {
        fetch(b);
        fold(b - 1, acc0);
        mul(acc0);
    }
    fold(nb - 1, acc0);
    const int n = n0 + wn * 32 + c;
    const bool post = p.bias != nullptr || p.lo > -1e30f || p.hi < 1e30f;
    const float bias = p.bias ? p.bias[min(n, p.N - 1)] : 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int m = m0 + wm * 32 + 8 * (i >> 2) + 4 * hh + (i & 3);
        float v = f[i];
        if constexpr (FOLD == FOLD_FAST) v = __fmul_rn(v, ws);
        if (post) v = fminf(fmaxf(v + bias, p.lo), p.hi);
        if (m < p.M && n < p.N) p.Y[(size_t)m * p.ldy + n] = v;
    }
}

template <class K>
int set_lds(K kern) {
    return check_hip(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024),
                     "gemm lds attribute");
}

int ring_lds(int nb) { return kRing * 24 * 1024 + nb * 256 + 512; }

// the grid of a kernel with BM x BN tiles: those of the first `few` rows, then the rest (tile_of)
struct TileGrid {
    int tiles_m, tiles;
    dim3 grid;
    TileGrid(const GemmArgs &p, int few, int bm, int bn) {
        const int tn = (p.N + bn - 1) / bn, tm = (p.M + bm - 1) / bm;
        tiles_m = (few + bm - 1) / bm;
        tiles = tiles_m * tn;
        grid = dim3((tiles + 7) / 8 * 8 + (tm - tiles_m) * tn);
    }
};

template <int EPI, int NW, int RU, int CU, int FOLD, int NC = 0>
int launch_s1(hipStream_t s, const GemmArgs &p, int few) {
    using T = Small<NW, RU, CU>;
    auto kern = k_gemm_s<EPI, NW, RU, CU, FOLD, NC>;
    static bool attr = false;
    if (!attr) {
        if (set_lds(kern)) return -1;
        attr = true;
    }
    const TileGrid g(p, few, T::BM, T::BN);
    hipLaunchKernelGGL(kern, g.grid, dim3(NW * 64), T::lds(p.K / kQBlock), s, p.rows, p, g.tiles_m, g.tiles, norm_in());
    return check_hip(hipGetLastError(), "gemm launch");
}
template <int EPI, int NW, int RU, int CU>
int launch_s(hipStream_t s, const GemmArgs &p, int few, bool tok) {
    if constexpr (EPI == EPI_F32 || EPI == EPI_I8Q)
        if (tok) return launch_s1<EPI, NW, RU, CU, FOLD_TOK>(s, p, few);
    return gemm_fold_fast() ? launch_s1<EPI, NW, RU, CU, FOLD_FAST>(s, p, few) : launch_s1<EPI, NW, RU, CU, FOLD_EXACT>(s, p, few);
}
template <int FOLD>
int launch_sk(hipStream_t s, const GemmArgs &p, int few) {
    auto kern = k_gemm_sk<FOLD>;
    static bool attr = false;
    if (!attr) {
        if (set_lds(kern)) return -1;
        attr = true;
    }
    const TileGrid g(p, few, 32, 32);
    hipLaunchKernelGGL(kern, g.grid, dim3(512), p.K / kQBlock * 8448, s, p.rows, p, g.tiles_m, g.tiles);
    return check_hip(hipGetLastError(), "gemm launch");
}

template <int FOLD>
int launch_ring(hipStream_t s, const GemmArgs &p, int few) {
    auto kern = k_gemm_ring<FOLD>;
    static bool attr = false;
    if (!attr) {
        if (set_lds(kern)) return -1;
        attr = true;
    }
    const TileGrid g(p, few, 64, 128);
    hipLaunchKernelGGL(kern, g.grid, dim3(512), ring_lds(p.K / kQBlock), s, p.rows, p, g.tiles_m, g.tiles);
    return check_hip(hipGetLastError(), "gemm launch");
}

constexpr int kLds = 160 * 1024;

// with the norm_add before it (NormInScope): 32-row tiles, rows of 512 or 768
template <int EPI, int NW>
int launch_norm1(hipStream_t s, const GemmArgs &p, int few) {
    const bool fast = gemm_fold_fast();
    if (p.K == 768)
        return fast ? launch_s1<EPI, NW, 2, 1, FOLD_FAST, 3>(s, p, few) : launch_s1<EPI, NW, 2, 1, FOLD_EXACT, 3>(s, p, few);
    return fast ? launch_s1<EPI, NW, 2, 1, FOLD_FAST, 2>(s, p, few) : launch_s1<EPI, NW, 2, 1, FOLD_EXACT, 2>(s, p, few);
}
int launch_norm(hipStream_t s, const GemmArgs &p, int epi, int few) {
    if (p.K != 512 && p.K != 768) {
        set_error("gemm: a norm_add before the GEMM needs rows of 512 or 768 (K=%d)", p.K);
        return -1;
    }
    switch (epi) {
    case EPI_F32: return launch_norm1<EPI_F32, 8>(s, p, few);
    case EPI_GELUMUL: return launch_norm1<EPI_GELUMUL, 8>(s, p, few);
    case EPI_GEGLU: return launch_norm1<EPI_GEGLU, 16>(s, p, few);
    case EPI_QKV: return launch_norm1<EPI_QKV, 16>(s, p, few);
    default: set_error("gemm: no norm_add before this GEMM"); return -1;
    }
}

thread_local NormIn t_norm;

}  // namespace

const NormIn &norm_in() { return t_norm; }
NormInScope::NormInScope(const NormIn &n) { t_norm = n; }
NormInScope::~NormInScope() { t_norm = NormIn{}; }

// Which kernel takes an M x N x K GEMM. The outputs are the same bits whichever it is; the lines lie
// where the measured times cross (us per launch, weights not in L2, gemm.hip's kernel last).
//
// 256-column tiles (GeGLU: the two 128-column halves of a quantization block; q|k|v: a head): 32-row
// tiles while one round of the CUs covers them, 64-row tiles while one round covers those. GeGLU
// 768 -> 2304: 7.0 | 9.0 | 14.2 at 32 rows, 13.3 | 10.6 | 15.1 at 1024 (288 and 144 tiles), 19.4 | 19.4 |
// 16.0 at 2048; q|k|v 768 -> 1280: 7.7 | 11.7 | 16.5 at 32, 9.6 | 13.0 | 17.5 at 1024, 17.2 | 15.1 | 19.3
// at 3008, 24.4 | 26.0 | 19.6 at 4096.
//
// 128-column tiles and the K-split 32 x 32 tiles: the least of five fitted times. A K-split tile keeps
// 8.25 KB of LDS a block, so up to 9 blocks two or more of them share a CU. 768 -> 768, K-split | 32 |
// 64 | gemm.hip: 3.4 | 5.3 | 6.3 | 9.8 at 32 rows, 6.1 | 6.7 | 8.6 | 10.8 at 1024, 11.7 | 16.1 | 16.3 |
// 12.0 at 3008, 15.2 | 17.2 | 17.0 | 12.6 at 4096; 2048 -> 512: 5.1 | 9.3 | - | 20.0 at 32, 18.8 | 12.4 |
// - | 21.5 at 2048, 27.0 | 20.6 | - | 22.0 at 3008; 512 -> 512 with the PLE gate's epilogue: 4.7 | 6.1 |
// 10.9 at 32 rows (32 | 64 | gemm.hip), 6.2 | 7.4 | 12.4 at 2048, 10.3 | 8.8 | 12.9 at 4096; per token
// 768 -> 1152: 3.4 | 5.1 | 5.7 | 8.0 at 32, 7.9 | 9.7 | 8.0 | 9.0 at 1024, 11.1 | 14.1 | 14.2 | 9.0 at 2048.
// With eight K-split tiles a CU the large tiles have caught up whatever K is (K-split | gemm.hip: 128 -> 768
// 7.2 | 6.6 at 3000 rows, 25.3 | 14.3 at 17408; 128 -> 4608 18.9 | 12.0 at 2048; 256 -> 1024 14.4 | 10.7 at
// 6000; 384 -> 40 53.3 | 34.5 at 262144).
// The ring up to two workgroups a CU, ring | the best of the others: 768 -> 768 8.0 | 5.7 at 1024 rows, 9.3 |
// 9.7 at 2048, 9.7 | 10.7 at 2520, 12.6 | 12.8 at 4096; 1152 -> 768 9.7 | 8.5, 10.7 | 12.1, 11.1 | 13.0, 14.8 |
// 16.1; 2048 -> 512 12.9 | 10.4, 13.6 | 12.7, 13.7 | 21.8, 15.0 | 22.9, 21.6 | 25.7 at 8192; 3072 -> 768 16.6 |
// 29.0 at 256, 26.4 | 32.6 at 4096, then 41.6 | 42.4 at 8192, 97.9 | 88.5 at 17408 (three and seven rounds).
int gemm_small_route(int M, int N, int K, int epi, bool tok) {
    const int C = num_cus(), nb = K / kQBlock;
    auto tiles = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
    if (epi == EPI_GEGLU || epi == EPI_QKV) {
        if (Small<16, 2, 1>::lds(nb) <= kLds && tiles(32, 256) <= C) return GEMM_S32;
        if (Small<8, 4, 2>::lds(nb) <= kLds && tiles(64, 256) <= C) return GEMM_S64;
        return 0;
    }
    auto rounds = [&](long t) { return (double)((t + C - 1) / C); };
    const double fill = (double)tiles(128, 128) / C, fr = (double)tiles(64, 128) / C;
    double best = tok ? 5.0 + 0.6 * nb : (epi == EPI_F32 ? 5.3 : 4.2) + 1.05 * nb + (epi == EPI_GELUMUL ? 2.5 : 0.0) + (fill > 0.5 ? 4.0 * (fill - 0.5) : 0.0);
    int route = 0;
    auto offer = [&](bool ok, double t, int r) {
        if (ok && t < best) {
            best = t;
            route = r;
        }
    };
    // (per-128 scales: a K-split tile of one to four blocks costs its loads and its exchange more than its blocks)
    const double sk = tok ? (nb <= 9 ? 0.69 : 1.0) * nb : std::max((nb <= 9 ? 0.69 : 1.1) * nb, 1.5 + 0.3 * nb);
    offer(epi == EPI_F32 && nb * 8448 <= kLds && (tok || tiles(32, 32) <= 8L * C), 3.0 + 1e-3 * sk * (double)tiles(32, 32) * 256 / C, GEMM_SK);
    offer(Small<8, 2, 1>::lds(nb) <= kLds, 1.2 + rounds(tiles(32, 128)) * (2.2 + 0.5 * nb), GEMM_S32);
    offer(Small<8, 4, 1>::lds(nb) <= kLds, 1.2 + rounds(tiles(64, 128)) * (3.4 + 0.85 * nb), GEMM_S64);
    offer(epi == EPI_F32 && !tok && ring_lds(nb) <= kLds && fr <= (ring_lds(nb) <= kLds / 2 ? 2.0 : 1.0),
          fr <= 1.0 ? 4.2 + 0.52 * nb + 2.4 * fr : 6.4 + 0.77 * nb + fr, GEMM_RING);
    return route;
}

// Runs the GEMM here when gemm_small_route takes it at `few` rows: 1 when it was launched, 0 when the
// caller's kernels take it, -1 on error.
int launch_gemm_small(hipStream_t s, const GemmArgs &p, int epi, int few, bool tok) {
    if (norm_in().y) return launch_norm(s, p, epi, few) ? -1 : 1;
    const int route = gemm_small_route(few, p.N, p.K, epi, tok);
    if (!route) return 0;
    int rc;
    if (route == GEMM_RING) {
        rc = gemm_fold_fast() ? launch_ring<FOLD_FAST>(s, p, few) : launch_ring<FOLD_EXACT>(s, p, few);
    } else if (route == GEMM_SK) {
        rc = tok ? launch_sk<FOLD_TOK>(s, p, few) : gemm_fold_fast() ? launch_sk<FOLD_FAST>(s, p, few) : launch_sk<FOLD_EXACT>(s, p, few);
    } else {
        const bool s64 = route == GEMM_S64;
        switch (epi) {
        case EPI_F32: rc = s64 ? launch_s<EPI_F32, 8, 4, 1>(s, p, few, tok) : launch_s<EPI_F32, 8, 2, 1>(s, p, few, tok); break;
        case EPI_I8Q: rc = s64 ? launch_s<EPI_I8Q, 8, 4, 1>(s, p, few, tok) : launch_s<EPI_I8Q, 8, 2, 1>(s, p, few, tok); break;
        case EPI_GELUMUL: rc = s64 ? launch_s<EPI_GELUMUL, 8, 4, 1>(s, p, few, tok) : launch_s<EPI_GELUMUL, 8, 2, 1>(s, p, few, tok); break;
        case EPI_GEGLU: rc = s64 ? launch_s<EPI_GEGLU, 8, 4, 2>(s, p, few, tok) : launch_s<EPI_GEGLU, 16, 2, 1>(s, p, few, tok); break;
        default: rc = s64 ? launch_s<EPI_QKV, 8, 4, 2>(s, p, few, tok) : launch_s<EPI_QKV, 16, 2, 1>(s, p, few, tok); break;
        }
    }
    return rc ? -1 : 1;
}

}  // namespace e2mi
