/*  p2hip_split.h – the exact-mode five-value GEMM on the bf16 matrix cores, with fp32 rows split into exact parts.
 *
 *  Included by p2hip.hip after p2hip_kernels.h (ExactArgs, the 4-bit selector records, silu_p2, DevScopeOut).
 */
#ifndef P2HIP_SPLIT_H
#define P2HIP_SPLIT_H

namespace p2k {

template <int WM_, int WN_, int FM_, int FN_>
struct XsGeo {
    static constexpr int WM = WM_, WN = WN_, FM = FM_, FN = FN_;
    static constexpr int BM = 16 * FM * WM, BN = 16 * FN * WN, NT = 64 * WM * WN;
    static constexpr int STEP = BM * 64 * 6;               /* bytes of one 64-row K step of the split rows */
    static constexpr int NO = (BM * 8 + NT - 1) / NT;       /* octets (8 consecutive k of a row) per thread and step */
    static constexpr int PITCH = BN + 4;                    /* floats per staged output row */
    static_assert(BM * PITCH * 4 <= 2 * STEP, "the outputs are staged in the ring");
    static_assert(BM <= 64, "a lane per row's flag");
};

/* The exact route for many rows: products and parts as gemm_xf's, but a workgroup splits its rows once into LDS for
 * all its waves (in gemm_xf every wave splits what it reads, and the split's VALU work bounds it), so the matrix cores
 * have 96 instructions a step for a thread's 16 split values. Waves are WM × WN over the tile, each FM row groups by
 * FN column groups; rows are two steps ahead in registers and one in the two-slot LDS ring (a barrier a step), records
 * a unit ahead in registers. At the end of each piece of K (XsCuts) the planes' sums are folded into running outputs,
 * which gives gemm_xf's bits. 64 × 128, two workgroups per CU: M = 6000, 4096 → 1024 421 → 214 µs and 1024 → 4096
 * 438 → 221 against the fp32 matrix cores, 1.41 PFLOP/s of bf16 products, where a loop of nothing but these matrix
 * instructions reaches 1.7 on random operands and 2.0 on planes this sparse (power). Counters, launched back to back:
 * the matrix cores are busy in 62 % of the cycles, at 1.9 GHz of the card's 2.4; three VALU instructions to a matrix
 * one. Launched for longer than a few ms the clock falls further (281 µs in a replayed graph). Other tiles, with the
 * sums folded every 512 rows: 48 × 128 1 to 4 % slower, 64 × 64 11 to 14 %, 96 × 128 spilled. */
template <class G, bool TAIL>
__global__ __launch_bounds__(G::NT, 2) void gemm_xs(ExactArgs g)
{
    constexpr int FM = G::FM, FN = G::FN, BM = G::BM, BN = G::BN, NT = G::NT, NO = G::NO, STEP = G::STEP;
    __shared__ __attribute__((aligned(16))) int8_t ring[2 * STEP];
    __shared__ __attribute__((aligned(16))) float f_lo[BN], f_hi[BN];
    __shared__ int lowbits[BM];   /* 1: a row with values whose parts leave bits out */

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, grp = lane >> 4, x = lane & 15;
    const int wm = wave / G::WN, wn = wave % G::WN;
    /* workgroup b runs on XCD b % 8: each XCD takes a run of consecutive tiles, columns first, so its L2 holds the
     * rows of few row bands and all the records */
    const int tiles = g.tiles_n * ((g.M + BM - 1) / BM), per = (tiles + 7) / 8;
    const int tile = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (tile >= tiles || ((int)blockIdx.x >> 3) >= per) return;
    const int tile_n = tile % g.tiles_n, tile_m = tile / g.tiles_n;
    const int n0 = tile_n * BN, m0 = tile_m * BM;
    const int M = g.M, N = g.N, K = g.K, units = g.units;

    /* weights are multiplied as ±1/2 (bf16 0x3f00: its low byte is zero), so the factors are twice lo and hi; hi as
     * the reference expands it, fmaf(1, hi − lo, lo) */
    for (int c = tid; c < BN; c += NT) {
        const int n = min(n0 + c, N - 1);
        const float lo = g.lo[n], hi = __builtin_fmaf(1.0f, g.hi[n] - lo, lo);
        f_lo[c] = 2.0f * lo;
        f_hi[c] = 2.0f * hi;
    }
    for (int c = tid; c < BM; c += NT) lowbits[c] = 0;

    /* octet q of this thread: row orow, k = 64 t + 8 o; its place in a part's 1 KB block of (16 rows, half h):
     * operand lane (o / 2, row % 16), the row turned by 4 (o / 2) + 2 h so that the eight octets of a row land on
     * eight different 16-byte columns of the banks */
    const float *asrc[NO];
    int adst[NO];
    uint32_t low[NO];
    const int o = tid & 7;
#pragma unroll
    for (int q = 0; q < NO; q++) {
        const int row = min((tid >> 3) + q * (NT / 8), BM - 1);
        asrc[q] = g.A + (size_t)min(m0 + row, M - 1) * g.lda + 8 * o;
        adst[q] = ((row >> 4) * 2 + (o & 1)) * 3072 + ((o >> 1) * 16 + ((row & 15) ^ (2 * o))) * 16;
        low[q] = 0u;
    }
    auto has = [&](int q) __attribute__((always_inline)) { return (q + 1) * NT <= BM * 8 || tid + q * NT < BM * 8; };
    const uint8_t *b_src[FN];
#pragma unroll
    for (int i = 0; i < FN; i++)
        b_src[i] = g.rec + (size_t)min((n0 >> 4) + wn * FN + i, N / 16 - 1) * units * 1024 + lane * 16;

    float av[2][NO][8];
    /* Straight-line loads (a branch around them would make the compiler wait for them where it ends). With TAIL
     * (K % 64 != 0, K % 4 == 0) a quad at or beyond K reads the row's last one and becomes 0 as it is split. */
    const int t_last = (K - 1) / 64;
    auto load_a = [&](int t, float (&av)[NO][8]) __attribute__((always_inline)) {
        const int k = 64 * min(t, t_last);
        const int k0 = TAIL ? min(k, K - 4 - 8 * o) : k, k1 = TAIL ? min(k + 4, K - 4 - 8 * o) : k + 4;
#pragma unroll
        for (int q = 0; q < NO; q++) {
            const float4 u = *reinterpret_cast<const float4 *>(asrc[q] + k0);
            const float4 v = *reinterpret_cast<const float4 *>(asrc[q] + k1);
            av[q][0] = u.x; av[q][1] = u.y; av[q][2] = u.z; av[q][3] = u.w;
            av[q][4] = v.x; av[q][5] = v.y; av[q][6] = v.z; av[q][7] = v.w;
        }
    };
    auto put_a = [&](int t, int buf, float (&av)[NO][8]) __attribute__((always_inline)) {
        const int k = 64 * t + 8 * o;
#pragma unroll
        for (int q = 0; q < NO; q++) {
            if (!has(q)) break;
            if (TAIL) {
#pragma unroll
                for (int e = 0; e < 8; e++) av[q][e] = k + (e & 4) < K ? av[q][e] : 0.0f;
            }
            v8bf p[3];
            split8(av[q], p, low[q]);
#pragma unroll
            for (int s = 0; s < 3; s++)
                *reinterpret_cast<v8bf *>(ring + buf * STEP + adst[q] + 1024 * s) = p[s];
        }
    };

    v4f accL[FN][FM], accH[FN][FM], run[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; i++)
#pragma unroll
        for (int j = 0; j < FM; j++) accL[i][j] = accH[i][j] = run[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    /* one 64-row step from ring slot `buf`, the records' dwords 2S and 2S + 1: half h multiplies k = 16 g + 8 h ..
     * + 7 of the step, lane group g; smallest part first */
    auto step = [&](auto stag, int buf, const uint4 (&rec)[FN]) __attribute__((always_inline)) {
        constexpr int S = decltype(stag)::value;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            v8bf a[3][FM];
            const int8_t *src = ring + buf * STEP + (wm * FM * 2 + h) * 3072 + (grp * 16 + (x ^ (4 * grp + 2 * h))) * 16;
#pragma unroll
            for (int j = 0; j < FM; j++)
#pragma unroll
                for (int p = 0; p < 3; p++)
                    a[p][j] = *reinterpret_cast<const v8bf *>(src + j * 6144 + p * 1024);
#pragma unroll
            for (int i = 0; i < FN; i++) {
                const uint32_t r = S == 0 ? (h == 0 ? rec[i].x : rec[i].y) : (h == 0 ? rec[i].z : rec[i].w);
                v8bf bl, bh;
                decode_planes(r, bl, bh);
#pragma unroll
                for (int p = 2; p >= 0; p--)
#pragma unroll
                    for (int j = 0; j < FM; j++) {
                        accL[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl, a[p][j], accL[i][j], 0, 0, 0);
                        accH[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh, a[p][j], accH[i][j], 0, 0, 0);
                    }
            }
        }
    };
    auto fold = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < FN; i++) {
            const int c = 16 * (wn * FN + i) + 4 * grp;
            const v4f lo = *reinterpret_cast<const v4f *>(f_lo + c), hi = *reinterpret_cast<const v4f *>(f_hi + c);
#pragma unroll
            for (int j = 0; j < FM; j++) {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    run[i][j][e] += __builtin_fmaf(lo[e], accL[i][j][e], hi[e] * accH[i][j][e]);
                accL[i][j] = accH[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
    };

    uint4 rec[FN], nrec[FN];
    auto rec_of = [&](int u, uint4 (&r)[FN]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < FN; i++) r[i] = *reinterpret_cast<const uint4 *>(b_src[i] + (size_t)min(u, units - 1) * 1024);
    };
    /* rows two steps ahead in registers, split into the ring one step ahead; records a unit ahead */
    rec_of(0, rec);
    load_a(0, av[0]);
    load_a(1, av[1]);
    put_a(0, 0, av[0]);
    const XsCuts cuts(units);
    int cut = cuts.half, piece = cuts.half;   /* the unit before which the next piece starts; this piece's length */
    for (int u = 0; u < units; u++) {
        if (u == cut) {
            fold();
            if (cuts.half < cuts.su) piece = cuts.su - piece;
            cut += piece;
        }
        rec_of(u + 1, nrec);
        load_a(2 * u + 2, av[0]);
        lds_barrier();   /* slot 0 is written (and slot 1 read out) by every wave */
        step(std::integral_constant<int, 0>{}, 0, rec);
        put_a(2 * u + 1, 1, av[1]);
        load_a(2 * u + 3, av[1]);
        lds_barrier();
        step(std::integral_constant<int, 1>{}, 1, rec);
        put_a(2 * u + 2, 0, av[0]);   /* past the last unit: unused */
#pragma unroll
        for (int i = 0; i < FN; i++) rec[i] = nrec[i];
    }
    fold();
#pragma unroll
    for (int q = 0; q < NO; q++)
        if (has(q) && (low[q] & 0xffffu)) lowbits[(tid >> 3) + q * (NT / 8)] = 1;
    lds_barrier();   /* every wave is done with the ring: the outputs are staged in it */
    if (__any(lowbits[lane % BM] != 0)) {   /* the same for every wave */
        const float *rows[FM];
#pragma unroll
        for (int j = 0; j < FM; j++) rows[j] = g.A + (size_t)min(m0 + 16 * (wm * FM + j) + x, M - 1) * g.lda;
        v4f sums[FN][FM];
#pragma unroll
        for (int i = 0; i < FN; i++)
#pragma unroll
            for (int j = 0; j < FM; j++) {
                sums[i][j] = run[i][j];
                run[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            }
        piece = cuts.half;
        for (int u = 0; u < units; u += piece, piece = cuts.half < cuts.su ? cuts.su - piece : piece) {
            xs_low_bits<FM, FN>(rows, b_src, K, u, min(units, u + piece), accL, accH);
            fold();
        }
#pragma unroll
        for (int i = 0; i < FN; i++)
#pragma unroll
            for (int j = 0; j < FM; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) run[i][j][e] = __builtin_fmaf(run[i][j][e], 1.0f / kXsLift, sums[i][j][e]);
    }
    float *stg = reinterpret_cast<float *>(ring);
#pragma unroll
    for (int i = 0; i < FN; i++)
#pragma unroll
        for (int j = 0; j < FM; j++)
            *reinterpret_cast<v4f *>(stg + (16 * (wm * FM + j) + x) * G::PITCH + 16 * (wn * FN + i) + 4 * grp) = run[i][j];
    lds_barrier();

    constexpr int TPR = BN / 4, RPP = NT / TPR;
    const int cq = tid % TPR, n = n0 + 4 * cq;
    const DevScopeOut cout(g.C + (size_t)m0 * g.ldc, (size_t)min(BM, M - m0) * g.ldc * 4, g.c_wt);
    if (n >= N) return;
    for (int row = tid / TPR; row < BM; row += RPP) {
        const int m = m0 + row;
        if (m >= M) break;
        const v4f sum = xs_finish(g, m, n, *reinterpret_cast<const v4f *>(stg + row * G::PITCH + 4 * cq));
        float *cp = g.C + (size_t)m * g.ldc + n;
        v4f c0 = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        if (g.beta != 0.0f) {
            if (g.c_vec4) {
                c0 = *reinterpret_cast<const v4f *>(cp);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) c0[e] = cp[e];
            }
            if (g.beta != 1.0f) {
#pragma unroll
                for (int e = 0; e < 4; e++) c0[e] = c0[e] * g.beta;
            }
        }
        v4f r;
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] = __builtin_fmaf(g.alpha, sum[e], c0[e]);
        if (g.act) {
#pragma unroll
            for (int e = 0; e < 4; e++) r[e] = silu_p2(r[e]);
        }
        if (g.c_vec4) {
            cout.st16(((size_t)row * g.ldc + n) * 4, r);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) cp[e] = r[e];
        }
    }
}

}  // namespace p2k

#endif
