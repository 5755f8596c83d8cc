// Kernels of the batched MoE backward on the forward's permutation
// (the reference's jt_moe_bwd_batch, src/moe_layer.c:1684-2502), gfx950.
//
// Index checks (every call, both the checked and the unchecked form):
//  k_bwd_check_q    : ids / weights / drop per pair, kept count, dWgate keys
//  k_bwd_check_off  : off[] from 0, monotone, <= T*k, off[E] == kept count
//  k_bwd_check_perm : perm[0..kept) an exact enumeration of the kept pairs
// A failed check raises EF_BAD_ID and clamps what later kernels index with,
// so every access stays in bounds; the result is then not used.
//
// Gate path (steps 1-4 of the reference):
//  k_bwd_dots   : dw[q] = fp64 dot(Ysel[q], dY[t]) in the reference's
//                 lane-4 order (src/moe_layer.c:67-86, 1985-2010)
//  k_bwd_token  : softmax Jacobian per token (:2011-2047), dLogits, the
//                 gate-path dX terms (:2048-2081) and the token's perm rows
//  k_bwd_dwgate : dWgate[e][j] in token/slot order (:2082-2103) over the
//                 stable expert sort of the kept pairs
// Expert path (steps 5-6): three bit-exact fp32 GEMM forms (per output, a
// k-ascending sequence of rounded multiplies and rounded adds, as
// src/moe_gemm.c:47-89), k_bwd_gemm_mx on 64x128 tiles where they are
// many, else k_bwd_gemm:
//  <AT, BT, EPI> with EPI_DSWIGLU (dY Wd^T -> SwiGLU backward
//  -> Dg, Du, S), EPI_DUAL ((float)((double)Dg Wg + (double)Du Wu)) and
//  EPI_STORE (D^T X weight gradients).
//  k_bwd_dx     : dX = (float)(gate + routed rows in perm order + shared)
//                 in fp64 (:2236-2245, 2354-2363, 2411-2429)
#include <algorithm>

#include "jt_dev.h"
#include "jt_launch.h"

namespace {

constexpr int EPI_STORE = 0, EPI_DUAL = 1, EPI_DSWIGLU = 2;
constexpr int MODE_ROWS = 0, MODE_WGRAD = 1;
constexpr int PAD = 4;

// Operands of one side of a launch (side 0: shared experts, side 1: routed).
// A GEMM computes C(r, c) = sum over k ascending of A(r, k) B(k, c) with
//  A_g = A[m] + g*sAg + kb*sAk, B_g = B[m] + g*sBg + kb*sBk,
//  AT: A_g(r, k) = A_g[k*lda + r], else A_g[r*lda + k];
//  BT: B_g(k, c) = B_g[c*ldb + k], else B_g[k*ldb + c];
// m selects one of three matrices (weight gradients), or A[1]/B[1] are the
// second product of EPI_DUAL; g is the expert (group), kb the first row of
// its K range (koff, ragged K) or 0.
struct Side {
    const float *A[3], *B[3];
    float *C[3];  // EPI_DSWIGLU: Dg, Du, S
    int lda, ldb, ldc;
    int64_t sAg, sBg, sCg, sAk, sBk;
    const float *G, *U;     // EPI_DSWIGLU: row q of G_g = G + g*sGg + q*ldg
    const int32_t *rowq;    // q of each output row (NULL: q = row)
    int ldg;
    int64_t sGg;
    int M, K;               // dense rows and fixed K
    const int32_t *koff;    // ragged K: rows koff[g] .. koff[g+1]
    const int4 *tiles;      // ragged M: {g, first row, rows}
    const int32_t *ntiles;
};
// MODE_ROWS: blockIdx.x < nsh are side 0's dense row tiles (mt_sh per
// group), the rest side 1's tile list; blockIdx.y the column tile.
// MODE_WGRAD: blockIdx.z < nsh is side 0, then side 1, z = 3*g + m;
// blockIdx.x / blockIdx.y the row / column tiles.
struct GemmP {
    Side sd[2];
    int nsh, mt_sh, N;
    uint32_t *err;
};

// SwiGLU backward of one element (src/moe_layer.c:1680-1682, 2204-2233) in
// fp64: sig = 1/(1+exp(-g)) with a correctly rounded division, exp within
// about an ulp of glibc's; false when acc or a result is not finite.
__device__ __forceinline__ bool dswiglu(float g, float u, float dot, float *dg, float *du,
                                        float *sv) {
    const double gi = (double)g, ui = (double)u, acc = (double)dot;
    const double sig = 1.0 / (1.0 + exp_tang(-gi));
    const double silu = gi * sig;
    const double dsilu = sig * (1.0 + gi * (1.0 - sig));
    const double gd = acc * ui * dsilu, ud = acc * silu, s = silu * ui;
    *dg = (float)gd;
    *du = (float)ud;
    *sv = (float)s;
    return isfinite(acc) && isfinite(gd) && isfinite(ud) && isfinite(s);
}

// A (R x BK) chunk of an operand: NL elements per thread, loaded into
// registers (next chunk, while the current one is computed) and stored to
// LDS as [k][r]. KMAJ: memory is contiguous along r (k-major), else along k.
template <int R, int BK, bool KMAJ>
struct Chunk {
    static constexpr int NL = R * BK / 256;
    float v[NL];
    __device__ __forceinline__ void load(const float *P, int ld, int b, int cnt, int k0, int K,
                                         int tid) {
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int idx = tid + 256 * it;
            const int r = KMAJ ? idx % R : idx / BK, kk = KMAJ ? idx / R : idx % BK;
            v[it] = (r < cnt && k0 + kk < K)
                        ? (KMAJ ? P[(int64_t)(k0 + kk) * ld + b + r] : P[(int64_t)(b + r) * ld + k0 + kk])
                        : 0.0f;
        }
    }
    __device__ __forceinline__ void store(float (*S)[R + PAD], int tid) const {
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int idx = tid + 256 * it;
            const int r = KMAJ ? idx % R : idx / BK, kk = KMAJ ? idx / R : idx % BK;
            S[kk][r] = v[it];
        }
    }
};

template <int N>
__device__ __forceinline__ void ld_row(float (&v)[N], const float *s) {
    if constexpr (N % 4 == 0) {
#pragma unroll
        for (int i = 0; i < N; i += 4) *(float4 *)&v[i] = *(const float4 *)(s + i);
    } else {
#pragma unroll
        for (int i = 0; i < N; i += 2) *(float2 *)&v[i] = *(const float2 *)(s + i);
    }
}
// acc[i][j] += a[i] * b[j]: one rounded multiply, one rounded add
template <int TM, int TN>
__device__ __forceinline__ void mul_add(float (&acc)[TM][TN], const float *as, const float *bs) {
    float av[TM], bv[TN];
    ld_row(av, as);
    ld_row(bv, bs);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = __fadd_rn(acc[i][j], __fmul_rn(av[i], bv[j]));
}

// What a block computes: rows rb .. rb+rc, columns cb .. cb+cc of group g
// (matrix m) on one side, K products from A, B. False: nothing.
struct Job {
    int side, g, m, rb, rc, cb, cc, K;
    const float *A[2], *B[2];
};
template <int EPI, int MODE, int BM, int BN>
__device__ __forceinline__ bool gemm_job(const GemmP &p, Job &j) {
    j.m = 0;
    if (MODE == MODE_ROWS) {
        const int bx = blockIdx.x;
        if (bx < p.nsh) {
            j.side = 0, j.g = bx / p.mt_sh, j.rb = (bx % p.mt_sh) * BM;
            j.rc = min(BM, p.sd[0].M - j.rb);
        } else {
            j.side = 1;
            if (bx - p.nsh >= *p.sd[1].ntiles) return false;
            const int4 tl = p.sd[1].tiles[bx - p.nsh];
            j.g = tl.x, j.rb = tl.y, j.rc = tl.z;
        }
    } else {
        int z = blockIdx.z;
        j.side = z < p.nsh ? 0 : 1;
        z -= j.side ? p.nsh : 0;
        j.g = z / 3, j.m = z % 3;
        j.rb = blockIdx.x * BM;
        j.rc = min(BM, p.sd[j.side].M - j.rb);
    }
    const Side &S = p.sd[j.side];
    j.cb = blockIdx.y * BN, j.cc = min(BN, p.N - j.cb);
    j.K = S.K;
    int64_t kb = 0;
    if (MODE == MODE_WGRAD && S.koff) {
        kb = S.koff[j.g];
        j.K = S.koff[j.g + 1] - S.koff[j.g];
    }
    j.A[0] = S.A[j.m] + j.g * S.sAg + kb * S.sAk;
    j.B[0] = S.B[j.m] + j.g * S.sBg + kb * S.sBk;
    j.A[1] = EPI == EPI_DUAL ? S.A[1] + j.g * S.sAg + kb * S.sAk : j.A[0];
    j.B[1] = EPI == EPI_DUAL ? S.B[1] + j.g * S.sBg + kb * S.sBk : j.B[0];
    return true;
}
// Output (r, c) of the block from its sums; false when not finite
template <int EPI>
__device__ __forceinline__ bool gemm_out(const Side &S, const Job &j, int r, int c, float acc,
                                         float acc2) {
    const int64_t row = j.rb + r, col = j.cb + c;
    const int64_t o = j.g * S.sCg + row * S.ldc + col;
    if constexpr (EPI == EPI_STORE) {
        S.C[j.m][o] = acc;
    } else if constexpr (EPI == EPI_DUAL) {
        S.C[0][o] = (float)((double)acc + (double)acc2);
    } else {
        const int64_t q = S.rowq ? S.rowq[row] : row;
        const int64_t at = j.g * S.sGg + q * S.ldg + col;
        float dg, du, sv;
        const bool ok = dswiglu(S.G[at], S.U[at], acc, &dg, &du, &sv);
        S.C[0][o] = dg;
        S.C[1][o] = du;
        S.C[2][o] = sv;
        return ok;
    }
    return true;
}

template <bool AT, bool BT, int EPI, int MODE, int TM, int TN>
__global__ __launch_bounds__(256) void k_bwd_gemm(GemmP p) {
    constexpr int BM = 16 * TM, BN = 16 * TN, BK = 2048 / (BM > BN ? BM : BN);
    constexpr int NP = EPI == EPI_DUAL ? 2 : 1;
    __shared__ __attribute__((aligned(16))) float As[NP][BK][BM + PAD];
    __shared__ __attribute__((aligned(16))) float Bs[NP][BK][BN + PAD];
    const int tid = threadIdx.x;
    Job j;
    if (!gemm_job<EPI, MODE, BM, BN>(p, j)) return;
    const Side &S = p.sd[j.side];
    const float *Ag = j.A[0], *Bg = j.B[0], *Ag2 = j.A[1], *Bg2 = j.B[1];
    const int rb = j.rb, rc = j.rc, cb = j.cb, cc = j.cc, K = j.K;
    const int ty = tid / 16, tx = tid % 16;
    float acc[TM][TN], acc2[EPI == EPI_DUAL ? TM : 1][EPI == EPI_DUAL ? TN : 1];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = 0.0f;
    if constexpr (EPI == EPI_DUAL) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc2[i][j] = 0.0f;
    }
    Chunk<BM, BK, AT> ca, ca2;
    Chunk<BN, BK, !BT> cbk, cb2;
    if (K > 0) {
        ca.load(Ag, S.lda, rb, rc, 0, K, tid);
        cbk.load(Bg, S.ldb, cb, cc, 0, K, tid);
        if (EPI == EPI_DUAL) {
            ca2.load(Ag2, S.lda, rb, rc, 0, K, tid);
            cb2.load(Bg2, S.ldb, cb, cc, 0, K, tid);
        }
    }
    for (int k0 = 0; k0 < K; k0 += BK) {
        ca.store(As[0], tid);
        cbk.store(Bs[0], tid);
        if (EPI == EPI_DUAL) {
            ca2.store(As[NP - 1], tid);
            cb2.store(Bs[NP - 1], tid);
        }
        __syncthreads();
        if (k0 + BK < K) {  // the next chunk's loads overlap this chunk's products
            ca.load(Ag, S.lda, rb, rc, k0 + BK, K, tid);
            cbk.load(Bg, S.ldb, cb, cc, k0 + BK, K, tid);
            if (EPI == EPI_DUAL) {
                ca2.load(Ag2, S.lda, rb, rc, k0 + BK, K, tid);
                cb2.load(Bg2, S.ldb, cb, cc, k0 + BK, K, tid);
            }
        }
        const int kend = min(BK, K - k0);
        if (kend == BK) {
#pragma unroll 8
            for (int kk = 0; kk < BK; kk++) {
                mul_add<TM, TN>(acc, &As[0][kk][ty * TM], &Bs[0][kk][tx * TN]);
                if constexpr (EPI == EPI_DUAL)
                    mul_add<TM, TN>(acc2, &As[NP - 1][kk][ty * TM], &Bs[NP - 1][kk][tx * TN]);
            }
        } else {
            for (int kk = 0; kk < kend; kk++) {
                mul_add<TM, TN>(acc, &As[0][kk][ty * TM], &Bs[0][kk][tx * TN]);
                if constexpr (EPI == EPI_DUAL)
                    mul_add<TM, TN>(acc2, &As[NP - 1][kk][ty * TM], &Bs[NP - 1][kk][tx * TN]);
            }
        }
        __syncthreads();
    }
    bool ok = true;
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int r = ty * TM + i;
        if (r >= rc) continue;
#pragma unroll
        for (int jc = 0; jc < TN; jc++) {
            const int c = tx * TN + jc;
            if (c >= cc) continue;
            float a2 = 0.0f;
            if constexpr (EPI == EPI_DUAL) a2 = acc2[i][jc];
            ok &= gemm_out<EPI>(S, j, r, c, acc[i][jc], a2);
        }
    }
    if (!ok) raise_err(p.err, EF_NONFINITE_MID);
}

typedef float v32f __attribute__((ext_vector_type(32)));

// The same sums on 64 x 128 tiles with the products made by the matrix
// cores: v_mfma_f32_32x32x1 with a zero accumulator gives 32 x 64 rounded
// products of one k (a product of -0 comes out as +0, which changes no sum:
// a sum that starts from +0 is never -0), the adds stay on the VALU. fp32
// MFMA and VALU share the lanes' multipliers, so the bound is that of a
// multiply and an add per product (56 ns of a SIMD for 2048 from registers,
// with v_mul and v_add as well: 37 T products/s on the chip). What it saves is
// everything around: one 4-byte LDS read of A and of B per lane and k for
// 2048 products, where 4 x 4 outputs a thread read 32 bytes for 1024.
// The two products of EPI_DUAL run one after the other.
template <bool AT, bool BT, int EPI, int MODE>
__global__ __launch_bounds__(256, EPI == EPI_DUAL ? 2 : 3) void k_bwd_gemm_mx(GemmP p) {
    constexpr int BM = 64, BN = 128, BK = 16;
    constexpr int NP = EPI == EPI_DUAL ? 2 : 1;
    __shared__ float As[BK][BM + PAD], Bs[BK][BN + PAD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    Job j;
    if (!gemm_job<EPI, MODE, BM, BN>(p, j)) return;
    const Side &S = p.sd[j.side];
    const int wm = wave >> 1, wn = wave & 1, K = j.K;  // wave tile 32 x 64
    v32f acc[NP];
#pragma unroll
    for (int pr = 0; pr < NP; pr++) {
        v32f sum = {};
        Chunk<BM, BK, AT> ca;
        Chunk<BN, BK, !BT> cb;
        if (K > 0) {
            ca.load(j.A[pr], S.lda, j.rb, j.rc, 0, K, tid);
            cb.load(j.B[pr], S.ldb, j.cb, j.cc, 0, K, tid);
        }
        const float *ap = &As[0][wm * 32 + (lane & 31)], *bp = &Bs[0][wn * 64 + lane];
        auto step = [&](int kk) {
            const v32f zero = {};
            sum = sum + __builtin_amdgcn_mfma_f32_32x32x1f32(ap[kk * (BM + PAD)],
                                                             bp[kk * (BN + PAD)], zero, 1, 0, 0);
        };
        for (int k0 = 0; k0 < K; k0 += BK) {
            ca.store(As, tid);
            cb.store(Bs, tid);
            __syncthreads();
            if (k0 + BK < K) {  // the next chunk's loads overlap this chunk's products
                ca.load(j.A[pr], S.lda, j.rb, j.rc, k0 + BK, K, tid);
                cb.load(j.B[pr], S.ldb, j.cb, j.cc, k0 + BK, K, tid);
            }
            if (K - k0 >= BK) {
#pragma unroll
                for (int kk = 0; kk < BK; kk++) step(kk);
            } else {
                for (int kk = 0; kk < K - k0; kk++) step(kk);
            }
            __syncthreads();
        }
        acc[pr] = sum;
    }
    bool ok = true;
#pragma unroll
    for (int v = 0; v < 32; v++) {
        const int r = wm * 32 + (v & 15) / 4 * 8 + (lane >> 5) * 4 + (v & 3);
        const int c = wn * 64 + (v >> 4) * 32 + (lane & 31);
        if (r < j.rc && c < j.cc) ok &= gemm_out<EPI>(S, j, r, c, acc[0][v], acc[NP - 1][v]);
    }
    if (!ok) raise_err(p.err, EF_NONFINITE_MID);
}

// rows: row tiles of 64 (MODE_ROWS, both sides) or output rows
// (MODE_WGRAD); groups: grid z; blocks: blocks of 64 x 64 outputs that have
// work, if the pairs spread evenly over the experts; serial, mx: MODE_WGRAD,
// see below. A form with 4x4 outputs a thread, or
//  - the matrix-core one (64 x 128 tiles, two blocks a CU with two sums, else
//    three) where the tiles hold little padding, are more than one round of
//    blocks and fill three quarters of the rounds: two sums, 900 to 1024 tiles 1
//    to 3.6% of the call below 4x4, 1056 to 1152 2 to 3% above; SwiGLU, 832 to
//    1024 tiles 1 to 1.6% above, from 1216 on 0.2 to 1.6% below. (One round of two
//    sums took 6% less or 7% more: where the list's unused blocks fall decides
//    it.) With h = 64, half of a tile padding, 7.5% above (16384 tokens, 64
//    experts top-8).
//  - 4x2 (row GEMMs) where blocks are few and a block's serial K loop is the
//    time: up to 544 blocks with two sums (448: 7 to 9% below 4x4, 528 and 544: 2%
//    above to 6% below, 768: 4% above) and 768 of the SwiGLU product (448: 6.5%
//    below, 704 and 768: 3.2% below to 2.4% above).
// (The calls: 64 to 4096 tokens, 16 to 128 experts, n 256 to 2048, h 64 to 512.)
template <bool AT, bool BT, int EPI, int MODE>
int launch_gemm(const GemmP &p, unsigned rows, unsigned groups, int64_t blocks, bool serial,
                bool mx, hipStream_t s) {
    if (rows == 0 || p.N <= 0 || groups == 0) return 0;
    auto grid = [&](int BM, int BN) {
        return dim3(MODE == MODE_ROWS ? rows : (rows + BM - 1) / BM,
                    (unsigned)((p.N + BN - 1) / BN), groups);
    };
    const dim3 g = grid(64, 128);
    const int64_t tiles = blocks / 2, slots = 256 * (EPI == EPI_DUAL ? 2 : 3);
    const bool full = MODE == MODE_ROWS ? tiles > slots && 4 * tiles > 3 * slots *
                                              ((tiles + slots - 1) / slots)
                                        : mx && tiles >= 1024;
    const bool few = MODE == MODE_ROWS ? blocks <= (EPI == EPI_DUAL ? 544 : 768)
                                       : serial || blocks < 512;
    if (full && 128 * (int64_t)g.y <= p.N + p.N / 8) {
        hipLaunchKernelGGL((k_bwd_gemm_mx<AT, BT, EPI, MODE>), g, dim3(256), 0, s, p);
    } else if (!few) {
        hipLaunchKernelGGL((k_bwd_gemm<AT, BT, EPI, MODE, 4, 4>), grid(64, 64), dim3(256), 0, s,
                           p);
    } else if constexpr (MODE == MODE_ROWS) {
        hipLaunchKernelGGL((k_bwd_gemm<AT, BT, EPI, MODE, 4, 2>), grid(64, 32), dim3(256), 0, s,
                           p);
    } else if (blocks >= 128) {
        hipLaunchKernelGGL((k_bwd_gemm<AT, BT, EPI, MODE, 2, 4>), grid(32, 64), dim3(256), 0, s,
                           p);
    } else {
        hipLaunchKernelGGL((k_bwd_gemm<AT, BT, EPI, MODE, 2, 2>), grid(32, 32), dim3(256), 0, s,
                           p);
    }
    return (int)hipGetLastError();
}

// Finiteness of up to 16 arrays in one launch (blockIdx.y = array); HBM bound
// (450 MB at 4096 tokens, n 1024: 85 us, 120 with one load in flight).
struct FinList {
    const float *p[16];
    int64_t n[16];
};
__global__ __launch_bounds__(256) void k_bwd_finite(FinList L, uint32_t *err) {
    const float *x = L.p[blockIdx.y];
    const int64_t n = L.n[blockIdx.y];
    int bad = 0;
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t step = (int64_t)gridDim.x * 256;
    if (((uintptr_t)x & 15) == 0) {  // float4 body
        const float4 *x4 = (const float4 *)x;
        for (; i + 3 * step < n / 4; i += 4 * step) {  // four loads in flight
            const float4 a = x4[i], b = x4[i + step], c = x4[i + 2 * step], d = x4[i + 3 * step];
            bad |= !isfinite(a.x) || !isfinite(a.y) || !isfinite(a.z) || !isfinite(a.w);
            bad |= !isfinite(b.x) || !isfinite(b.y) || !isfinite(b.z) || !isfinite(b.w);
            bad |= !isfinite(c.x) || !isfinite(c.y) || !isfinite(c.z) || !isfinite(c.w);
            bad |= !isfinite(d.x) || !isfinite(d.y) || !isfinite(d.z) || !isfinite(d.w);
        }
        for (; i < n / 4; i += step) {
            const float4 v = x4[i];
            bad |= !isfinite(v.x) || !isfinite(v.y) || !isfinite(v.z) || !isfinite(v.w);
        }
        for (i = n / 4 * 4 + blockIdx.x * 256 + threadIdx.x; i < n; i += step)
            bad |= !isfinite(x[i]);
    } else {
        for (; i < n; i += step) bad |= !isfinite(x[i]);
    }
    bad = wave_or_i(bad);
    if (bad && (threadIdx.x & 63) == 0) raise_err(err, EF_NONFINITE_INPUT);
}

__device__ __forceinline__ int block_sum_256(int v, int *red) {
    v = wave_sum_i(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
}

// ctrl[0] = number of kept pairs (drop == 0), ctrl[1] = kept as used (off[E]
// when the checks pass, else 0); ctrl must be zero before.
__global__ __launch_bounds__(256) void k_bwd_check_q(const uint64_t *__restrict__ ids,
                                                     const float *__restrict__ w,
                                                     const uint8_t *__restrict__ drop, int Tk,
                                                     int E, int validate,
                                                     int32_t *__restrict__ key,
                                                     int32_t *__restrict__ inv,
                                                     uint32_t *__restrict__ seen,
                                                     uint32_t *ctrl, uint32_t *err) {
    __shared__ int red[4];
    const int q = blockIdx.x * 256 + threadIdx.x;
    int kept = 0;
    if (q < Tk) {
        const uint8_t d = drop[q];
        const uint64_t id = ids[q];
        bool bad;
        if (validate) {
            const float wv = w[q];
            bad = id >= (uint64_t)E || !(wv >= 0.0f && wv <= 1.0f) || d > 1;
        } else {
            bad = d == 0 && id >= (uint64_t)E;
        }
        if (bad) raise_err(err, EF_BAD_ID);
        key[q] = (d != 0 || id >= (uint64_t)E) ? E : (int)id;
        inv[q] = -1;
        seen[q] = 0;
        kept = d == 0;
    }
    kept = block_sum_256(kept, red);
    if (threadIdx.x == 0 && kept) atomicAdd(ctrl, (uint32_t)kept);
}

__global__ __launch_bounds__(1024) void k_bwd_check_off(const uint64_t *__restrict__ off, int E,
                                                        int Tk, int32_t *__restrict__ off32,
                                                        uint32_t *ctrl, uint32_t *err) {
    bool bad = false;
    for (int e = threadIdx.x; e <= E; e += 1024) {
        const uint64_t v = off[e];
        bad |= v > (uint64_t)Tk || (e == 0 && v != 0) || (e > 0 && off[e - 1] > v);
    }
    bad = __syncthreads_or(bad);
    const uint64_t kept = off[E];
    bad = bad || kept != (uint64_t)ctrl[0];
    for (int e = threadIdx.x; e <= E; e += 1024) off32[e] = bad ? 0 : (int)off[e];
    if (threadIdx.x == 0) {
        ctrl[1] = bad ? 0u : (uint32_t)kept;
        if (bad) raise_err(err, EF_BAD_ID);
    }
}

__global__ __launch_bounds__(256) void k_bwd_check_perm(const uint64_t *__restrict__ perm,
                                                        const uint8_t *__restrict__ drop,
                                                        int Tk, const uint32_t *ctrl,
                                                        uint32_t *__restrict__ seen,
                                                        int32_t *__restrict__ inv,
                                                        uint32_t *err) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= (int)ctrl[1]) return;
    const uint64_t q = perm[i];
    if (q >= (uint64_t)Tk || drop[q] != 0 || atomicAdd(&seen[q], 1u) != 0) {
        raise_err(err, EF_BAD_ID);
        return;
    }
    inv[q] = i;
}

// Row i of the kept rows in perm order: Xp[i] = X[t], dYp[i] =
// (float)((double)w*(double)dY[t]) (src/moe_layer.c:2164-2194), rowq[i] = q.
__global__ __launch_bounds__(256) void k_bwd_gather(const uint64_t *__restrict__ perm,
                                                    const float *__restrict__ X,
                                                    const float *__restrict__ dY,
                                                    const float *__restrict__ w, int Tk, int k,
                                                    int n, const uint32_t *ctrl,
                                                    float *__restrict__ Xp,
                                                    float *__restrict__ dYp,
                                                    int32_t *__restrict__ rowq) {
    const int i = blockIdx.x;
    if (i >= (int)ctrl[1]) return;
    const uint64_t q0 = perm[i];
    const int q = q0 < (uint64_t)Tk ? (int)q0 : 0;
    const int64_t t = q / k;
    const double wv = (double)w[q];
    if (threadIdx.x == 0) rowq[i] = q;
    const float *x = X + t * n, *d = dY + t * n;
    float *xp = Xp + (int64_t)i * n, *dp = dYp + (int64_t)i * n;
    if ((n & 3) == 0 && (((uintptr_t)X | (uintptr_t)dY) & 15) == 0) {
        for (int j = threadIdx.x; j < n / 4; j += 256) {
            const float4 a = ((const float4 *)x)[j], b = ((const float4 *)d)[j];
            ((float4 *)xp)[j] = a;
            ((float4 *)dp)[j] = make_float4((float)(wv * (double)b.x), (float)(wv * (double)b.y),
                                            (float)(wv * (double)b.z), (float)(wv * (double)b.w));
        }
        return;
    }
    for (int j = threadIdx.x; j < n; j += 256) {
        xp[j] = x[j];
        dp[j] = (float)(wv * (double)d[j]);
    }
}

__device__ __forceinline__ float quad_xor1(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x),
                                                                 0xB1, 0xf, 0xf, true));
}
__device__ __forceinline__ float quad_xor2(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x),
                                                                 0x4E, 0xf, 0xf, true));
}
__device__ __forceinline__ double quad_xor1(double x) {
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, 0xB1, 0xf, 0xf, true);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0xB1, 0xf, 0xf, true);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ double quad_xor2(double x) {
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, 0x4E, 0xf, 0xf, true);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x4E, 0xf, 0xf, true);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
// v.x .. v.w of the quad's four lanes -> x[i] = element (lane & 3) of lane i
__device__ __forceinline__ void quad_transpose(float4 v, int lq, float (&x)[4]) {
    float s0 = lq & 1 ? v.x : v.y, s1 = lq & 1 ? v.z : v.w;
    s0 = quad_xor1(s0), s1 = quad_xor1(s1);
    const float y0 = lq & 1 ? s0 : v.x, y1 = lq & 1 ? v.y : s0;
    const float y2 = lq & 1 ? s1 : v.z, y3 = lq & 1 ? v.w : s1;
    float u0 = lq & 2 ? y0 : y2, u1 = lq & 2 ? y1 : y3;
    u0 = quad_xor2(u0), u1 = quad_xor2(u1);
    x[0] = lq & 2 ? u0 : y0, x[1] = lq & 2 ? u1 : y1;
    x[2] = lq & 2 ? y2 : u0, x[3] = lq & 2 ? y3 : u1;
}

// dw[q] for every pair, 0 for dropped ones. Four lanes a pair, one for each
// of the sum's four chains over j % 4; with n % 16 == 0 and aligned rows the
// quad reads 64 bytes of a row at a time and transposes them so that lane c
// has the next four values of chain c (products of two floats are exact in
// fp64, so the fused step rounds as the separate one). Bound by reading Ysel:
// 134 MB at 4096 tokens x top-8, n 1024: 47 us (74 without the next 64 values in
// flight; a thread a pair, each lane on its own row: 83).
__global__ __launch_bounds__(256) void k_bwd_dots(const float *__restrict__ Ysel,
                                                  const float *__restrict__ dY,
                                                  const uint8_t *__restrict__ drop, int Tk,
                                                  int k, int n, double *__restrict__ dw,
                                                  uint32_t *err) {
    const int q = blockIdx.x * 64 + (threadIdx.x >> 2), lq = threadIdx.x & 3;
    const bool live = q < Tk && !drop[q];
    const float *y = Ysel + (int64_t)q * n, *d = dY + (int64_t)(q / k) * n;
    double l = 0.0;
    const int n4 = n & ~3;
    if ((n & 15) == 0 && (((uintptr_t)Ysel | (uintptr_t)dY) & 15) == 0) {
        const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        float4 a[2][4], b[2][4];
        auto load = [&](int j0, int p) {
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int j = j0 + 16 * u + 4 * lq;
                a[p][u] = live && j < n ? *(const float4 *)(y + j) : zero;
                b[p][u] = live && j < n ? *(const float4 *)(d + j) : zero;
            }
        };
        auto sums = [&](int p) {
#pragma unroll
            for (int u = 0; u < 4; u++) {
                float x[4], z[4];
                quad_transpose(a[p][u], lq, x);
                quad_transpose(b[p][u], lq, z);
#pragma unroll
                for (int i = 0; i < 4; i++) l = fma((double)x[i], (double)z[i], l);
            }
        };
        load(0, 0);
        for (int j0 = 0; j0 < n; j0 += 128) {  // the next 64 values in flight
            load(j0 + 64, 1);
            sums(0);
            load(j0 + 128, 0);
            sums(1);
        }
    } else if (live) {
        for (int j = lq; j < n4; j += 4) l = l + (double)y[j] * (double)d[j];
    }
    l = l + quad_xor1(l);  // (l0 + l1) + (l2 + l3), in all four lanes
    l = l + quad_xor2(l);
    if (q >= Tk || lq != 0) return;
    if (!live) {
        dw[q] = 0.0;
        return;
    }
    for (int j = n4; j < n; j++) l = l + (double)y[j] * (double)d[j];
    if (!isfinite(l)) raise_err(err, EF_NONFINITE_MID);
    dw[q] = l;
}

// Per token: s = sum_kept (double)w*dw in slot order; dlog[q] =
// (double)w*(dw - s); dLogits[t][id] = (float)dlog; the first two kept slots
// ordered by expert id for the gate-path dX; the token's perm rows in
// ascending order (= experts ascending, then the expert's row order).
__global__ __launch_bounds__(256) void k_bwd_token(
    const uint64_t *__restrict__ ids, const float *__restrict__ w,
    const uint8_t *__restrict__ drop, const double *__restrict__ dw,
    const int32_t *__restrict__ inv, int T, int k, int E, double *__restrict__ dlog,
    float *__restrict__ dLogits, int32_t *__restrict__ gate_e, double *__restrict__ gate_dl,
    int32_t *__restrict__ gate_n, int32_t *__restrict__ tokpos, int32_t *__restrict__ tokcnt,
    uint32_t *err) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= T) return;
    const int64_t q0 = (int64_t)t * k;
    double s = 0.0;
    for (int p = 0; p < k; p++)
        if (!drop[q0 + p]) s = s + (double)w[q0 + p] * dw[q0 + p];
    bool bad = !isfinite(s);
    int es[2] = {0, 0}, nk = 0, c = 0;
    double dl[2] = {0.0, 0.0};
    int32_t *pos = tokpos + q0;
    for (int p = 0; p < k; p++) {
        const int64_t q = q0 + p;
        if (drop[q]) {
            dlog[q] = 0.0;
            continue;
        }
        const uint64_t id0 = ids[q];
        const int id = id0 < (uint64_t)E ? (int)id0 : 0;
        if (id0 >= (uint64_t)E) raise_err(err, EF_BAD_ID);
        const double v = (double)w[q] * (dw[q] - s);
        bad |= !isfinite(v);
        dlog[q] = v;
        if (dLogits) dLogits[(int64_t)t * E + id] = (float)v;
        if (nk < 2) {
            es[nk] = id;
            dl[nk] = v;
            nk++;
        }
        const int i = inv[q];
        if (i >= 0) {  // insertion into the ascending list
            int at = c++;
            while (at > 0 && pos[at - 1] > i) {
                pos[at] = pos[at - 1];
                at--;
            }
            pos[at] = i;
        }
    }
    if (bad) raise_err(err, EF_NONFINITE_MID);
    if (nk == 2 && es[0] > es[1]) {
        const int te = es[0];
        const double td = dl[0];
        es[0] = es[1], dl[0] = dl[1];
        es[1] = te, dl[1] = td;
    }
    gate_e[2 * t] = es[0];
    gate_e[2 * t + 1] = es[1];
    gate_dl[2 * t] = dl[0];
    gate_dl[2 * t + 1] = dl[1];
    gate_n[t] = nk;
    tokcnt[t] = c;
}

// dWgate[e][j] = float sum over the kept pairs of expert e in flattened
// index order of (float)(dlog*(double)X[t][j]); 0 for experts without one.
// 64 columns a block; the pairs' rows and dlog go through LDS 256 at a time,
// and 32 rows' values are loaded ahead of the (ordered) sums, so a batch costs
// one load latency, not the three of pair, dlog and row (4096 tokens x top-8,
// 64 experts, n 1024: 32 us, 65 with 16 rows a batch from global indices).
__global__ __launch_bounds__(64) void k_bwd_dwgate(const int32_t *__restrict__ off2,
                                                   const int32_t *__restrict__ perm2,
                                                   const double *__restrict__ dlog,
                                                   const float *__restrict__ X, int k, int n,
                                                   float *__restrict__ dWgate) {
    __shared__ int rows[256];
    __shared__ double dls[256];
    const int e = blockIdx.x, j = blockIdx.y * 64 + threadIdx.x, jc = min(j, n - 1);
    float rg = 0.0f;
    const int i0 = off2[e], i1 = off2[e + 1];
    for (int b = i0; b < i1; b += 256) {
        const int m = min(256, i1 - b);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 256; u += 64) {
            const int i = u + threadIdx.x;
            if (i < m) {
                const int q = perm2[b + i];
                rows[i] = q / k;
                dls[i] = dlog[q];
            }
        }
        __syncthreads();
        int i = 0;
        for (; i + 32 <= m; i += 32) {
            float x[32];
#pragma unroll
            for (int u = 0; u < 32; u++) x[u] = X[(int64_t)rows[i + u] * n + jc];
#pragma unroll
            for (int u = 0; u < 32; u++) rg = rg + (float)(dls[i + u] * (double)x[u]);
        }
        for (; i < m; i++) rg = rg + (float)(dls[i] * (double)X[(int64_t)rows[i] * n + jc]);
    }
    if (j < n) dWgate[(int64_t)e * n + j] = rg;
}

// dX[t][j] = (float)(0 + gate term + routed rows in ascending perm order +
// shared experts in index order), all in fp64.
__global__ __launch_bounds__(256) void k_bwd_dx(
    const float *__restrict__ Wgate, const int32_t *__restrict__ gate_e,
    const double *__restrict__ gate_dl, const int32_t *__restrict__ gate_n,
    const int32_t *__restrict__ tokpos, const int32_t *__restrict__ tokcnt,
    const float *__restrict__ Dxe, const float *__restrict__ SDxe, int S, int T, int k, int n,
    float *__restrict__ dX, uint32_t *err) {
    const int t = blockIdx.x, nk = gate_n[t], c = tokcnt[t];
    const int32_t *pos = tokpos + (int64_t)t * k;
    if ((n & 3) == 0 && (((uintptr_t)Wgate | (uintptr_t)dX) & 15) == 0) {
        // four columns a thread with 16-byte loads
        const int j = blockIdx.y * 256 + threadIdx.x;
        if (4 * j >= n) return;
        double acc[4] = {}, dx[4] = {};
        auto add = [](double (&s)[4], double m, float4 v) {
            s[0] = s[0] + m * (double)v.x, s[1] = s[1] + m * (double)v.y;
            s[2] = s[2] + m * (double)v.z, s[3] = s[3] + m * (double)v.w;
        };
        auto row = [&](const float *p, int64_t r) { return ((const float4 *)(p + r * n))[j]; };
        for (int a = 0; a < nk; a++)
            add(acc, gate_dl[2 * t + a], row(Wgate, gate_e[2 * t + a]));
#pragma unroll
        for (int i = 0; i < 4; i++) dx[i] = dx[i] + acc[i];
        int u = 0;
        for (; u + 4 <= c; u += 4) {  // four rows in flight
            float4 v[4];
#pragma unroll
            for (int q = 0; q < 4; q++) v[q] = row(Dxe, pos[u + q]);
#pragma unroll
            for (int q = 0; q < 4; q++) add(dx, 1.0, v[q]);
        }
        for (; u < c; u++) add(dx, 1.0, row(Dxe, pos[u]));
        for (int s = 0; s < S; s++) add(dx, 1.0, row(SDxe, (int64_t)s * T + t));
        if (!isfinite(dx[0]) || !isfinite(dx[1]) || !isfinite(dx[2]) || !isfinite(dx[3]))
            raise_err(err, EF_NONFINITE_MID);
        ((float4 *)(dX + (int64_t)t * n))[j] =
            make_float4((float)dx[0], (float)dx[1], (float)dx[2], (float)dx[3]);
        return;
    }
    // one column a thread (blockIdx.y walks n / 4 columns' worth of threads)
    for (int j = blockIdx.y * 256 + threadIdx.x; j < n; j += gridDim.y * 256) {
        double acc = 0.0;
        for (int a = 0; a < nk; a++)
            acc = acc + gate_dl[2 * t + a] * (double)Wgate[(int64_t)gate_e[2 * t + a] * n + j];
        double dx = 0.0;
        dx = dx + acc;
        for (int u = 0; u < c; u++) dx = dx + (double)Dxe[(int64_t)pos[u] * n + j];
        for (int s = 0; s < S; s++) dx = dx + (double)SDxe[((int64_t)s * T + t) * n + j];
        if (!isfinite(dx)) raise_err(err, EF_NONFINITE_MID);
        dX[(int64_t)t * n + j] = (float)dx;
    }
}

inline unsigned cdiv(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

constexpr int BM_ROWS = 64;  // rows of a routed tile

}  // namespace

// Workspace carve-up (256-byte aligned pieces); returns the total bytes.
extern "C" size_t jtk_bwd_ws_layout(int T, int n, int h, int E, int k, int S, jtk_bwd_ws *w,
                                    char *base) {
    const int64_t Tk = (int64_t)T * k;
    const int64_t NB = (Tk + 255) / 256;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        char *p = base ? base + at : nullptr;
        at += (bytes + 255) / 256 * 256;
        return (void *)p;
    };
    jtk_bwd_ws v;
    v.ctrl = (uint32_t *)take(64);
    v.key = (int32_t *)take(Tk * 4);
    v.inv = (int32_t *)take(Tk * 4);
    v.seen = (uint32_t *)take(Tk * 4);
    v.rowq = (int32_t *)take(Tk * 4);
    v.rank = (int32_t *)take(Tk * 4);
    v.cnt = (int32_t *)take(NB * (E + 1) * 4);
    v.tot = (int32_t *)take(((size_t)E + 1) * 4);
    v.off2 = (int32_t *)take(((size_t)E + 2) * 4);
    v.perm2 = (int32_t *)take(Tk * 4);
    v.off32 = (int32_t *)take(((size_t)E + 1) * 4);
    v.tiles = (int32_t *)take((Tk / BM_ROWS + E + 1) * 16);
    v.ntiles = (int32_t *)take(4);
    v.dw = (double *)take(Tk * 8);
    v.dlog = (double *)take(Tk * 8);
    v.gate_e = (int32_t *)take((size_t)T * 8);
    v.gate_dl = (double *)take((size_t)T * 16);
    v.gate_n = (int32_t *)take((size_t)T * 4);
    v.tokpos = (int32_t *)take(Tk * 4);
    v.tokcnt = (int32_t *)take((size_t)T * 4);
    v.Xp = (float *)take(Tk * n * 4);
    v.dYp = (float *)take(Tk * n * 4);
    v.Dg = (float *)take(Tk * h * 4);
    v.Du = (float *)take(Tk * h * 4);
    v.Ss = (float *)take(Tk * h * 4);
    v.Dxe = (float *)take(Tk * n * 4);
    v.SDg = (float *)take((int64_t)S * T * h * 4);
    v.SDu = (float *)take((int64_t)S * T * h * 4);
    v.SSs = (float *)take((int64_t)S * T * h * 4);
    v.SDxe = (float *)take((int64_t)S * T * n * 4);
    if (w) *w = v;
    return at;
}

extern "C" int jtk_bwd_batch(const jtk_bwd_io *io, int T, int n, int h, int E, int k, int S,
                             int validate, const jtk_bwd_ws *w, uint32_t *err, hipStream_t s) {
    const int Tk = T * k;
    const int64_t nh = (int64_t)n * h;
    int le = 0;
    // index checks
    le |= jtk_zero_u32(w->ctrl, 16, s);
    hipLaunchKernelGGL(k_bwd_check_q, dim3(cdiv(Tk, 256)), dim3(256), 0, s, io->ids,
                       io->weights, io->drop, Tk, E, validate, w->key, w->inv, w->seen, w->ctrl,
                       err);
    hipLaunchKernelGGL(k_bwd_check_off, dim3(1), dim3(1024), 0, s, io->off, E, Tk, w->off32,
                       w->ctrl, err);
    hipLaunchKernelGGL(k_bwd_check_perm, dim3(cdiv(Tk, 256)), dim3(256), 0, s, io->perm,
                       io->drop, Tk, w->ctrl, w->seen, w->inv, err);
    le |= (int)hipGetLastError();
    if (validate) {  // src/moe_layer.c:1766-1800
        FinList L{};
        int c = 0;
        auto add = [&](const float *x, int64_t cnt) {
            L.p[c] = x;
            L.n[c++] = cnt;
        };
        add(io->dY, (int64_t)T * n);
        add(io->X, (int64_t)T * n);
        add(io->Wgate, (int64_t)E * n);
        add(io->Wg, E * nh);
        add(io->Wu, E * nh);
        add(io->Wd, E * nh);
        add(io->weights, Tk);
        add(io->Gsel, (int64_t)Tk * h);
        add(io->Usel, (int64_t)Tk * h);
        add(io->Ysel, (int64_t)Tk * n);
        if (S) {
            add(io->Wg_s, S * nh);
            add(io->Wu_s, S * nh);
            add(io->Wd_s, S * nh);
            add(io->Gs, (int64_t)T * S * h);
            add(io->Us, (int64_t)T * S * h);
        }
        hipLaunchKernelGGL(k_bwd_finite, dim3(1024, (unsigned)c), dim3(256), 0, s, L, err);
        le |= (int)hipGetLastError();
    }
    // gate path
    if (io->dLogits) le |= jtk_zero_u32((uint32_t *)io->dLogits, (int64_t)T * E, s);
    hipLaunchKernelGGL(k_bwd_dots, dim3(cdiv(Tk, 64)), dim3(256), 0, s, io->Ysel, io->dY,
                       io->drop, Tk, k, n, w->dw, err);
    hipLaunchKernelGGL(k_bwd_token, dim3(cdiv(T, 256)), dim3(256), 0, s, io->ids, io->weights,
                       io->drop, w->dw, w->inv, T, k, E, w->dlog, io->dLogits, w->gate_e,
                       w->gate_dl, w->gate_n, w->tokpos, w->tokcnt, err);
    le |= (int)hipGetLastError();
    le |= jtk_sort(w->key, Tk, E + 1, (int64_t)Tk, w->rank, w->cnt, w->tot, w->off2, nullptr,
                   w->perm2, nullptr, nullptr, err, s);
    hipLaunchKernelGGL(k_bwd_dwgate, dim3((unsigned)E, cdiv(n, 64)), dim3(64), 0, s, w->off2,
                       w->perm2, w->dlog, io->X, k, n, io->dWgate);
    // expert rows in perm order
    hipLaunchKernelGGL(k_bwd_gather, dim3((unsigned)Tk), dim3(256), 0, s, io->perm, io->X,
                       io->dY, io->weights, Tk, k, n, w->ctrl, w->Xp, w->dYp, w->rowq);
    le |= (int)hipGetLastError();
    le |= jtk_make_tiles(w->off32, E, BM_ROWS, w->tiles, w->ntiles, s);
    const unsigned mt = (unsigned)(Tk / BM_ROWS + E);  // bound on the routed tile count
    const int mt_sh = (int)cdiv(T, BM_ROWS);
    // row tiles to expect: each expert's last one is half full on average
    const int64_t ex = S * mt_sh + std::max(std::min(E, Tk), Tk / BM_ROWS + E / 2);
    // Dg, Du, S = SwiGLU backward of (rows Wd^T): shared experts on all
    // tokens with dY unweighted, routed experts on their perm rows
    GemmP p{};
    p.err = err, p.N = h, p.nsh = S * mt_sh, p.mt_sh = mt_sh;
    {
        Side &a = p.sd[0];
        a.A[0] = io->dY, a.lda = n;
        a.B[0] = io->Wd_s, a.ldb = n, a.sBg = nh;
        a.C[0] = w->SDg, a.C[1] = w->SDu, a.C[2] = w->SSs, a.ldc = h, a.sCg = (int64_t)T * h;
        a.G = io->Gs, a.U = io->Us, a.ldg = S * h, a.sGg = h;
        a.M = T, a.K = n;
        Side &b = p.sd[1];
        b.A[0] = w->dYp, b.lda = n;
        b.B[0] = io->Wd, b.ldb = n, b.sBg = nh;
        b.C[0] = w->Dg, b.C[1] = w->Du, b.C[2] = w->Ss, b.ldc = h;
        b.G = io->Gsel, b.U = io->Usel, b.rowq = w->rowq, b.ldg = h;
        b.K = n, b.tiles = (const int4 *)w->tiles, b.ntiles = w->ntiles;
    }
    le |= launch_gemm<false, true, EPI_DSWIGLU, MODE_ROWS>(p, p.nsh + mt, 1, ex * cdiv(h, 64), false,
                                                           false, s);
    // dx rows = (float)((double)(Dg Wg) + (double)(Du Wu))
    p = GemmP{};
    p.err = err, p.N = n, p.nsh = S * mt_sh, p.mt_sh = mt_sh;
    {
        Side &a = p.sd[0];
        a.A[0] = w->SDg, a.A[1] = w->SDu, a.lda = h, a.sAg = (int64_t)T * h;
        a.B[0] = io->Wg_s, a.B[1] = io->Wu_s, a.ldb = n, a.sBg = nh;
        a.C[0] = w->SDxe, a.ldc = n, a.sCg = (int64_t)T * n;
        a.M = T, a.K = h;
        Side &b = p.sd[1];
        b.A[0] = w->Dg, b.A[1] = w->Du, b.lda = h;
        b.B[0] = io->Wg, b.B[1] = io->Wu, b.ldb = n, b.sBg = nh;
        b.C[0] = w->Dxe, b.ldc = n;
        b.K = h, b.tiles = (const int4 *)w->tiles, b.ntiles = w->ntiles;
    }
    le |= launch_gemm<false, false, EPI_DUAL, MODE_ROWS>(p, p.nsh + mt, 1, ex * cdiv(n, 64), false,
                                                         false, s);
    // weight gradients D^T rows: dWg = Dg^T X, dWu = Du^T X, dWd = S^T dY
    // (routed: weighted dY rows, over the expert's rows in perm order)
    p = GemmP{};
    p.err = err, p.N = n, p.nsh = 3 * S;
    {
        Side &a = p.sd[0];
        a.A[0] = w->SDg, a.A[1] = w->SDu, a.A[2] = w->SSs, a.lda = h, a.sAg = (int64_t)T * h;
        a.B[0] = io->X, a.B[1] = io->X, a.B[2] = io->dY, a.ldb = n;
        a.C[0] = io->dWg_s, a.C[1] = io->dWu_s, a.C[2] = io->dWd_s, a.ldc = n, a.sCg = nh;
        a.M = h, a.K = T;
        Side &b = p.sd[1];
        b.A[0] = w->Dg, b.A[1] = w->Du, b.A[2] = w->Ss, b.lda = h, b.sAk = h;
        b.B[0] = w->Xp, b.B[1] = w->Xp, b.B[2] = w->dYp, b.ldb = n, b.sBk = n;
        b.C[0] = io->dWg, b.C[1] = io->dWu, b.C[2] = io->dWd, b.ldc = n, b.sCg = nh;
        b.M = h, b.koff = w->off32;
    }
    // A sum over all T tokens (a shared expert's, or one that every token
    // chose) takes T steps of 154 ns with the matrix cores, 123 with 4x4, 92 with
    // 2x4, 61 with 2x2; the chip does a tile's step in 0.33 ns, T * steps of them
    // in all. The forms cross where that says (one shared expert, 4096 tokens: 240
    // steps 2x4 83 us below 4x4 of 1119, 324 equal, 360 43 above of 1409; matrix
    // cores 53 above 4x4 of 1670 at 432 steps, 40 below of 2006 at 540). Without a
    // shared expert 4x4 below 540 unless blocks are few: 2x4 is 18 to 50 us above it
    // with even routing, and if all tokens choose the same experts the matrix cores
    // 122 to 142 above of 1150.
    const int64_t steps = 3LL * (S + k) * cdiv(h, 64) * cdiv(n, 128);
    le |= launch_gemm<true, false, EPI_STORE, MODE_WGRAD>(
        p, h, 3 * (S + E), 3LL * (S + E) * cdiv(h, 64) * cdiv(n, 64), S && steps < 330,
        steps >= 540, s);
    hipLaunchKernelGGL(k_bwd_dx, dim3((unsigned)T, cdiv(n, 1024)), dim3(256), 0, s, io->Wgate,
                       w->gate_e, w->gate_dl, w->gate_n, w->tokpos, w->tokcnt, w->Dxe, w->SDxe,
                       S, T, k, n, io->dX, err);
    le |= (int)hipGetLastError();
    return le;
}

extern "C" int jtk_preload_bwd(void) {
    hipFuncAttributes a;
    return (int)hipFuncGetAttributes(&a, (const void *)(k_bwd_dx));
}
