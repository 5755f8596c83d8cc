// Gated DeltaNet-2 (the reference's src/gdn2.c) on gfx950: the decode step
// and the WY-form prefill chunk, batched over independent heads.
//
// Every output keeps the reference's fp32 operation order (separate
// multiply and add roundings, the same summation chains), so results are
// bit-identical to src/gdn2.c. Both kernels run the columns j of a head's
// state S [dk][dv] in parallel: the reference's update treats each column
// independently once the per-head vectors (normalised q/k, decay products,
// the WY matrices) are known.
//
//  k_gdn2_decode      : one block per head. Checks the head's inputs (a bad
//                       head raises EF_NONFINITE_INPUT and is left as it
//                       was), the two L2 norms (sequential fp64 sums, as
//                       src/gdn2.c:219-250), then per column: decay and the
//                       erase coefficient (pass 1), erase + write + read-out
//                       (pass 2), src/gdn2.c:333-405.
//  k_gdn2_prep        : per (chunk, head), all chunks at once: the check of
//                       the chunk's inputs and everything that does not
//                       depend on the state -- norms, ke, the decay
//                       products, the strictly lower L and the lower P
//                       (src/gdn2.c:537-714), the row weights of the state
//                       update (:768-788).
//  k_gdn2_scan        : per (head, columns), every chunk in order in one
//                       launch: B, the forward substitution, Out and the
//                       state update (:614-680, 716-842).
//  k_gdn2_check, k_gdn2_prep_wide, k_gdn2_cols: the same where a chunk's
//                       rows do not fit in LDS (C * dk > 4096) or the
//                       workspace holds no chunk's records for the scan; the
//                       check also before a prefill in parts.
#include "jt_dev.h"
#include "gemm_w8a8.h"
#include "jt_launch.h"

namespace {

constexpr float GDN2_EPS = 1e-6f;

// 1 / ||x|| as the reference rounds it: fp64 sum of squares in index order,
// fp64 sqrt and divide, then float; *zero when the norm is below eps.
// The loads (element i at x[i*ST]) go out 16 at a time ahead of the ordered
// sum.
template <int ST = 1>
__device__ __forceinline__ float inv_norm(const float *x, int n, bool *zero) {
    double ss = 0.0;
    int i = 0;
    for (; i + 16 <= n; i += 16) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = x[(i + u) * ST];
#pragma unroll
        for (int u = 0; u < 16; u++) ss = ss + (double)v[u] * (double)v[u];
    }
    for (; i < n; i++) ss = ss + (double)x[i * ST] * (double)x[i * ST];
    const double nrm = sqrt(ss);
    *zero = nrm < (double)GDN2_EPS;
    return *zero ? 0.0f : (float)(1.0 / nrm);
}

__device__ __forceinline__ bool bad_vec(const float *x, int n, int tid, int nt) {
    bool bad = false;
    for (int i = tid; i < n; i += nt) bad |= !isfinite(x[i]);
    return bad;
}

__device__ __forceinline__ bool bad_alpha(const float *a, int n, int tid, int nt) {
    bool bad = false;
    for (int i = tid; i < n; i += nt) bad |= !(a[i] >= 0.0f && a[i] <= 1.0f);
    return bad;
}

__device__ __forceinline__ bool bad4(float4 x) {
    return !(isfinite(x.x) && isfinite(x.y) && isfinite(x.z) && isfinite(x.w));
}
__device__ __forceinline__ bool bad_unit4(float4 x) {
    return !(x.x >= 0.0f && x.x <= 1.0f && x.y >= 0.0f && x.y <= 1.0f && x.z >= 0.0f &&
             x.z <= 1.0f && x.w >= 0.0f && x.w <= 1.0f);
}
template <int CTRL>
__device__ __forceinline__ float dpp_f(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x),
                                                                 CTRL, 0xf, 0xf, true));
}
// lane E of each 16-lane row, in every lane of the row (DPP row_newbcast)
template <int E>
__device__ __forceinline__ float row_bcast(float x) {
    return dpp_f<0x150 + E>(x);
}
// the value of lane ^ M within a quad
template <int M>
__device__ __forceinline__ float quad_xor(float x) {
    return dpp_f<M == 1 ? 0xB1 : 0x4E>(x);
}

// LDS: qn, kn, ke, al [dk] (dk <= 1024). One thread per column (blockDim
// = dv rounded up to 64, at most 256). Both passes read the column in
// chunks of 64 rows (then 32, then single rows), all of a chunk's loads
// issued before its ordered arithmetic (measured at 512 heads of 128x128:
// 18.3 us against 20.0 us with chunks of 32 and 20.9 us with 128); pass 2 re-reads the column (from cache) and recomputes the
// decayed value, which is the same product as pass 1's.
__global__ __launch_bounds__(256) void k_gdn2_decode(float *__restrict__ S, float *__restrict__ O,
                                                     const float *__restrict__ q,
                                                     const float *__restrict__ k,
                                                     const float *__restrict__ v,
                                                     const float *__restrict__ b,
                                                     const float *__restrict__ w,
                                                     const float *__restrict__ alpha, int dk,
                                                     int dv, uint32_t *err) {
    __shared__ float qn[1024], kn[1024], ke[1024], al[1024];
    __shared__ float invs[2];
    __shared__ int zeros[2];
    const int h = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
    const float *qh = q + (int64_t)h * dk, *kh = k + (int64_t)h * dk;
    const float *bh = b + (int64_t)h * dk, *ah = alpha + (int64_t)h * dk;
    const float *vh = v + (int64_t)h * dv, *wh = w + (int64_t)h * dv;
    float *Sh = S + (int64_t)h * dk * dv, *Oh = O + (int64_t)h * dv;
    bool bad = bad_vec(qh, dk, tid, nt) || bad_vec(kh, dk, tid, nt) || bad_vec(bh, dk, tid, nt) ||
               bad_vec(ah, dk, tid, nt) || bad_alpha(ah, dk, tid, nt) ||
               bad_vec(vh, dv, tid, nt) || bad_vec(wh, dv, tid, nt);
    if (__syncthreads_or(bad)) {  // fail-closed: this head's S and o untouched
        if (tid == 0) raise_err(err, EF_NONFINITE_INPUT);
        return;
    }
    for (int i = tid; i < dk; i += nt) {  // raw q, k into LDS for the norms
        qn[i] = qh[i];
        kn[i] = kh[i];
        al[i] = ah[i];
    }
    __syncthreads();
    const int kt = nt > 64 ? 64 : 1;  // the k norm on a second wave when there is one
    if (tid == 0 || tid == kt) {
        bool z;
        const float iv = inv_norm(tid ? kn : qn, dk, &z);
        invs[tid ? 1 : 0] = iv;
        zeros[tid ? 1 : 0] = z;
    }
    __syncthreads();
    for (int i = tid; i < dk; i += nt) {
        const float qi = zeros[0] ? 0.0f : qn[i] * invs[0];
        const float ki = zeros[1] ? 0.0f : kn[i] * invs[1];
        qn[i] = qi;
        kn[i] = ki;
        ke[i] = bh[i] * ki;
    }
    __syncthreads();
    for (int j = tid; j < dv; j += nt) {
        const float *col = Sh + j;
        float c = 0.0f, o = 0.0f;
        const float vw = wh[j] * vh[j];
        // rows in chunks of 64, then one of 32, then one at a time; each
        // chunk's loads all issue before its ordered arithmetic
        int i0 = 0;
        for (; i0 + 64 <= dk; i0 += 64) {
            float x[64];
#pragma unroll
            for (int u = 0; u < 64; u++) x[u] = col[(int64_t)(i0 + u) * dv];
#pragma unroll
            for (int u = 0; u < 64; u++) c = c + ke[i0 + u] * (x[u] * al[i0 + u]);
        }
        for (; i0 + 32 <= dk; i0 += 32) {
            float x[32];
#pragma unroll
            for (int u = 0; u < 32; u++) x[u] = col[(int64_t)(i0 + u) * dv];
#pragma unroll
            for (int u = 0; u < 32; u++) c = c + ke[i0 + u] * (x[u] * al[i0 + u]);
        }
        for (; i0 < dk; i0++) c = c + ke[i0] * (col[(int64_t)i0 * dv] * al[i0]);
        auto upd = [&](int i, float xv) {
            float r = xv * al[i] - kn[i] * c;
            r = r + kn[i] * vw;
            Sh[(int64_t)i * dv + j] = r;
            o = o + qn[i] * r;
        };
        i0 = 0;
        for (; i0 + 64 <= dk; i0 += 64) {
            float x[64];
#pragma unroll
            for (int u = 0; u < 64; u++) x[u] = col[(int64_t)(i0 + u) * dv];
#pragma unroll
            for (int u = 0; u < 64; u++) upd(i0 + u, x[u]);
        }
        for (; i0 + 32 <= dk; i0 += 32) {
            float x[32];
#pragma unroll
            for (int u = 0; u < 32; u++) x[u] = col[(int64_t)(i0 + u) * dv];
#pragma unroll
            for (int u = 0; u < 32; u++) upd(i0 + u, x[u]);
        }
        for (; i0 < dk; i0++) upd(i0, col[(int64_t)i0 * dv]);
        Oh[j] = o;
    }
}

// ---- prefill with a chunk's operands in LDS (C * dk <= CHUNK_LDS) ----
//
// Record of one (head, chunk), written by k_gdn2_prep in the order in which
// k_gdn2_scan reads it, so that a wave copies it to LDS with linear 16-byte
// loads and stores (floats; dk padded to nv = scan_blocks(dk) blocks of 16
// with zeros, roles r < C/8: rows 16*(r % (C/16)) + tt of -ke*CF for the first
// C/16 roles, of q*CF for the others, CF the forward decay products):
//   P    [block][s/4][tt][s%4]        16x16 blocks (0,0), (1,0), (1,1) of P
//                                     (C = 16: one block), whole 1-KiB pieces
//   M    [role][i/4][tt][i%4]         operands of the chains over i
//   WG   [i/16][s/4][i%16][s%4]       row weights of the state update
//   L    [block][s/4][tt][s%4]        the same blocks of -L
//   CF   [i]                          the last row's decay products
//   FLAG                              nonzero: a bad value in this chunk
constexpr int CHUNK_LDS = 4096;
// blocks of 16 rows of S: even up to 8, then 16 (C = 16, dk > 128), the
// widths k_gdn2_scan is compiled for
__host__ __device__ constexpr int scan_blocks(int dk) {
    return dk > 128 ? 16 : (dk + 31) / 32 * 2;
}
template <int C>
struct ScanRec {
    static constexpr int R = C / 8;               // roles (waves per column group)
    static constexpr int NB = C == 32 ? 3 : 1;    // 16x16 blocks of L and of P
    static constexpr int M = 256 * NB;            // after P
    static __host__ __device__ constexpr int wg(int nv) { return M + 256 * R * nv; }
    static __host__ __device__ constexpr int l(int nv) { return wg(nv) + 16 * C * nv; }
    static __host__ __device__ constexpr int cf(int nv) { return l(nv) + 256 * NB; }
    static __host__ __device__ constexpr int flag(int nv) { return cf(nv) + 16 * nv; }
    // whole 1-KiB pieces, two halves for each of up to two waves
    static __host__ __device__ constexpr int floats(int nv) {
        return (flag(nv) + 1 + 1023) / 1024 * 1024;
    }
};
// Record of the kernels for larger dk: CF, WI = ke*CF, QI = q*CF, WG, then
// Qn, Kn, KE [C][dk] and L, P [C][C].
__host__ __device__ constexpr int64_t wide_rec_floats(int C, int dk) {
    return 7LL * C * dk + 2LL * C * C;
}
__host__ __device__ constexpr int64_t scan_rec_floats(int C, int dk) {
    const int nv = scan_blocks(dk);
    return C == 32 ? ScanRec<32>::floats(nv) : ScanRec<16>::floats(nv);
}

// Everything of a chunk that does not depend on the state, and the check of
// its inputs: one block per (chunk, head), all chunks of a prefill at once.
// L[t][s] = (ke_t*cum(t,s)).k_s (t > s), P[t][s] = (q_t*cum(t,s)).k_s
// (t >= s), cum(t,s) = alpha_{s+1}*...*alpha_t in that order, each a sum in
// four chains over i % 4 (the tail i >= dk & ~3 into chain 0), then
// (c0+c1)+(c2+c3) (src/gdn2.c:537-714, 768-788).
// A wave forms one 16x16 block of L and P: lane (s, chain) walks its chain
// in i order and, for each i, the block's 16 rows t with the running
// product in a register, 16 + 16 sums in registers. The operands are held
// transposed, [i][t] at a stride of C + 4, so that the 16 rows of an i are
// four 16-byte LDS reads an array (48 4-byte reads an i made the walk wait
// on LDS issue). The waves without a
// block write the decay products and the row weights meanwhile.
template <int C>
__global__ __launch_bounds__(256) void k_gdn2_prep(
    const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ B,
    const float *__restrict__ A, const float *__restrict__ V, const float *__restrict__ W,
    int64_t hk, int64_t hv, int dk, int dv, float *__restrict__ rec, uint32_t *err) {
    typedef ScanRec<C> RL;
    constexpr int LT = C + 4, TB = C / 16;
    extern __shared__ __attribute__((aligned(16))) float pm[];  // a, q, k, e: [16 nv][LT]
    __shared__ float invs[2 * C];
    __shared__ int zeros[2 * C];
    const int c = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const int nv = scan_blocks(dk), Ck = C * dk, Cv = C * dv;
    float *a_l = pm, *q_l = a_l + 16 * nv * LT, *k_l = q_l + 16 * nv * LT;
    float *e_l = k_l + 16 * nv * LT;
    const int64_t at0 = h * hk + (int64_t)c * Ck, vt0 = h * hv + (int64_t)c * Cv;
    const float *Qh = Q + at0, *Kh = K + at0, *Bh = B + at0, *Ah = A + at0;
    const float *Vh = V + vt0, *Wh = W + vt0;
    float *r = rec + ((int64_t)h * gridDim.x + c) * RL::floats(nv);
    bool bad = false;
    // A wave reads 16 rows x 16 values: 64-byte pieces, and its transposed
    // LDS stores fall on distinct banks. Job n: row n % 16 (+ 16 for odd
    // blocks when C = 32), values 4 * (..) .. + 3.
    auto row_of = [&](int n) { return (n & 15) + 16 * ((n >> 6) % TB); };
    auto i4_of = [&](int n) { return ((n >> 4) & 3) + 4 * ((n >> 6) / TB); };
    auto put = [&](float *l, int t, int i4, float4 v) {
        float *d = l + 4 * i4 * LT + t;
        d[0] = v.x, d[LT] = v.y, d[2 * LT] = v.z, d[3 * LT] = v.w;
    };
    const uintptr_t al = (uintptr_t)Qh | (uintptr_t)Kh | (uintptr_t)Bh | (uintptr_t)Ah;
    const bool vec = (dk & 3) == 0 && (al & 15) == 0;
    for (int n0 = tid; n0 < 4 * C * nv; n0 += 1024) {
        float4 qv[4], kv[4], bv[4], av[4];  // every load out before the first use
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int n = n0 + 256 * u, t = row_of(n), i = 4 * i4_of(n), at = t * dk + i;
            qv[u] = kv[u] = bv[u] = av[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (n >= 4 * C * nv || i >= dk) continue;
            if (vec) {
                qv[u] = *(const float4 *)(Qh + at);
                kv[u] = *(const float4 *)(Kh + at);
                bv[u] = *(const float4 *)(Bh + at);
                av[u] = *(const float4 *)(Ah + at);
            } else {
                auto ld = [&](const float *p) {
                    return make_float4(p[at], i + 1 < dk ? p[at + 1] : 0.0f,
                                       i + 2 < dk ? p[at + 2] : 0.0f,
                                       i + 3 < dk ? p[at + 3] : 0.0f);
                };
                qv[u] = ld(Qh), kv[u] = ld(Kh), bv[u] = ld(Bh), av[u] = ld(Ah);
            }
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int n = n0 + 256 * u;
            if (n >= 4 * C * nv) continue;
            put(q_l, row_of(n), i4_of(n), qv[u]);
            put(k_l, row_of(n), i4_of(n), kv[u]);
            put(e_l, row_of(n), i4_of(n), bv[u]);
            put(a_l, row_of(n), i4_of(n), av[u]);
            bad |= bad4(qv[u]) || bad4(kv[u]) || bad4(bv[u]) || bad_unit4(av[u]);
        }
    }
    if ((Cv & 3) == 0 && (((uintptr_t)Vh | (uintptr_t)Wh) & 15) == 0) {
        const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        for (int n0 = tid; n0 < Cv / 4; n0 += 1024) {
            float4 v[4], w[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int n = n0 + 256 * u;
                v[u] = n < Cv / 4 ? ((const float4 *)Vh)[n] : zero;
                w[u] = n < Cv / 4 ? ((const float4 *)Wh)[n] : zero;
            }
#pragma unroll
            for (int u = 0; u < 4; u++) bad |= bad4(v[u]) || bad4(w[u]);
        }
    } else {
        for (int n = tid; n < Cv; n += 256) bad |= !isfinite(Vh[n]) || !isfinite(Wh[n]);
    }
    bad = __syncthreads_or(bad);
    if (tid == 0) {
        r[RL::flag(nv)] = bad ? 1.0f : 0.0f;
        if (bad) raise_err(err, EF_NONFINITE_INPUT);
    }
    // row norms: the q rows on the first wave, the k rows on the second
    if ((tid & 63) < C && tid < 128) {
        const int t = tid & 63, w = tid >> 6;
        bool z;
        invs[w * C + t] = inv_norm<LT>((w ? k_l : q_l) + t, dk, &z);
        zeros[w * C + t] = z;
    }
    __syncthreads();
    for (int n = tid; n < Ck; n += 256) {
        const int t = n % C, l = n / C * LT + t;
        const float kv = zeros[C + t] ? 0.0f : k_l[l] * invs[C + t];
        q_l[l] = zeros[t] ? 0.0f : q_l[l] * invs[t];
        k_l[l] = kv;
        e_l[l] = e_l[l] * kv;
    }
    __syncthreads();
    const int wave = tid >> 6, lane = tid & 63;
    if (wave < RL::NB) {
        // block (tb, sb) of L and P
        const int tb = wave > 0, sb = wave > 1;
        const int sl = lane >> 2, ch = lane & 3;
        float la[16], pa[16];
#pragma unroll
        for (int t = 0; t < 16; t++) la[t] = pa[t] = 0.0f;
        const int dk4 = dk & ~3;
        auto walk = [&](int i) {
            const float kv = k_l[i * LT + 16 * sb + sl];
            const float *ai = a_l + i * LT + 16 * tb;
            const float *ei = e_l + i * LT + 16 * tb, *qi = q_l + i * LT + 16 * tb;
            float cu = 1.0f;
            auto rows = [&](bool tri) {
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const float4 a4 = *(const float4 *)(ai + 4 * u);
                    const float4 e4 = *(const float4 *)(ei + 4 * u);
                    const float4 q4 = *(const float4 *)(qi + 4 * u);
                    const float av[4] = {a4.x, a4.y, a4.z, a4.w};
                    const float ev[4] = {e4.x, e4.y, e4.z, e4.w};
                    const float qv[4] = {q4.x, q4.y, q4.z, q4.w};
#pragma unroll
                    for (int w = 0; w < 4; w++) {
                        const int t = 4 * u + w;
                        // in a diagonal block the product starts after row
                        // s (rows t < s form sums that are not used)
                        const float p = cu * av[w];
                        cu = !tri || t > sl ? p : cu;
                        la[t] = la[t] + (ev[w] * cu) * kv;
                        pa[t] = pa[t] + (qv[w] * cu) * kv;
                    }
                }
            };
            if (tb != sb) {  // the rows s+1 .. 15 before the block
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const float4 a4 = *(const float4 *)(a_l + i * LT + 4 * u);
                    const float av[4] = {a4.x, a4.y, a4.z, a4.w};
#pragma unroll
                    for (int w = 0; w < 4; w++) cu = 4 * u + w > sl ? cu * av[w] : cu;
                }
                rows(false);
            } else {
                rows(true);
            }
        };
        for (int i = ch; i < dk4; i += 4) walk(i);
        if (ch == 0)
            for (int i = dk4; i < dk; i++) walk(i);
        float *Lb = r + RL::l(nv) + 256 * wave, *Pb = r + 256 * wave;
#pragma unroll
        for (int t = 0; t < 16; t++) {  // (c0+c1)+(c2+c3), in all four lanes
            la[t] = la[t] + quad_xor<1>(la[t]);
            la[t] = la[t] + quad_xor<2>(la[t]);
            pa[t] = pa[t] + quad_xor<1>(pa[t]);
            pa[t] = pa[t] + quad_xor<2>(pa[t]);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {  // lane (s, ch) stores rows t = 4u + ch
            const float lv = ch == 0 ? la[4 * u] : ch == 1 ? la[4 * u + 1] : ch == 2 ? la[4 * u + 2] : la[4 * u + 3];
            const float pv = ch == 0 ? pa[4 * u] : ch == 1 ? pa[4 * u + 1] : ch == 2 ? pa[4 * u + 2] : pa[4 * u + 3];
            const int t = 4 * u + ch, at = (sl >> 2) * 64 + t * 4 + (sl & 3);
            Lb[at] = tb != sb || sl < t ? -lv : 0.0f;
            Pb[at] = tb != sb || sl <= t ? pv : 0.0f;
        }
    } else {
        // lane = value i: decay products forward with -ke*CF and q*CF, four
        // rows transposed within each quad into 16-byte stores, then the
        // row weights backward
        const int lq = lane & 3;
        auto store4 = [&](float *m, float (&x)[4]) {
            float s0 = lq & 1 ? x[0] : x[1], s1 = lq & 1 ? x[2] : x[3];
            s0 = quad_xor<1>(s0), s1 = quad_xor<1>(s1);
            const float y0 = lq & 1 ? s0 : x[0], y1 = lq & 1 ? x[1] : s0;
            const float y2 = lq & 1 ? s1 : x[2], y3 = lq & 1 ? x[3] : s1;
            float u0 = lq & 2 ? y0 : y2, u1 = lq & 2 ? y1 : y3;
            u0 = quad_xor<2>(u0), u1 = quad_xor<2>(u1);
            *(float4 *)m = lq & 2 ? make_float4(u0, u1, y2, y3) : make_float4(y0, y1, u0, u1);
        };
        for (int i = (wave - RL::NB) * 64 + lane; i < 16 * nv; i += (4 - RL::NB) * 64) {
            const float *ai = a_l + i * LT, *ei = e_l + i * LT, *qi = q_l + i * LT;
            const float *ki = k_l + i * LT;
            float f = 1.0f;
#pragma unroll
            for (int t = 0; t < C; t += 4) {
                const float4 a4 = *(const float4 *)(ai + t);
                const float4 e4 = *(const float4 *)(ei + t), q4 = *(const float4 *)(qi + t);
                const float f0 = f * a4.x, f1 = f0 * a4.y, f2 = f1 * a4.z, f3 = f2 * a4.w;
                float w[4] = {-(e4.x * f0), -(e4.y * f1), -(e4.z * f2), -(e4.w * f3)};
                float q[4] = {q4.x * f0, q4.y * f1, q4.z * f2, q4.w * f3};
                f = f3;
                // lane lq of the quad: row t + lq, values i & ~3 .. + 3
                float *m = r + RL::M + ((t >> 4) * 4 * nv + (i >> 2)) * 64 + ((t & 15) + lq) * 4;
                store4(m, w);
                store4(m + TB * 256 * nv, q);
            }
            r[RL::cf(nv) + i] = f;
            f = 1.0f;
            float *g = r + RL::wg(nv) + (i >> 4) * 16 * C + (i & 15) * 4;
#pragma unroll
            for (int s = C - 4; s >= 0; s -= 4) {
                const float4 k4 = *(const float4 *)(ki + s), a4 = *(const float4 *)(ai + s);
                const float f3 = f, f2 = f3 * a4.w, f1 = f2 * a4.z, f0 = f1 * a4.y;
                f = f0 * a4.x;
                *(float4 *)(g + (s >> 2) * 64) =
                    make_float4(k4.x * f0, k4.y * f1, k4.z * f2, k4.w * f3);
            }
        }
    }
}

typedef float v4f __attribute__((ext_vector_type(4)));

// x += m[u] * s[u], u ascending: 16 steps of a chain
__device__ __forceinline__ void mac4(float &x, float4 m, float4 s) {
    x = x + m.x * s.x;
    x = x + m.y * s.y;
    x = x + m.z * s.z;
    x = x + m.w * s.w;
}
__device__ __forceinline__ void mac16(float &x, const float4 (&m)[4], const float4 (&s)[4]) {
#pragma unroll
    for (int u = 0; u < 4; u++) mac4(x, m[u], s[u]);
}
// the steps s <= tt of 16 (a lower triangular block's row)
__device__ __forceinline__ void mac16_lower(float &x, const float4 (&m)[4], const float4 (&s)[4],
                                            int tt) {
#pragma unroll
    for (int u = 0; u < 4; u++) {
        float y = x + m[u].x * s[u].x;
        x = tt >= 4 * u ? y : x;
        y = x + m[u].y * s[u].y;
        x = tt >= 4 * u + 1 ? y : x;
        y = x + m[u].z * s[u].z;
        x = tt >= 4 * u + 2 ? y : x;
        y = x + m[u].w * s[u].w;
        x = tt >= 4 * u + 3 ? y : x;
    }
}
// Forward substitution of a 16x16 block, a column per 16-lane row: at step E
// lane E's x is final and goes to the row; lanes tt > E take x + m * x_E. The
// lanes up to E go on with values that are not used; theirs are kept in e.
template <int E>
__device__ __forceinline__ void solve_step(float &x, float &e, float m, int tt) {
    e = tt == E ? x : e;
    x = x + m * row_bcast<E>(x);
}
__device__ __forceinline__ float solve16(float x, const float4 (&m)[4], int tt) {
    float e = x;
    solve_step<0>(x, e, m[0].x, tt);
    solve_step<1>(x, e, m[0].y, tt);
    solve_step<2>(x, e, m[0].z, tt);
    solve_step<3>(x, e, m[0].w, tt);
    solve_step<4>(x, e, m[1].x, tt);
    solve_step<5>(x, e, m[1].y, tt);
    solve_step<6>(x, e, m[1].z, tt);
    solve_step<7>(x, e, m[1].w, tt);
    solve_step<8>(x, e, m[2].x, tt);
    solve_step<9>(x, e, m[2].y, tt);
    solve_step<10>(x, e, m[2].z, tt);
    solve_step<11>(x, e, m[2].w, tt);
    solve_step<12>(x, e, m[3].x, tt);
    solve_step<13>(x, e, m[3].y, tt);
    solve_step<14>(x, e, m[3].z, tt);
    return tt == 15 ? x : e;
}

// The state recurrence over all chunks, in order, in one launch. Each chain
// keeps the reference's order (src/gdn2.c:614-680, 716-842), so the work is
// split over chains only: a column group of 4 columns belongs to C/8 + 2
// waves, and lane (16*jr + tt) of a wave holds, for column jr,
//   phase 1, waves 0 .. C/8-1: row t = 16*(wave % (C/16)) + tt of B (first
//            C/16 waves; starts from w*v) or of Out (the others; from 0):
//            the sum over i of M[t][i] * S[i], M = -WI or QI;
//   phase 2: the forward substitution (I + L) E = B in 16x16 blocks: the
//            solve of a diagonal block by its wave (each step's E_s goes to
//            its row with the multiply's own DPP broadcast), then E of the
//            block through LDS; Out += P E by the last wave;
//   phase 3, the other waves without a solve to do: rows i = 16v + tt of the
//            state: S <- CF S + sum_s WG[s][i] E_s.
// The last two waves also copy the next chunk's record to LDS during phase
// 1, through registers (by LDS-DMA, 60 to 90 cycles of the issuing wave a
// KiB, the copy held the other waves for 800 cycles a chunk or one wave for
// 5000).
// A step of a chain is a multiply and an add (two roundings), and its
// operands come 4 at a time from LDS, the next 16 steps' while the current
// ones run: a row's M, WG, L or P values and the column's S or E values
// (both read by 16 lanes of the wave at once). The chains are serial and
// hold one wave per SIMD with 1024 columns on the chip, so a chunk is bound
// by instruction latency: of 4800 cycles, phase 1 takes 2000 (128 steps of
// two instructions, 9.7 cycles), the two solves 900, phase 3 800, LDS round
// trips and barriers the rest. 8 heads x 4096 tokens of 128x128 in chunks of
// 32: 256 us (with a thread per column for the solve and four barriers a
// chunk: 1142 us).
__host__ __device__ constexpr int scan_threads(int C, int NSUB) {
    return 64 * NSUB * (C / 8 + 2);
}
template <int C, int NV, int NSUB>
__global__ __launch_bounds__(scan_threads(C, NSUB)) void k_gdn2_scan(
    float *__restrict__ S, float *__restrict__ Out, const float *__restrict__ V,
    const float *__restrict__ W, int64_t hv, int nch, int dk, int dv,
    const float *__restrict__ rec, const int *__restrict__ flag) {
    typedef ScanRec<C> RL;
    constexpr int R = RL::R, HB = C / 16;       // phase 1 waves, solver waves
    constexpr int OWN = R + 2 - HB;             // waves that hold state rows
    constexpr int NVO = (NV + OWN - 1) / OWN;   // 16-row blocks of each
    constexpr int recf = RL::floats(NV), SK = 16 * NV + 4, EK = C + 4;
    constexpr int NT = scan_threads(C, NSUB);
    extern __shared__ __attribute__((aligned(1024))) float sm[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sub = wave / (R + 2), role = wave % (R + 2);
    const int tt = lane & 15, jr = lane >> 4;
    const bool solver = role < HB;
    // OWN: no state rows
    const int own = role == 0 ? 0 : role < HB || role > R ? OWN : role - HB + 1;
    // per column group: state [jr][i], E and the phase 1 sums of Out
    // [jr][t]
    constexpr int CGF = 4 * (SK + 2 * EK);
    float *sx = sm + 2 * recf + sub * CGF + jr * SK;
    float *eb = sm + 2 * recf + sub * CGF + 4 * SK + jr * EK, *xb = eb + 4 * EK;
    const int h = blockIdx.x;
    const float *rh = rec + (int64_t)h * nch * recf;
    bool bad = flag && flag[h];
    for (int c = tid; c < nch; c += NT) bad |= rh[(int64_t)c * recf + RL::flag(NV)] != 0.0f;
    if (__syncthreads_or(bad)) return;  // a rejected head keeps its S and Out
    const int j = (blockIdx.y * NSUB + sub) * 4 + jr;  // the lane's column
    // a chunk's record to LDS through registers, PB 1-KiB pieces a helper
    constexpr int PB = recf / 256 / (2 * NSUB);
    static_assert(NSUB <= 2, "the record is padded for four waves");
    v4f pc[PB];
    const int at = ((role - R) * NSUB + sub) * PB * 256 + lane * 4;
    auto fetch = [&](int c) {
        const float *src = rh + (int64_t)min(c, nch - 1) * recf + at;
#pragma unroll
        for (int k = 0; k < PB; k++) pc[k] = *(const v4f *)(src + k * 256);
    };
    auto put = [&](int c) {
        float *dst = sm + (c & 1) * recf + at;
#pragma unroll
        for (int k = 0; k < PB; k++) *(v4f *)(dst + k * 256) = pc[k];
    };
    if (role >= R) {
        fetch(0);
        put(0);
    }
    float *Sh = S + (int64_t)h * dk * dv;
    float so[NVO], x = 0.0f, pv = 0.0f, pw = 0.0f;
#pragma unroll
    for (int u = 0; u < NVO; u++) {
        const int i = 16 * (own + OWN * u) + tt;
        so[u] = own < OWN && j < dv && i < dk ? Sh[(int64_t)i * dv + j] : 0.0f;
        if (own < OWN && i < 16 * NV) sx[i] = so[u];
    }
    const int64_t vrow = (int64_t)h * hv + (int64_t)(16 * role + tt) * dv + j;
    auto load_vw = [&](int c) {
        if (j < dv) {
            pv = V[vrow + (int64_t)c * C * dv];
            pw = W[vrow + (int64_t)c * C * dv];
        }
    };
    if (solver) load_vw(0);
    // phase 3: the wave's state rows
    float4 ev[4], w4[NVO][4];
    auto load_w = [&](const float *rl, int b) {
        const float4 *wg = (const float4 *)(rl + RL::wg(NV)) + tt;
#pragma unroll
        for (int u = 0; u < NVO; u++)
            if (NV % OWN == 0 || own + OWN * u < NV)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    w4[u][q] = wg[(own + OWN * u) * 4 * C + 64 * b + 16 * q];
    };
    auto load_e = [&](int b) {
#pragma unroll
        for (int u = 0; u < 4; u++) ev[u] = *(const float4 *)(eb + 16 * b + 4 * u);
    };
    auto decay = [&](const float *rl) {
#pragma unroll
        for (int u = 0; u < NVO; u++)
            if (NV % OWN == 0 || own + OWN * u < NV) {
                const float cv = rl[RL::cf(NV) + 16 * (own + OWN * u) + tt];
                so[u] = so[u] * cv;
            }
    };
    auto state_sums = [&]() {
#pragma unroll
        for (int u = 0; u < NVO; u++)
            if (NV % OWN == 0 || own + OWN * u < NV) {
                mac16(so[u], w4[u], ev);
                // (not moved behind the next barrier)
                asm volatile("" : "+v"(so[u]));
            }
    };
    auto store_state = [&]() {  // the padded rows stay zero (E may be infinite)
#pragma unroll
        for (int u = 0; u < NVO; u++) {
            const int i = 16 * (own + OWN * u) + tt;
            if (NV % OWN == 0 || own + OWN * u < NV) sx[i] = i < dk ? so[u] : 0.0f;
        }
    };
    // Barriers of a chunk: its record and the state are in LDS; the first
    // block of E and the phase 1 sums of Out are; the second block is.
    if (role > R) {
        const int64_t o0 = (int64_t)h * hv + (int64_t)tt * dv + j;
        for (int c = 0; c < nch; c++) {
            lds_barrier();
            const float4 *pp = (const float4 *)(sm + (c & 1) * recf) + tt;
            fetch(c + 1);
            put(c + 1);
            float4 p4[RL::NB][4];
#pragma unroll
            for (int b = 0; b < RL::NB; b++)
#pragma unroll
                for (int u = 0; u < 4; u++) p4[b][u] = pp[64 * b + 16 * u];
            lds_barrier();
            load_e(0);
            float o[HB];
#pragma unroll
            for (int b = 0; b < HB; b++)
                o[b] = xb[16 * b + tt];
            mac16_lower(o[0], p4[0], ev, tt);
            if constexpr (C == 32) {
                mac16(o[1], p4[1], ev);
                asm volatile("" : "+v"(o[0]), "+v"(o[1]));
                lds_barrier();
                load_e(1);
                mac16_lower(o[1], p4[2], ev, tt);
            }
            if (j < dv) {
#pragma unroll
                for (int b = 0; b < HB; b++)
                    Out[o0 + (int64_t)(c * C + 16 * b) * dv] = o[b];
            }
        }
    } else if (role == R) {
        for (int c = 0; c < nch; c++) {
            lds_barrier();
            const float *rl = sm + (c & 1) * recf;
            fetch(c + 1);
            put(c + 1);
            load_w(rl, 0);
            decay(rl);
            lds_barrier();
            load_e(0);
            state_sums();
            if constexpr (C == 32) {
                load_w(rl, 1);
                lds_barrier();
                load_e(1);
                state_sums();
            }
            store_state();
        }
    } else {
        for (int c = 0; c < nch; c++) {
            lds_barrier();
            const float *rl = sm + (c & 1) * recf;
            const float4 *lp = (const float4 *)(rl + RL::l(NV)) + tt;
            const float4 *m4 = (const float4 *)(rl + RL::M + role * 256 * NV) + tt;
            float4 m[2][4], sv[2][4], b4[4];
            auto load_ms = [&](int v) {
#pragma unroll
                for (int u = 0; u < 4; u++) m[v & 1][u] = m4[16 * (4 * v + u)];
#pragma unroll
                for (int u = 0; u < 4; u++) sv[v & 1][u] = *(const float4 *)(sx + 16 * v + 4 * u);
            };
            load_ms(0);
            x = solver ? pw * pv : 0.0f;
            if (solver && c + 1 < nch) load_vw(c + 1);
            // ---- phase 1 ----
#pragma unroll
            for (int v = 0; v < NV; v++) {
                if (v + 1 < NV) {
                    load_ms(v + 1);
                } else {
                    if (own < OWN) load_w(rl, 0);
                    if (solver) {
#pragma unroll
                        for (int u = 0; u < 4; u++) b4[u] = lp[64 * role + 16 * u];
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                mac16(x, m[v & 1], sv[v & 1]);
                asm volatile("" : "+v"(x));
                __builtin_amdgcn_sched_barrier(0);
            }
            if (C == 32 && role == 1) {  // the last solver
                float4 d4[4];
#pragma unroll
                for (int u = 0; u < 4; u++) d4[u] = lp[128 + 16 * u];
                lds_barrier();
                load_e(0);
                mac16(x, b4, ev);
                eb[16 + tt] = solve16(x, d4, tt);
                lds_barrier();
                continue;
            }
            if (role == 0) {
                eb[tt] = solve16(x, b4, tt);
            } else {
                xb[16 * (role - HB) + tt] = x;
            }
            decay(rl);
            lds_barrier();
            load_e(0);
            state_sums();
            if constexpr (C == 32) {
                load_w(rl, 1);
                lds_barrier();
                load_e(1);
                state_sums();
            }
            store_state();
        }
    }
    if (j >= dv || own >= OWN) return;
#pragma unroll
    for (int u = 0; u < NVO; u++) {
        const int i = 16 * (own + OWN * u) + tt;
        if (i < dk) Sh[(int64_t)i * dv + j] = so[u];
    }
}

// ---- prefill with larger dk: operands read from global memory ----

// flag[h] |= 1 when head h's inputs (nk values of each dk-wide array from
// h*hk, nv of each dv-wide one from h*hv) hold a non-finite value or an
// alpha outside [0,1]; the later kernels leave such a head as it was.
// blockIdx.y = head, blockIdx.x strides over the values; flag zeroed before.
__global__ __launch_bounds__(256) void k_gdn2_check(const float *__restrict__ Q,
                                                    const float *__restrict__ K,
                                                    const float *__restrict__ B,
                                                    const float *__restrict__ A,
                                                    const float *__restrict__ V,
                                                    const float *__restrict__ W, int64_t hk,
                                                    int64_t hv, int nk, int nv,
                                                    int *__restrict__ flag, uint32_t *err) {
    const int h = blockIdx.y;
    const int i0 = blockIdx.x * 256 + threadIdx.x, st = gridDim.x * 256;
    const float *q = Q + h * hk, *k = K + h * hk, *b = B + h * hk, *a = A + h * hk;
    const float *v = V + h * hv, *w = W + h * hv;
    bool bad = false;
    const uintptr_t al = (uintptr_t)q | (uintptr_t)k | (uintptr_t)b | (uintptr_t)a |
                         (uintptr_t)v | (uintptr_t)w;
    if (((nk | nv) & 3) == 0 && (al & 15) == 0) {
        // 16-byte loads, four element groups of each array per thread in flight
        const float4 *q4 = (const float4 *)q, *k4 = (const float4 *)k, *b4 = (const float4 *)b;
        const float4 *a4 = (const float4 *)a, *v4 = (const float4 *)v, *w4 = (const float4 *)w;
#pragma unroll 4
        for (int i = i0; i < nk / 4; i += st)
            bad |= bad4(q4[i]) || bad4(k4[i]) || bad4(b4[i]) || bad_unit4(a4[i]);
#pragma unroll 4
        for (int i = i0; i < nv / 4; i += st) bad |= bad4(v4[i]) || bad4(w4[i]);
    } else {
        for (int i = i0; i < nk; i += st)
            bad |= !isfinite(q[i]) || !isfinite(k[i]) || !isfinite(b[i]) ||
                   !(a[i] >= 0.0f && a[i] <= 1.0f);
        for (int i = i0; i < nv; i += st) bad |= !isfinite(v[i]) || !isfinite(w[i]);
    }
    bad = wave_or_i(bad);
    if (bad && (threadIdx.x & 63) == 0) {
        atomicOr(&flag[h], 1);
        raise_err(err, EF_NONFINITE_INPUT);
    }
}

// Everything of a chunk that does not depend on the state: one block per
// (chunk, head), all chunks of a prefill at once; the arithmetic of
// k_gdn2_prep, thread (t, s, chain) forming its own products from the
// record's Qn, Kn, KE.
__global__ __launch_bounds__(256) void k_gdn2_prep_wide(const float *__restrict__ Q,
                                                        const float *__restrict__ K,
                                                        const float *__restrict__ B,
                                                        const float *__restrict__ A, int64_t hk,
                                                        int C, int dk,
                                                        const int *__restrict__ flag,
                                                        float *__restrict__ rec) {
    __shared__ float invs[64];
    __shared__ int zeros[64];
    __shared__ float part[2][32][32][4];  // [L/P][s][t][chain]
    const int c = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    if (flag[h]) return;
    const int64_t Ck = (int64_t)C * dk;
    const int64_t at0 = h * hk + c * Ck;
    const float *Qh = Q + at0, *Kh = K + at0, *Bh = B + at0, *Ah = A + at0;
    float *r = rec + ((int64_t)h * gridDim.x + c) * wide_rec_floats(C, dk);
    float *CF = r, *WI = CF + Ck, *QI = WI + Ck, *WG = QI + Ck;
    float *L = WG + Ck, *P = L + (int64_t)C * C, *Qn = P + (int64_t)C * C, *Kn = Qn + Ck;
    float *KE = Kn + Ck;
    if (tid < 2 * C) {  // one row norm per thread
        const int t = tid % C;
        bool z;
        invs[tid] = inv_norm((tid < C ? Qh : Kh) + (int64_t)t * dk, dk, &z);
        zeros[tid] = z;
    }
    __syncthreads();
    for (int64_t n = tid; n < Ck; n += 256) {
        const int t = (int)(n / dk);
        const float kv = zeros[C + t] ? 0.0f : Kh[n] * invs[C + t];
        Qn[n] = zeros[t] ? 0.0f : Qh[n] * invs[t];
        Kn[n] = kv;
        KE[n] = Bh[n] * kv;
    }
    __syncthreads();
    for (int i = tid; i < dk; i += 256) {
        float cf = 1.0f;  // alpha_0 * ... * alpha_t, t ascending
        for (int t = 0; t < C; t++) {
            const int64_t n = (int64_t)t * dk + i;
            cf = cf * Ah[n];
            CF[n] = cf;
            WI[n] = KE[n] * cf;
            QI[n] = Qn[n] * cf;
        }
        float sf = 1.0f;  // alpha_{s+1} * ..., accumulated from the end
        for (int s = C - 1; s >= 0; s--) {
            const int64_t n = (int64_t)s * dk + i;
            WG[n] = Kn[n] * sf;
            sf = sf * Ah[n];
        }
    }
    const int dk4 = dk & ~3;
    for (int job = tid; job < 4 * C * C; job += 256) {
        const int ch = job & 3, pr = job >> 2, t = pr / C, s = pr % C;
        if (s > t) continue;
        const float *ks = Kn + (int64_t)s * dk, *qt = Qn + (int64_t)t * dk;
        const float *et = KE + (int64_t)t * dk;
        float lsum = 0.0f, psum = 0.0f;
        auto term = [&](int i) {
            float cu = 1.0f;
            for (int rr = s + 1; rr <= t; rr++) cu = cu * Ah[(int64_t)rr * dk + i];
            lsum = lsum + (et[i] * cu) * ks[i];
            psum = psum + (qt[i] * cu) * ks[i];
        };
        for (int i = ch; i < dk4; i += 4) term(i);
        if (ch == 0)
            for (int i = dk4; i < dk; i++) term(i);
        part[0][s][t][ch] = lsum;
        part[1][s][t][ch] = psum;
    }
    __syncthreads();
    for (int pr = tid; pr < C * C; pr += 256) {
        const int t = pr / C, s = pr % C;
        const float *pl = part[0][s][t], *pp = part[1][s][t];
        L[pr] = s < t ? (pl[0] + pl[1]) + (pl[2] + pl[3]) : 0.0f;
        P[pr] = s <= t ? (pp[0] + pp[1]) + (pp[2] + pp[3]) : 0.0f;
    }
}

// The state recurrence over all chunks, in order, in one launch: one block
// per (head, NC = 256/C columns) -- the columns of S never mix. Per chunk,
// phase 1 thread (t, column) runs the chains over i of
// B_t = vw_t - sum_i WI[t][i] S[i] and Out_t = sum_i QI[t][i] S[i]; phase 2
// the forward substitution (I + L) E = B per column with the column's C
// values in registers; phase 3 Out_t += sum_{s<=t} P[t][s] E_s; phase 4
// thread (i, column) S[i] <- CF[C-1][i] S[i] + sum_s WG[s][i] E_s
// (src/gdn2.c:614-680, 716-842).
template <int C>
__global__ __launch_bounds__(256) void k_gdn2_cols(float *__restrict__ S, float *__restrict__ Out,
                                                   const float *__restrict__ V,
                                                   const float *__restrict__ W, int64_t hv,
                                                   int nch, int dk, int dv,
                                                   const int *__restrict__ flag,
                                                   const float *__restrict__ rec) {
    constexpr int NC = 256 / C;
    __shared__ float G[C][NC], Ob[C][NC];
    const int h = blockIdx.x, j0 = blockIdx.y * NC, tid = threadIdx.x;
    if (flag[h]) return;  // a rejected head keeps its S and Out
    const int64_t Ck = (int64_t)C * dk;
    float *Sh = S + (int64_t)h * dk * dv;
    const int ncol = min(NC, dv - j0);
    const int t = tid / NC, jj = tid % NC, j = j0 + jj;
    const bool live = jj < ncol;
    for (int c = 0; c < nch; c++) {
        const float *r = rec + ((int64_t)h * nch + c) * wide_rec_floats(C, dk);
        const float *CF = r, *WI = CF + Ck, *QI = WI + Ck, *WG = QI + Ck;
        const float *L = WG + Ck, *P = L + C * C;
        const int64_t vo = h * hv + ((int64_t)c * C + t) * dv + j;
        if (live) {
            float g = W[vo] * V[vo];  // vw_t
            float o = 0.0f;
            const float *wi = WI + (int64_t)t * dk, *qi = QI + (int64_t)t * dk;
#pragma unroll 8
            for (int i = 0; i < dk; i++) {
                const float sv = Sh[(int64_t)i * dv + j];
                g = g - wi[i] * sv;
                o = o + qi[i] * sv;
            }
            G[t][jj] = g;
            Ob[t][jj] = o;
        }
        __syncthreads();
        if (tid < ncol) {
            float g[C];
#pragma unroll
            for (int tt = 0; tt < C; tt++) g[tt] = G[tt][tid];
#pragma unroll
            for (int tt = 1; tt < C; tt++)
#pragma unroll
                for (int s = 0; s < tt; s++) g[tt] = g[tt] - L[tt * C + s] * g[s];
#pragma unroll
            for (int tt = 0; tt < C; tt++) G[tt][tid] = g[tt];
        }
        __syncthreads();
        if (live) {
            float o = Ob[t][jj];
            for (int s = 0; s <= t; s++) o = o + P[t * C + s] * G[s][jj];
            Out[vo] = o;
        }
        for (int idx = tid; idx < dk * NC; idx += 256) {
            const int i = idx / NC, cc = idx % NC;
            if (cc >= ncol) continue;
            float *sp = Sh + (int64_t)i * dv + j0 + cc;
            float rv = *sp * CF[(int64_t)(C - 1) * dk + i];
#pragma unroll 8
            for (int s = 0; s < C; s++) rv = rv + WG[(int64_t)s * dk + i] * G[s][cc];
            *sp = rv;
        }
        __syncthreads();
    }
}

}  // namespace

// Workspace of jtk_gdn2_prefill: H flag words (padded to 64 floats) and one
// record per (head, chunk).
static size_t prefill_ws(int H, int T, int C, int64_t rec_floats) {
    const int64_t flags = ((int64_t)H + 63) / 64 * 64;
    return (size_t)(flags + (int64_t)H * (T / C) * rec_floats) * sizeof(float);
}
extern "C" size_t jtk_gdn2_prefill_ws_min(int H, int T, int C, int dk) {
    return prefill_ws(H, T, C, wide_rec_floats(C, dk));
}
// The scan's padded record is the larger one up to dk = 22 (C = 16) and 13
// (C = 32).
extern "C" size_t jtk_gdn2_prefill_ws_bytes(int H, int T, int C, int dk) {
    const int64_t wide = wide_rec_floats(C, dk), scan = scan_rec_floats(C, dk);
    return prefill_ws(H, T, C, (int64_t)C * dk <= CHUNK_LDS && scan > wide ? scan : wide);
}

// H heads, one decode step each. dk, dv in 1..1024.
extern "C" int jtk_gdn2_decode(float *S, float *O, const float *q, const float *k,
                               const float *v, const float *b, const float *w,
                               const float *alpha, int H, int dk, int dv, uint32_t *err,
                               hipStream_t s) {
    if (H <= 0 || dk <= 0 || dv <= 0 || dk > 1024 || dv > 1024) return (int)hipErrorInvalidValue;
    const unsigned nt = (unsigned)(dv >= 256 ? 256 : (dv + 63) / 64 * 64);
    hipLaunchKernelGGL(k_gdn2_decode, dim3((unsigned)H), dim3(nt), 0, s, S, O, q, k, v, b, w,
                       alpha, dk, dv, err);
    return (int)hipGetLastError();
}

template <int C>
static hipError_t launch_prep(const float *Q, const float *K, const float *B, const float *A,
                              const float *V, const float *W, int64_t hk, int64_t hv, int H,
                              int nch, int dk, int dv, float *rec, uint32_t *err,
                              hipStream_t s) {
    auto kern = k_gdn2_prep<C>;
    auto lds = [](int nv) { return (int)sizeof(float) * 4 * 16 * nv * (C + 4); };
    // dynamic LDS above 64 KiB must be enabled per device, once
    static std::atomic<bool> attr_set[64];  // set once per device; a repeat is harmless
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    if (!attr_set[dev]) {
        e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                lds(CHUNK_LDS / C / 16));
        if (e != hipSuccess) return e;
        attr_set[dev] = true;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)nch, (unsigned)H), dim3(256), lds(scan_blocks(dk)), s,
                       Q, K, B, A, V, W, hk, hv, dk, dv, rec, err);
    return hipGetLastError();
}

template <int C, int NV, int NSUB>
static hipError_t launch_scan(float *S, float *Out, const float *V, const float *W, int64_t hv,
                              int H, int nch, int dk, int dv, const float *rec, const int *flag,
                              hipStream_t s) {
    typedef ScanRec<C> RL;
    auto kern = k_gdn2_scan<C, NV, NSUB>;
    constexpr int lds =
        (int)sizeof(float) * (2 * RL::floats(NV) + NSUB * 4 * (16 * NV + 4 + 2 * (C + 4)));
    // dynamic LDS above 64 KiB must be enabled per device, once
    static std::atomic<bool> attr_set[64];  // set once per device; a repeat is harmless
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    if (!attr_set[dev]) {
        e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                lds);
        if (e != hipSuccess) return e;
        attr_set[dev] = true;
    }
    const int cols = 4 * NSUB;
    hipLaunchKernelGGL(kern, dim3((unsigned)H, (unsigned)((dv + cols - 1) / cols)),
                       dim3(scan_threads(C, NSUB)), lds, s, S, Out, V, W, hv, nch, dk, dv, rec,
                       flag);
    return hipGetLastError();
}

// One column group a block while that gives every CU at most one block, else
// two, whose waves share the record and the SIMDs: 32 heads x 2048 tokens of
// 128x128 in chunks of 32 472 us against 618, in chunks of 16 449 against
// 588; at 1024 columns, which two groups a block leave half the CUs without,
// 406 us against 322 (8 heads x 4096 tokens, chunks of 32).
template <int C, int NV>
static hipError_t launch_scan_nv(float *S, float *Out, const float *V, const float *W,
                                 int64_t hv, int H, int nch, int dk, int dv, const float *rec,
                                 const int *flag, hipStream_t s) {
    return (int64_t)H * ((dv + 3) / 4) <= 256
               ? launch_scan<C, NV, 1>(S, Out, V, W, hv, H, nch, dk, dv, rec, flag, s)
               : launch_scan<C, NV, 2>(S, Out, V, W, hv, H, nch, dk, dv, rec, flag, s);
}
template <int C>
static hipError_t launch_scan_c(float *S, float *Out, const float *V, const float *W,
                                int64_t hv, int H, int nch, int dk, int dv, const float *rec,
                                const int *flag, hipStream_t s) {
    switch (scan_blocks(dk)) {
        case 2: return launch_scan_nv<C, 2>(S, Out, V, W, hv, H, nch, dk, dv, rec, flag, s);
        case 4: return launch_scan_nv<C, 4>(S, Out, V, W, hv, H, nch, dk, dv, rec, flag, s);
        case 6: return launch_scan_nv<C, 6>(S, Out, V, W, hv, H, nch, dk, dv, rec, flag, s);
        case 8: return launch_scan_nv<C, 8>(S, Out, V, W, hv, H, nch, dk, dv, rec, flag, s);
        default: break;
    }
    if constexpr (C == 16)
        return launch_scan_nv<C, 16>(S, Out, V, W, hv, H, nch, dk, dv, rec, flag, s);
    else
        return hipErrorInvalidValue;  // not reached: C * dk <= CHUNK_LDS
}

// H heads, T tokens each in T/C chunks of C (16 or 32): head h's rows of
// the dk-wide inputs start at h*hk, of V, W and Out at h*hv. All of a
// head's T tokens are checked first (a head with a bad value keeps its S
// and Out), every chunk's state-independent part is prepared in one
// launch, then one launch runs the chunks' state updates in order. ws of
// at least jtk_gdn2_prefill_ws_min(H, T, C, dk) bytes; where it does not hold
// the scan's records of every chunk the sequence goes in parts of the chunks
// that fit, after a check of all of it (8 heads x 4096 tokens, dk 8, dv 16:
// 215 us in three parts, 194 in one), and with room for no chunk of every head
// the kernels for larger dk take the call. The bits are the same.
extern "C" int jtk_gdn2_prefill(float *S, float *Out, const float *Q, const float *K,
                                const float *V, const float *B, const float *W,
                                const float *A, int64_t hk, int64_t hv, int H, int T, int C,
                                int dk, int dv, float *ws, size_t ws_bytes, uint32_t *err,
                                hipStream_t s) {
    if (H <= 0 || H > 65535 || (C != 16 && C != 32) || T <= 0 || T % C || dk <= 0 || dv <= 0 ||
        dk > 1024 || dv > 1024 || (int64_t)T * (dk > dv ? dk : dv) > INT32_MAX ||
        ws_bytes < jtk_gdn2_prefill_ws_min(H, T, C, dk))
        return (int)hipErrorInvalidValue;
    const int nch = T / C;
    const int64_t flags = ((int64_t)H + 63) / 64 * 64;
    float *rec = ws + flags;
    int *flag = (int *)ws;
    // chunks of every head whose scan records fit
    const int64_t fit = ((int64_t)(ws_bytes / sizeof(float)) - flags) / (H * scan_rec_floats(C, dk));
    const bool scan = (int64_t)C * dk <= CHUNK_LDS && fit > 0;
    int le = 0;
    if (!scan || fit < nch) {  // (in one part the preparation checks, and the scan asks its records)
        le |= jtk_zero_u32((uint32_t *)flag, H, s);
        const int64_t most = (int64_t)T * (dk > dv ? dk : dv);
        const unsigned nb = (unsigned)((most + 255) / 256 < 64 ? (most + 255) / 256 : 64);
        hipLaunchKernelGGL(k_gdn2_check, dim3(nb, (unsigned)H), dim3(256), 0, s, Q, K, B, A, V,
                           W, hk, hv, T * dk, T * dv, flag, err);
    }
    if (scan) {
        const int part = (int)(fit < nch ? fit : nch);
        const int *whole = part < nch ? flag : nullptr;
        for (int c0 = 0; c0 < nch; c0 += part) {
            const int m = part < nch - c0 ? part : nch - c0;
            const int64_t k0 = (int64_t)c0 * C * dk, v0 = (int64_t)c0 * C * dv;
            hipError_t e = C == 32
                ? launch_prep<32>(Q + k0, K + k0, B + k0, A + k0, V + v0, W + v0, hk, hv, H, m,
                                  dk, dv, rec, err, s)
                : launch_prep<16>(Q + k0, K + k0, B + k0, A + k0, V + v0, W + v0, hk, hv, H, m,
                                  dk, dv, rec, err, s);
            if (e != hipSuccess) return (int)e;
            e = C == 32 ? launch_scan_c<32>(S, Out + v0, V + v0, W + v0, hv, H, m, dk, dv, rec,
                                            whole, s)
                        : launch_scan_c<16>(S, Out + v0, V + v0, W + v0, hv, H, m, dk, dv, rec,
                                            whole, s);
            if (e != hipSuccess) return (int)e;
        }
        return le;
    }
    hipLaunchKernelGGL(k_gdn2_prep_wide, dim3((unsigned)nch, (unsigned)H), dim3(256), 0, s, Q,
                       K, B, A, hk, C, dk, flag, rec);
    auto cols = C == 32 ? k_gdn2_cols<32> : k_gdn2_cols<16>;
    hipLaunchKernelGGL(cols, dim3((unsigned)H, (unsigned)((dv + 256 / C - 1) / (256 / C))),
                       dim3(256), 0, s, S, Out, V, W, hv, nch, dk, dv, flag, rec);
    return le | (int)hipGetLastError();
}

// y = x / ||x|| (the reference's l2norm) for R rows of n.
__global__ __launch_bounds__(64) void k_gdn2_l2norm(const float *__restrict__ x,
                                                    float *__restrict__ y, int n, float eps) {
    const int r = blockIdx.x;
    __shared__ float inv;
    __shared__ int zero;
    const float *xr = x + (int64_t)r * n;
    if (threadIdx.x == 0) {
        double ss = 0.0;
        for (int i = 0; i < n; i++) ss = ss + (double)xr[i] * (double)xr[i];
        const double nrm = sqrt(ss);
        zero = nrm < (double)eps;
        inv = zero ? 0.0f : (float)(1.0 / nrm);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 64) y[(int64_t)r * n + i] = zero ? 0.0f : xr[i] * inv;
}

extern "C" int jtk_gdn2_l2norm(const float *x, float *y, int rows, int n, float eps,
                               hipStream_t s) {
    hipLaunchKernelGGL(k_gdn2_l2norm, dim3((unsigned)rows), dim3(64), 0, s, x, y, n, eps);
    return (int)hipGetLastError();
}

extern "C" int jtk_preload_gdn2(void) {
    hipFuncAttributes a;
    return (int)hipFuncGetAttributes(&a, (const void *)(k_gdn2_l2norm));
}
