// Tier-1 split kernel on the fp64 matrix instructions (gfx950): 4, 8 or 16 query rows of one
// (sequence, KV head) share every K and V element a wave loads. It takes the d = 128 steps whose segments
// have 3 or more rows and too few for the int8 prefill kernel (wide GQA groups, draft chains and
// trees) or 1 or 2 rows of few keys, and every other head size.
//
// What bounds it: on gfx950 an fp64 MFMA runs on the vector unit's own fp64 lanes (measured: 16
// MACs per cycle and SIMD for v_mfma_f64_16x16x4 (64 cycles), v_mfma_f64_4x4x4 (17 cycles) and
// v_fma_f64 alike, and an MFMA on one wave does not overlap another wave's VALU work), so the matrix
// forms gain no rate. What they gain is operand reuse: the conversion bf16 -> fp64 of K and V (2.5
// VALU instructions per element) is paid once for all the rows of the block, where ea_decode pays
// it once per 2 rows and ea_split once per 4, and no q operand moves through SGPRs. Per wave and 16
// keys at d = 128 the VALU time is about 700 cycles of conversions, 260 per row for q.k and P.V and
// 25 per pair and lane for the certified weight.
//
// Measured against what ran before (MI355X, equal bits): 8 sequences of 16K keys, 16 rows, d = 128
// 693 -> 226 us (ea_decode, 8 row blocks); 32 ragged sequences to 4K keys, 8 rows 228 -> 82 us;
// 16 ragged sequences to 8K keys, 4 rows, d = 64 157 -> 41 us (ea_split); causal prefill of 2048
// tokens, 32/8 heads, d = 64 2.89 -> 0.65 ms (ea_split). The VALU's own time is 162 of the 226 us
// (16 rows), 102 of 143 us (8 rows, 32 x 4K keys) and 65 of 115 us (4 rows, bound by memory).
//
// The undecided pairs' exact path lives outside the step loop (a list in LDS, flush()): in it, its
// registers spilled the loop's.
//
// Rounding: both instructions accumulate as a chain of four single-rounding FMAs in ascending k
// order (ea_hip_kat_mfma_f64 runs them on given operands, and its test compares them bit for bit with
// fma()), so the bounds are those of
// ea_decode's FMA chains: scores 66 u |q|_1 |k|_inf over at most 64 terms per chain, P.V sums of
// 16 keys per 64-key tile and wave.
//
// Layout. A block is 4 waves over one (segment, row block of RS rows, key range); wave w takes keys
// 16 w .. 16 w + 15 of each 64-key tile and meets the other waves only in the epilogue: there is no
// barrier in the loop. Lane l: x = l / 16, c = l % 16; below 16 rows blk = c / 4, y = c % 4.
//   K     lane (x, c) loads key c, dims 8 (4 j + x) .. + 7 for j < DK: 16 keys x 64 contiguous bytes
//         per instruction; element e of chunk j is the A operand (M = key, K = dim) of one MFMA.
//   q     fp64 in LDS, converted by the block; B operand (K = dim, N = row).
//   S     16 rows: D = keys 4 i + x (i = 0..3) of row c. 4 rows: D = key 4 blk + x of row y, the
//         four blocks of the 4x4x4 form holding 4 keys each; 8 rows are two such sets.
//   W     the weight registers are the A operand of P.V (M = row, K = key) as they stand: 16 rows,
//         register i pairs with keys 4 i + x; 4 rows, the weights rotated by 4 s' lanes within 16
//         (DPP) pair with keys 4 ((blk + s') % 4) + x, so no weight passes through LDS.
//   V     instruction i loads those keys' channels CPL c .. CPL c + CPL - 1; channel e of the lane
//         is the B operand of one MFMA. O: lane (x, c) ends with rows 4 i + x (or 4 s + x),
//         channels CPL c + e: 2 CPL registers per row quad.
// K and V go straight from memory to VGPRs (8 KB in flight per wave).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <type_traits>

#include "ea_params.h"
#include "ea_pf_common.h"

using namespace ea;

namespace {

// 128 x 2 threads: whoever looks for a captured step's fp64 tier-1 node knows it by that width
constexpr int MR_THREADS = 256, MR_BX = 128;
constexpr int MR_NONE = -1200000000;  // reference exponent of a row without a visible key so far
constexpr int MR_HEAD = 64;           // a weight may exceed the row's reference by 2^64 before it moves
constexpr int MR_LIST = 64;
typedef double v4d __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Waves per SIMD each variant is compiled for (512 registers per lane are shared among them), and
// whether it keeps two steps of K and V in registers. A 4-row step is short, so its loads need the
// longer lead: 32 x 4K keys, 4 rows 126 -> 115 us (4.7 TB/s) with two steps at 2 waves, 147 us at 4
// waves, where the registers no longer hold one (scratch reads wait for every load before them). At
// 8 and 16 rows one step is enough (143 and 220 us; 147 and 228 us with two). Non-temporal loads
// cost 50% at 64 dims (a 128-byte line is read by two instructions) and nothing either way at 128.
template <int RS, int DK>
constexpr int mr_waves() { return RS == 16 && DK == 2 ? 3 : 2; }
template <int RS>
constexpr bool mr_two_steps() { return RS == 4; }

template <int RS, int DK, int CPL>
struct MRowSmem {
    static constexpr int QST = DK * 32 + 2;  // doubles per q row: 16 bytes of padding spread the rows over the banks
    double q[RS * QST];
    double T1[256], T2[256];  // exp2 tables, T1 times 2^23
    double red[2][RS * 16 * CPL];
    double q1[RS];            // upper bound of sum |q_i|
    double wZ[4][RS];
    int wR[4][RS], wf[4][RS];  // per wave: reference exponent, flag
    int kvl[RS];               // rows' visible prefixes (rows past the segment: none) and tree masks
    uint64_t tmk[RS];
    float vred[4][16];
    // pairs the score interval left undecided, per wave: (row, key). Flushed when MR_LIST are
    // waiting, so a step's 16 RS more always fit
    int2 list[4][MR_LIST + (mr_two_steps<RS>() ? 32 : 16) * RS];
};

// the larger of x and the values 16, 32 and 48 lanes away (lanes l, l ^ 16, l ^ 32, l ^ 48)
__device__ __forceinline__ int max_x(int v) {
    auto a = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    v = max((int)a[0], (int)a[1]);
    auto b = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    return max((int)b[0], (int)b[1]);
}
template <int CTRL>
__device__ __forceinline__ int dpp(int x) {
    return __builtin_amdgcn_update_dpp(x, x, CTRL, 0xF, 0xF, false);
}
// rotation by 4 s lanes within each 16 lanes: lane (x, blk, y) receives (x, (blk + s) % 4, y)
template <int S>
__device__ __forceinline__ double rot4(double w) {
    if constexpr (S == 0) return w;
    const int lo = dpp<0x120 + 16 - 4 * S>((int)__double2loint(w)), hi = dpp<0x120 + 16 - 4 * S>(__double2hiint(w));
    return __hiloint2double(hi, lo);
}

}  // namespace

template <int RS, int DK, int CPL>
__global__ void __launch_bounds__(MR_THREADS, (mr_waves<RS, DK>())) ea_mrow(Params P) {
    constexpr int NS = RS == 16 ? 1 : RS / 4;  // row sets of the 4x4x4 form
    constexpr int NP = RS / 4;                 // pairs per lane and step
    constexpr int NR = RS == 16 ? 1 : NS;      // rows a lane holds in the score layout
    constexpr int NACC = RS / 4;               // row quads of the output layout
    constexpr bool DB = mr_two_steps<RS>();
    typedef MRowSmem<RS, DK, CPL> Smem;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    Smem& S = *reinterpret_cast<Smem*>(smem_raw);
    const int tid = (int)(threadIdx.x + MR_BX * threadIdx.y);
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int d = P.g.head_dim, dv = P.g.head_dim_v;

    S.T1[tid] = u64_as_f64(EA_T1_BITS[tid]) * 8388608.0;  // 2^23: exact
    S.T2[tid] = u64_as_f64(EA_T2_BITS[tid]);
    if (blockIdx.x == 0 && blockIdx.y == 0) {
        // on uniform splits the step's first kernel clears the tier-2 work list and chunk counts
        if (!P.dq_stream && tid < EA_T2_CNT) P.wl_cnt[tid] = 0;
        if (tid == 0 && P.stats) atomicAdd((unsigned long long*)&P.stats[9], (unsigned long long)P.rows);
        if (tid == 0 && P.stats_x) atomicAdd((unsigned long long*)&P.stats_x[0], (unsigned long long)P.rows);
    }

    // One piece: keys [kA, kB) of unit `item` (segment, row block), clipped to the unit's visible
    // end, as partial slot `split`.
    auto piece = [&](const int item, const int split, const int kA, const int kB) __attribute__((always_inline)) {
        const int lane = tid & 63;
        const int x = lane >> 4, c = lane & 15, blk = c >> 2;
        const int seg = item / P.nrb, rbk = item % P.nrb;
        const int Hkv = P.g.num_kv_heads;
        const int b = seg / Hkv, hk = seg % Hkv;
        const int row0 = rbk * RS;
        const int nrow = min(RS, P.r_seg - row0);
        // ---- q rows to LDS in fp64 (dims past d and rows past the segment are 0), |q| sums
        for (int r = w; r < RS; r += 4) {
            double aq = 0.0;
            if (r < nrow) {
                const int lr = row0 + r, t = lr / P.grp, gi = lr % P.grp;
                const uint16_t* qr = P.q + (int64_t)b * P.g.q_seq_stride + (int64_t)t * P.g.q_tok_stride +
                                     (int64_t)(hk * P.grp + gi) * P.g.q_head_stride;
#pragma unroll
                for (int h = 0; h < DK / 2; ++h) {
                    const int i = lane + 64 * h;
                    const double qv = i < d ? (double)__uint_as_float((uint32_t)qr[i] << 16) : 0.0;
                    S.q[r * Smem::QST + i] = qv;
                    aq += fabs(qv);
                }
            } else {
#pragma unroll
                for (int h = 0; h < DK / 2; ++h) S.q[r * Smem::QST + lane + 64 * h] = 0.0;
            }
            aq = wave_sum(aq);  // at most 128 terms in any order: times 1 + 2^-40 bounds the exact sum
            if (lane == 0) S.q1[r] = aq * (1.0 + 0x1p-40);
        }
        // ---- the rows' visible keys: prefix and tree mask in LDS (steps inside every prefix do not
        // read them), the last visible key and the shortest prefix of the block
        const int slen = P.seq_len[b];
        const int tb = P.tree_mask ? P.tree_base[b] : 0;
        int kend = 0, kvmin = INT_MAX;
        {
            const int r = lane & (RS - 1);
            const int tok = b * P.g.num_tokens + (row0 + min(r, nrow - 1)) / P.grp;
            const int kvl = P.kv_len[tok];
            const uint64_t tmk = P.tree_mask ? P.tree_mask[tok] : 0ull;
            kend = tmk ? max(kvl, tb + 64 - (int)__clzll(tmk)) : kvl;
            kvmin = kvl;
            if (w == 0 && lane < RS) {
                S.kvl[r] = r < nrow ? kvl : INT_MIN;
                S.tmk[r] = r < nrow ? tmk : 0ull;
            }
        }
        kend = min(wave_max_dpp(kend), slen);
        kvmin = min(-wave_max_dpp(-kvmin), slen);
        const int k1 = min(kB, kend);
        const int k0w = kA + 16 * w;  // this wave's keys: k0w + 64 it .. + 15
        const int nst = k1 > k0w ? (k1 - k0w + 63) >> 6 : 0;
        cint_t* btb = (cint_t*)P.bt + (P.bt ? (P.bt_off ? P.bt_off[b] : (int64_t)b * P.g.block_table_stride) : 0);
        const int pshift = P.pshift, pmask = (1 << pshift) - 1;
        const int64_t kps2 = 2 * P.g.k_page_stride, vps2 = 2 * P.g.v_page_stride;
        const int64_t kss2 = 2 * P.g.k_slot_stride, vss2 = 2 * P.g.v_slot_stride;
        const char* const kh = (const char*)(P.k + (int64_t)hk * P.g.k_head_stride);
        const char* const vh = (const char*)(P.v + (int64_t)hk * P.g.v_head_stride);
        // per-lane byte offsets from key n0 of a step; lanes of keys at or past k1, dims past d and
        // channels past dv take EA_OOB: the buffer range check returns zeros without an access
        constexpr int EA_OOB = (int)0x80000000u;
        const int koff = c * (int)kss2 + 16 * x;
        const int ss4 = 4 * (int)vss2;
        const int voff = x * (int)vss2 + 2 * CPL * c;
        // 16 consecutive keys starting at a multiple of 16 lie in one page (page size >= 16)
        auto page_of = [&](int n) __attribute__((always_inline)) { return P.bt ? btb[min(n, k1 - 1) >> pshift] : b; };
        auto issue_k = [&](int n0, int pg, u32x4 (&kr)[DK]) __attribute__((always_inline)) {
            const int64_t sl = P.bt ? (n0 & pmask) : n0;
            const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
                (void*)(kh + (int64_t)pg * kps2 + sl * kss2), (short)0, 0x7FFFFFFF, 0x00020000);
            const int kd = n0 + c < k1 ? d : 0;
#pragma unroll
            for (int j = 0; j < DK; ++j)
                kr[j] = __builtin_amdgcn_raw_buffer_load_b128(rk, 8 * (4 * j + x) < kd ? koff + 64 * j : EA_OOB, 0, 0);
        };
        auto issue_v = [&](int n0, int pg, u32x4 (&vr)[4]) __attribute__((always_inline)) {
            const int64_t sl = P.bt ? (n0 & pmask) : n0;
            const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
                (void*)(vh + (int64_t)pg * vps2 + sl * vss2), (short)0, 0x7FFFFFFF, 0x00020000);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int kq = RS == 16 ? i : (blk + i) & 3;  // the lane's key is 4 kq + x
                const int o = (n0 + 4 * kq + x < k1 && CPL * c < dv) ? voff + kq * ss4 : EA_OOB;
                if constexpr (CPL == 8) {
                    vr[i] = __builtin_amdgcn_raw_buffer_load_b128(rv, o, 0, 0);
                } else {
                    const u32x2 t2 = __builtin_amdgcn_raw_buffer_load_b64(rv, o, 0, 0);
                    vr[i] = (u32x4){t2.x, t2.y, 0u, 0u};
                }
            }
        };

        const double alpha = P.alpha;
        // score bound per pair: |alpha| 66 u |q|_1 max|k| (the last factor per key), with slack for
        // the roundings of the products themselves
        double q1a[NR];
        int R[NR];
        double z[NR];
        int rfl = 0;  // bit s: the lane saw an undecided pair of its row s
        int n5 = 0, n6 = 0, n8 = 0, cnt = 0;  // wave-uniform
        double acc[NACC][CPL];
        v4d acc16[CPL];
#pragma unroll
        for (int e = 0; e < CPL; ++e) {
            acc16[e] = (v4d){0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int i = 0; i < NACC; ++i) acc[i][e] = 0.0;
        }
        float vmx = 0.0f;
        __syncthreads();  // q, its sums and the tables are in LDS
#pragma unroll
        for (int s = 0; s < NR; ++s) {
            q1a[s] = fabs(alpha) * (66.0 * 0x1p-53 * (1.0 + 0x1p-20)) * S.q1[RS == 16 ? c : (c & 3) + 4 * s];
            R[s] = MR_NONE;
            z[s] = 0.0;
        }

        auto step = [&](int n0, int pgn, u32x4 (&kr)[DK], u32x4 (&vr)[4], u32x4 (&kn)[DK], u32x4 (&vn)[4]) __attribute__((always_inline)) {
            if constexpr (DB) {
                issue_k(n0 + 64, pgn, kn);
                issue_v(n0 + 64, pgn, vn);
                __builtin_amdgcn_sched_barrier(0);
            }
            // ---- scores
            double s_[NP];
            float km = 0.0f;
            {
                v4d a16[2] = {(v4d){0.0, 0.0, 0.0, 0.0}, (v4d){0.0, 0.0, 0.0, 0.0}};
                // 4 chains of 4x4x4 products at least: a dependent one waits for its predecessor
                constexpr int NC = RS == 4 ? 4 : 2;
                double a4[NS][NC];
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int q = 0; q < NC; ++q) a4[s][q] = 0.0;
#pragma unroll
                for (int j = 0; j < DK; ++j) {
                    double kf[8];
                    double2 qq[NS][4];
#pragma unroll
                    for (int s = 0; s < NS; ++s)
#pragma unroll
                        for (int h = 0; h < 4; ++h)
                            qq[s][h] = ((const double2*)&S.q[(RS == 16 ? c : (c & 3) + 4 * s) * Smem::QST + 8 * (4 * j + x)])[h];
#pragma unroll
                    for (int h = 0; h < 4; ++h) {
                        const float lo = __uint_as_float(kr[j][h] << 16), hi = __uint_as_float(kr[j][h] & 0xFFFF0000u);
                        km = fmaxf(fmaxf(km, __builtin_fabsf(lo)), __builtin_fabsf(hi));
                        kf[2 * h] = (double)lo;
                        kf[2 * h + 1] = (double)hi;
                    }
#pragma unroll
                    for (int h = 0; h < 4; ++h)
#pragma unroll
                        for (int s = 0; s < NS; ++s) {
                            if constexpr (RS == 16) {
                                a16[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(kf[2 * h], qq[s][h].x, a16[0], 0, 0, 0);
                                a16[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(kf[2 * h + 1], qq[s][h].y, a16[1], 0, 0, 0);
                            } else {
                                constexpr int M2 = NC - 1;
                                double& u0 = a4[s][(2 * h) & M2];
                                u0 = __builtin_amdgcn_mfma_f64_4x4x4f64(kf[2 * h], qq[s][h].x, u0, 0, 0, 0);
                                double& u1 = a4[s][(2 * h + 1) & M2];
                                u1 = __builtin_amdgcn_mfma_f64_4x4x4f64(kf[2 * h + 1], qq[s][h].y, u1, 0, 0, 0);
                            }
                        }
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int p = 0; p < NP; ++p) {
                    if constexpr (RS == 16) s_[p] = a16[0][p] + a16[1][p];
                    else if constexpr (NC == 4) s_[p] = (a4[p][0] + a4[p][1]) + (a4[p][2] + a4[p][3]);
                    else s_[p] = a4[p][0] + a4[p][1];
                }
            }
            // K of the next step into the registers the scores are done with
            if constexpr (!DB) {
                __builtin_amdgcn_sched_barrier(0);
                issue_k(n0 + 64, pgn, kn);
                __builtin_amdgcn_sched_barrier(0);
            }
            // ---- max |k| of the pairs' keys: over the 4 lanes of key c, then from the lane of the key
            const int kmx = max_x(__float_as_int(km));  // non-negative floats order as integers
            double adel[NP];
            uint32_t vism = 0;  // bit p: pair visible
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                const int key = (RS == 16 ? 4 * p : 4 * blk) + x;
                adel[p] = q1a[RS == 16 ? 0 : p] * (double)__int_as_float(__shfl(kmx, key, 64));
                vism |= ((RS == 16 ? c : (c & 3) + 4 * p) < nrow) ? (1u << p) : 0u;
            }
            if (n0 + 16 > min(kvmin, k1)) {
                vism = 0;
#pragma unroll
                for (int p = 0; p < NP; ++p) {
                    const int r = RS == 16 ? c : (c & 3) + 4 * p, n = n0 + (RS == 16 ? 4 * p : 4 * blk) + x, ti = n - tb;
                    const bool in = ((unsigned)ti < 64u) & (((S.tmk[r] >> (ti & 63)) & 1ull) != 0);
                    vism |= ((n < k1) & ((n < S.kvl[r]) | in)) ? (1u << p) : 0u;
                }
            }
            // ---- certified weights
            int M[NP], E[NP];
            bool ok[NP];
            pf::cert_pairs<NP>(s_, adel, alpha, S.T1, S.T2, M, E, ok);
            uint32_t good = 0;
#pragma unroll
            for (int p = 0; p < NP; ++p) good |= ok[p] ? (1u << p) : 0u;
            uint32_t slow = vism & ~good;
            good &= vism;
            if (__builtin_expect(__ballot(slow != 0) != 0, 0)) {
                // undecided pairs (about 1 in 10^5) wait in the wave's list for flush(); a row that
                // is flagged already needs no more of them
#pragma unroll
                for (int p = 0; p < NP; ++p) {
                    const int s = RS == 16 ? 0 : p;
                    const bool put = ((slow >> p) & 1) && !((rfl >> s) & 1);
                    const uint64_t m = __ballot(put);
                    if (put)
                        S.list[w][cnt + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                  __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0))] =
                            make_int2(RS == 16 ? c : (c & 3) + 4 * s, n0 + (RS == 16 ? 4 * p : 4 * blk) + x);
                    cnt += (int)__popcll(m);
                }
            }
            // ---- the reference exponent moves only when a weight passes it by 2^MR_HEAD (or at the
            // row's first key): fp64 has the range, and the usual step then has no reduction
            bool need = false;
#pragma unroll
            for (int p = 0; p < NP; ++p) need |= ((good >> p) & 1) && E[p] + 23 > R[RS == 16 ? 0 : p] + MR_HEAD;
            if (__ballot(need) != 0) {
#pragma unroll
                for (int s = 0; s < NR; ++s) {
                    int m = MR_NONE;
#pragma unroll
                    for (int p = 0; p < NP; ++p)
                        if (RS == 16 || p == s) m = ((good >> p) & 1) ? max(m, E[p] + 23) : m;
                    m = max_x(m);
                    if constexpr (RS != 16) {
                        m = max(m, dpp<0x124>(m));
                        m = max(m, dpp<0x128>(m));
                    }
                    double f = 1.0;
                    if (m > R[s] + MR_HEAD) {
                        if (R[s] != MR_NONE) {
                            const int dsh = R[s] - m;
                            if (dsh < -900) rfl |= 1 << s;
                            f = ldexp(1.0, max(dsh, -1000));
                            z[s] *= f;
                        }
                        R[s] = m;
                    }
                    if constexpr (RS == 16) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const double fi = __shfl(f, 4 * i + x, 64);
#pragma unroll
                            for (int e = 0; e < CPL; ++e) acc16[e][i] *= fi;
                        }
                    } else {
                        const double fi = __shfl(f, x, 64);
#pragma unroll
                        for (int e = 0; e < CPL; ++e) acc[s][e] *= fi;
                    }
                }
            }
            double om[NP];
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                const int s = RS == 16 ? 0 : p;
                const int de = E[p] - R[s];
                const bool g = (good >> p) & 1, far = de < -1000;
                if (g && far) rfl |= 1 << s;
                om[p] = (g && !far) ? ldexp((double)M[p], de) : 0.0;
                z[s] += om[p];
            }
            // ---- P.V
            auto pv = [&](auto ic) __attribute__((always_inline)) {
                __builtin_amdgcn_sched_barrier(0);
                constexpr int i = decltype(ic)::value;
                double wr[NS];
                if constexpr (RS != 16) {
#pragma unroll
                    for (int s = 0; s < NS; ++s) wr[s] = rot4<i>(om[s]);
                }
#pragma unroll
                for (int h = 0; h < CPL / 2; ++h) {
                    const float lo = __uint_as_float(vr[i][h] << 16), hi = __uint_as_float(vr[i][h] & 0xFFFF0000u);
                    vmx = fmaxf(fmaxf(vmx, __builtin_fabsf(lo)), __builtin_fabsf(hi));
                    const double dlo = (double)lo, dhi = (double)hi;
                    if constexpr (RS == 16) {
                        acc16[2 * h] = __builtin_amdgcn_mfma_f64_16x16x4f64(om[i], dlo, acc16[2 * h], 0, 0, 0);
                        acc16[2 * h + 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(om[i], dhi, acc16[2 * h + 1], 0, 0, 0);
                    } else {
#pragma unroll
                        for (int s = 0; s < NS; ++s) {
                            acc[s][2 * h] = __builtin_amdgcn_mfma_f64_4x4x4f64(wr[s], dlo, acc[s][2 * h], 0, 0, 0);
                            acc[s][2 * h + 1] = __builtin_amdgcn_mfma_f64_4x4x4f64(wr[s], dhi, acc[s][2 * h + 1], 0, 0, 0);
                        }
                    }
                }
            };
            pv(std::integral_constant<int, 0>{});
            pv(std::integral_constant<int, 1>{});
            pv(std::integral_constant<int, 2>{});
            pv(std::integral_constant<int, 3>{});
            if constexpr (!DB) {
                __builtin_amdgcn_sched_barrier(0);
                issue_v(n0 + 64, pgn, vn);
                __builtin_amdgcn_sched_barrier(0);
            }
        };

        // ---- the pairs waiting in the list: every product of the score separately, TwoSum-accumulated
        // (a lane per pair), the certified weight, then one pair after another into the row's sums.
        // Out of the step loop, so that its registers do not weigh on the loop's
        auto flush = [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll 1
            for (int at = 0; at < cnt; at += 64) {
                const bool have = at + lane < cnt;
                const int2 en = have ? S.list[w][at + lane] : make_int2(0, 0);
                int32_t Mi = 0, Ei = 0;
                bool live = false;
                int why = 0;  // 1 score not certified, 2 weight not certified
                bool fin = false;
                if (have) {
                    const uint4* kp = (const uint4*)(P.k + kv_off(P, b, en.y, hk, 0));
                    const double* qr = &S.q[en.x * Smem::QST];
                    double ss = 0.0, es = 0.0, ea = 0.0;
#pragma unroll 1
                    for (int ch = 0; 8 * ch < d; ++ch) {
                        const uint4 kv = kp[ch];
                        const uint32_t wd[4] = {kv.x, kv.y, kv.z, kv.w};
#pragma unroll
                        for (int h = 0; h < 4; ++h) {
                            double e0, e1;
                            ss = two_sum(ss, qr[8 * ch + 2 * h] * bf16lo_f64(wd[h]), &e0);
                            ss = two_sum(ss, qr[8 * ch + 2 * h + 1] * bf16hi_f64(wd[h]), &e1);
                            es += e0 + e1;
                            ea += fabs(e0) + fabs(e1);
                        }
                    }
                    uint32_t tbits = 0;
                    int ls = 3;
                    fin = isfinite(ss);
                    if (fin) {
                        ls = (ss == 0.0 && es == 0.0 && ea == 0.0) ? 1 : logit_cert(alpha, ss, es, ea * 0x1p-44, &tbits);
                        if (ls == 1) tbits = 0;
                    }
                    if (ls == 2 || ls == 3) {
                        why = 1;  // undecided, or an overflow (tier 2 reports the domain error)
                    } else if (pf::table_weight(tbits, S.T1, S.T2, &Mi, &Ei)) {
                        live = true;
                    } else {
                        int64_t E2 = 0;
                        live = weight_wide(tbits, &Mi, &E2) == 0 && E2 > -(1LL << 30) && E2 < (1LL << 30);
                        if (!live) why = 2;
                        Ei = (int32_t)E2;
                    }
                }
                n5 += (int)__popcll(__ballot(why == 1));
                n6 += (int)__popcll(__ballot(why == 2));
                n8 += (int)__popcll(__ballot(fin));
                // rows of the lane: bit s of rfl is set in every lane that holds the row
                auto flag_row = [&](int r) __attribute__((always_inline)) {
                    if (RS == 16 ? c == r : (c & 3) == (r & 3)) rfl |= RS == 16 ? 1 : 1 << (r >> 2);
                };
                for (uint64_t m = __ballot(have && !live); m; m &= m - 1)
                    flag_row(__builtin_amdgcn_readlane(en.x, __builtin_ctzll(m)));
                for (uint64_t m = __ballot(live); m; m &= m - 1) {
                    const int l = __builtin_ctzll(m);
                    const int r = __builtin_amdgcn_readlane(en.x, l), n = __builtin_amdgcn_readlane(en.y, l);
                    const int Mr = __builtin_amdgcn_readlane(Mi, l), Er = __builtin_amdgcn_readlane(Ei, l);
                    const bool mine = RS == 16 ? c == r : (c & 3) == (r & 3);  // score layout
                    const bool acc_mine = x == (r & 3);                        // output layout, quad r / 4
                    double f = 1.0;
                    int Rr = MR_NONE;
#pragma unroll
                    for (int s = 0; s < NR; ++s)
                        if (RS == 16 || s == (r >> 2)) {
                            Rr = __builtin_amdgcn_readlane(R[s], RS == 16 ? r : (r & 3));
                            if (Er + 23 > Rr + MR_HEAD) {
                                if (Rr != MR_NONE) {
                                    if (Rr - (Er + 23) < -900) flag_row(r);
                                    f = ldexp(1.0, max(Rr - (Er + 23), -1000));
                                }
                                Rr = Er + 23;
                                if (mine) {
                                    R[s] = Rr;
                                    z[s] *= f;
                                }
                            }
                        }
                    const int de = Er - Rr;
                    if (de < -1000) flag_row(r);
                    const double om = de < -1000 ? 0.0 : ldexp((double)Mr, de);
#pragma unroll
                    for (int s = 0; s < NR; ++s)
                        if (RS == 16 || s == (r >> 2)) z[s] += (mine && x == 0 && (RS == 16 || blk == 0)) ? om : 0.0;
                    uint32_t vd[4] = {0, 0, 0, 0};
                    if (acc_mine && CPL * c < dv) {
                        const uint2* vp = (const uint2*)(P.v + kv_off(P, b, n, hk, 1) + CPL * c);
                        const uint2 v0 = vp[0];
                        vd[0] = v0.x;
                        vd[1] = v0.y;
                        if constexpr (CPL == 8) {
                            const uint2 v1 = vp[1];
                            vd[2] = v1.x;
                            vd[3] = v1.y;
                        }
                    }
                    const double fa = acc_mine ? f : 1.0, oa = acc_mine ? om : 0.0;
#pragma unroll
                    for (int i = 0; i < NACC; ++i) {
                        if (i != (r >> 2)) continue;
#pragma unroll
                        for (int e = 0; e < CPL; ++e) {
                            const double v = (e & 1) ? bf16hi_f64(vd[e >> 1]) : bf16lo_f64(vd[e >> 1]);
                            if constexpr (RS == 16) acc16[e][i] = __fma_rn(oa, v, acc16[e][i] * fa);
                            else acc[i][e] = __fma_rn(oa, v, acc[i][e] * fa);
                        }
                    }
                }
            }
            cnt = 0;
        };

        // ---- the wave's steps: K of the next one is requested once the scores have read this one's
        // registers, V once P.V has; pages are looked up a step ahead. A flush (rare) drops the
        // loads in flight, so that their registers are not live across it, and starts over
        for (int it = 0; it < nst;) {
            u32x4 ka[DK], va[4], kb[DK], vb[4];
            int pg = page_of(k0w + 64 * it);
            issue_k(k0w + 64 * it, pg, ka);
            issue_v(k0w + 64 * it, pg, va);
            pg = page_of(k0w + 64 * it + 64);
#pragma unroll 1
            for (; it < nst && cnt < MR_LIST; it += DB ? 2 : 1) {
                const int n0 = k0w + 64 * it;
                int pgn = pg;
                pg = page_of(n0 + 128);
                if constexpr (DB) {
                    step(n0, pgn, ka, va, kb, vb);
                    pgn = pg;
                    pg = page_of(n0 + 192);
                    if (it + 1 < nst) step(n0 + 64, pgn, kb, vb, ka, va);
                } else {
                    step(n0, pgn, ka, va, ka, va);
                }
            }
            if (cnt > 0) flush();
        }

        // ---- epilogue: row totals of the wave, then the 4 waves' partials at the rows' largest
        // reference exponent (exact powers of two), two additions deep
#pragma unroll
        for (int s = 0; s < NR; ++s) {
            double zs = z[s];
            int fl = (rfl >> s) & 1;
            if constexpr (RS != 16) {
                zs += __shfl_xor(zs, 4, 64);
                fl |= __shfl_xor(fl, 4, 64);
                zs += __shfl_xor(zs, 8, 64);
                fl |= __shfl_xor(fl, 8, 64);
            }
            zs += __shfl_xor(zs, 16, 64);
            fl |= __shfl_xor(fl, 16, 64);
            zs += __shfl_xor(zs, 32, 64);
            fl |= __shfl_xor(fl, 32, 64);
            if (RS == 16 ? x == 0 : (x == 0 && blk == 0)) {
                const int r = RS == 16 ? c : c + 4 * s;
                S.wR[w][r] = R[s];
                S.wZ[w][r] = zs;
                S.wf[w][r] = fl;
            }
        }
        vmx = __int_as_float(max_x(__float_as_int(vmx)));
        if (x == 0) S.vred[w][c] = vmx;
        __syncthreads();
        int far4 = 0;  // bit i: row 4 i + x spans more than 2^900 over the waves
#pragma unroll
        for (int i = 0; i < NACC; ++i) {
            const int r = 4 * i + x;
            int Rm = MR_NONE;
            for (int ww = 0; ww < 4; ++ww) Rm = max(Rm, S.wR[ww][r]);
            const int Rw = S.wR[w][r];
            const double f = Rw == MR_NONE ? 1.0 : ldexp(1.0, max(Rw - Rm, -1000));
            if (Rw != MR_NONE && Rw - Rm < -900) far4 |= 1 << i;
#pragma unroll
            for (int e = 0; e < CPL; ++e) {
                if constexpr (RS == 16) acc[i][e] = acc16[e][i] * f;
                else acc[i][e] *= f;
            }
            if (far4 >> i & 1 && c == 0) S.wf[w][r] = 1;
        }
        auto put = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NACC; ++i)
#pragma unroll
                for (int e = 0; e < CPL; ++e) S.red[buf][(4 * i + x) * (16 * CPL) + e * 16 + c] = acc[i][e];
        };
        auto add = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NACC; ++i)
#pragma unroll
                for (int e = 0; e < CPL; ++e) acc[i][e] += S.red[buf][(4 * i + x) * (16 * CPL) + e * 16 + c];
        };
        if (w >= 2) put(w - 2);
        __syncthreads();
        if (w < 2) add(w);
        __syncthreads();
        if (w == 1) put(0);
        __syncthreads();
        const int64_t pbase = (int64_t)split * P.rows;
        if (w == 0) {
            add(0);
#pragma unroll
            for (int i = 0; i < NACC; ++i) {
                const int r = 4 * i + x;
                if (r >= nrow || CPL * c >= dv) continue;
                const int lr = row0 + r;
                const int64_t gr = row_index(P, b, lr / P.grp, hk * P.grp + lr % P.grp);
                double2* o = (double2*)(P.pN + (pbase + gr) * dv + CPL * c);
#pragma unroll
                for (int e = 0; e < CPL; e += 2) o[e / 2] = make_double2(acc[i][e], acc[i][e + 1]);
            }
        } else if (w == 1) {
            if (lane < nrow) {
                const int r = lane;
                int Rm = MR_NONE, fl = 0;
                for (int ww = 0; ww < 4; ++ww) {
                    Rm = max(Rm, S.wR[ww][r]);
                    fl |= S.wf[ww][r];
                }
                // keys of the piece up to the row's last visible one: at least the keys summed
                const uint64_t tm = S.tmk[r];
                const int ke = min(tm ? max(S.kvl[r], tb + 64 - (int)__clzll(tm)) : S.kvl[r], k1);
                const int n = Rm == MR_NONE ? 0 : ke - kA;
                double zs[4];
                for (int ww = 0; ww < 4; ++ww)
                    zs[ww] = S.wR[ww][r] == MR_NONE ? 0.0 : ldexp(S.wZ[ww][r], max(S.wR[ww][r] - Rm, -1000));
                const int lr = row0 + r;
                const int64_t o = pbase + row_index(P, b, lr / P.grp, hk * P.grp + lr % P.grp);
                P.pR[o] = Rm == MR_NONE ? INT_MIN : Rm;
                P.pZ[o] = (zs[0] + zs[2]) + (zs[1] + zs[3]);
                P.pn[o] = fl ? -1 : n;
            }
        } else if (w == 2) {
            for (int ch = lane; ch < dv; ch += 64) {
                const int q = ch / CPL;
                P.pV[(((int64_t)split * P.nseg + seg) * P.nrb + rbk) * dv + ch] =
                    fmaxf(fmaxf(S.vred[0][q], S.vred[1][q]), fmaxf(S.vred[2][q], S.vred[3][q]));
            }
        }
        if (P.stats && lane == 0) {
            if (n5) atomicAdd((unsigned long long*)&P.stats[5], (unsigned long long)n5);
            if (n6) atomicAdd((unsigned long long*)&P.stats[6], (unsigned long long)n6);
            if (n8) atomicAdd((unsigned long long*)&P.stats[8], (unsigned long long)n8);
        }
    };

    // One piece per block on uniform splits; on the equal-share plan (Params::dq_*) one per unit its
    // share reaches, read as the decode kernel reads it. A segment's row blocks go to one XCD
    // (ea_decode.hip has both placements and their reasons).
    int u, start, end, share = 1, gb = 0;
    const int32_t* Su = P.dq_plan + 2;
    if (P.dq_stream) {
        gb = (int)blockIdx.x;
        if (P.nrb > 1 && (P.dq_blocks & 7) == 0 && (int64_t)P.dq_units * 8 > P.dq_blocks)
            gb = (gb & 7) * (P.dq_blocks >> 3) + (gb >> 3);
        const int4 rec = ((const int4*)(P.dq_plan + P.dq_rec_off))[gb];
        u = rec.x;
        share = rec.w;
        if (u >= P.dq_units || share <= 0) return;  // past the last share: no tile
        start = gb * share;
        end = min(start + share, P.dq_plan[0]);
    } else {
        u = (int)blockIdx.x;
        if (P.nrb > 1 && (P.nseg & 7) == 0) {
            const int lo = u & 7, hi = u >> 3;
            u = ((hi / P.nrb) * 8 + lo) * P.nrb + hi % P.nrb;
        }
        start = (int)blockIdx.y * (P.split_len >> 6);
        end = start + (P.split_len >> 6);
    }
    for (bool first = true;; first = false) {
        int t0 = start, t1 = end, slot = (int)blockIdx.y;
        if (P.dq_stream) {
            if (start >= end || u >= P.dq_units) break;
            const int su = Su[u], eu = Su[u + 1];
            if (eu <= start) {
                ++u;
                continue;
            }
            slot = gb - su / share;
            t0 = start - su;
            t1 = min(end, eu) - su;
            start = min(end, eu);
            if (slot >= P.nsplit) break;  // share >= dq_min_share keeps every unit within nsplit slots
            if (!first) __syncthreads();  // the previous piece's LDS reads are done
        }
        piece(u, slot, t0 * 64, t1 * 64);
        if (!P.dq_stream) break;
        ++u;
    }
}

namespace {

template <int RS>
const void* mrow_fn(bool small) {
    return small ? (const void*)ea_mrow<RS, 2, 4> : (const void*)ea_mrow<RS, 4, 8>;
}
template <int RS>
size_t mrow_lds(bool small) {
    return small ? sizeof(MRowSmem<RS, 2, 4>) : sizeof(MRowSmem<RS, 4, 8>);
}
// head sizes up to 64 take half the K chunks and 4 channels per lane
bool mrow_small(const Params& P) { return P.g.head_dim <= 64 && P.g.head_dim_v <= 64; }
const void* mrow_fn_for(const Params& P) {
    const bool s = mrow_small(P);
    return P.rb == 4 ? mrow_fn<4>(s) : (P.rb == 8 ? mrow_fn<8>(s) : mrow_fn<16>(s));
}
size_t mrow_lds_for(const Params& P) {
    const bool s = mrow_small(P);
    return P.rb == 4 ? mrow_lds<4>(s) : (P.rb == 8 ? mrow_lds<8>(s) : mrow_lds<16>(s));
}
hipError_t mrow_attrs() {
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        const void* fns[6] = {mrow_fn<4>(false), mrow_fn<8>(false), mrow_fn<16>(false),
                              mrow_fn<4>(true),  mrow_fn<8>(true),  mrow_fn<16>(true)};
        for (const void* f : fns) {
            hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(MRowSmem<16, 4, 8>));
            if (e != hipSuccess) err = e;
        }
    });
    return err;
}
}  // namespace

int ea::ea_mrow_eligible(const Params& P) {
    const ea_geometry& g = P.g;
    if (P.bt && P.pshift < 4) return 0;  // one page lookup per 16 keys
    // 16-byte loads of K rows, loads of CPL channels (8 or 16 bytes) of V rows
    const int cpl = mrow_small(P) ? 4 : 8;
    if (((uintptr_t)P.k & 15) || ((g.k_page_stride | g.k_slot_stride | g.k_head_stride) & 7)) return 0;
    if (((uintptr_t)P.v & (2 * cpl - 1)) || ((g.v_page_stride | g.v_slot_stride | g.v_head_stride | g.head_dim_v) & (cpl - 1)))
        return 0;
    const int64_t lim = (int64_t)1 << 30;
    if (P.rows >= lim || (int64_t)g.max_seq_len + 256 >= lim) return 0;
    if (g.k_slot_stride < 0 || g.v_slot_stride < 0 || 32 * g.k_slot_stride + 256 >= lim || 32 * g.v_slot_stride + 256 >= lim)
        return 0;
    return 1;
}

int ea::ea_mrow_slots(const Params& P, int* slots) {
    // blocks resident on the current device at once, cached per device and kernel
    static std::mutex mu;
    static int cache[64][6] = {};
    hipError_t e = mrow_attrs();
    if (e != hipSuccess) return -100 - (int)e;
    int dev = 0;
    if ((e = hipGetDevice(&dev)) != hipSuccess) return -100 - (int)e;
    const int ki = (P.rb == 4 ? 0 : (P.rb == 8 ? 1 : 2)) + (mrow_small(P) ? 3 : 0);
    std::lock_guard<std::mutex> lk(mu);
    if (dev < 0 || dev >= 64) return -1;
    if (!cache[dev][ki]) {
        int cus = 0, per = 0;
        if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return -100 - (int)e;
        if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, mrow_fn_for(P), MR_THREADS, mrow_lds_for(P))) !=
            hipSuccess)
            return -100 - (int)e;
        cache[dev][ki] = (cus > 0 ? cus : 1) * (per > 0 ? per : 1);
    }
    *slots = cache[dev][ki];
    return 0;
}

int ea::ea_launch_mrow(const Params& P, hipStream_t st) {
    hipError_t e = mrow_attrs();
    if (e != hipSuccess) return -100 - (int)e;
    Params Pc = P;
    void* args[] = {&Pc};
    const dim3 grid = P.dq_stream ? dim3((unsigned)P.dq_blocks) : dim3((unsigned)(P.nseg * P.nrb), (unsigned)P.nsplit);
    e = hipLaunchKernel(mrow_fn_for(P), grid, dim3(MR_BX, MR_THREADS / MR_BX), args, mrow_lds_for(P), st);
    return e == hipSuccess ? 0 : -100 - (int)e;
}
