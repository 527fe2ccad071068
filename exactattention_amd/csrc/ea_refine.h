// Tier 2's first pass: a listed row again in double-double (error-free transformed) fp64.
//
// The tier-1 error bounds are worst cases of about 2^-36 to 2^-40 of the outputs, so final roundings
// fail for 3 to 20% of the rows of an fp32 step (70 of 2048 causal rows, 400 of 2048 decode rows of 4K
// keys) and for one row in 10^5 in bf16. The
// 128-bit path decides them with integer work of some 0.43 ms per 2048-key row and block. Here every
// product is exact in fp64, every sum keeps its rounding errors (TwoSum, errors summed beside it,
// their magnitudes bounded by a third sum), and N / Z is rounded from a residual N - m Z against the
// one midpoint m in reach: the result is left undecided only where N / Z is within about 2^-90 of a
// midpoint. Rows that stay undecided keep flag 1 for the 128-bit path.
//
// A block of 8 waves takes 128 keys at a time: 4 lanes per key for the score (32 dims each), then
// wave v the V rows of keys 16 v .. 16 v + 15, two channels per lane; about 950 VALU instructions per
// wave and pass. The figures are at ea_tier2 (ea_hip.hip).
#pragma once
#include "ea_params.h"
#include "ea_pf_common.h"

namespace ea {

#define EA_DD_THREADS 512
#define EA_DD_WAVES (EA_DD_THREADS / 64)
#define EA_DD_KEYS (EA_DD_THREADS / 4)  // keys per pass
#define EA_DD_PARTS 512                 // chunk partials in flight (C > 1)

// A sum in three parts: hi + lo is the value up to the roundings of lo's own additions, at most
// (number of additions) 2^-53 mag with mag >= the sum of |each TwoSum error|, and up to err, the terms
// left out because their weight is below 2^-120 of the row's reference (the 128-bit path's window).
struct DD {
    double hi, lo, mag, err;
};
constexpr int DD_WINDOW = -120;
__device__ __forceinline__ void dd_add(DD& s, double x) {
    double e;
    s.hi = two_sum(s.hi, x, &e);
    s.lo += e;
    s.mag += fabs(e);
}
__device__ __forceinline__ void dd_join(DD& s, const DD& a, double f = 1.0) {  // f an exact power of two
    dd_add(s, a.hi * f);
    s.lo += a.lo * f;
    s.mag += a.mag * f;
    s.err += a.err * f;
}
__device__ __forceinline__ double dd_size(const DD& a) { return fabs(a.hi) + fabs(a.lo) + a.mag + a.err; }
__device__ __forceinline__ void dd_scale(DD& s, double f) {  // f an exact power of two
    s.hi *= f;
    s.lo *= f;
    s.mag *= f;
    s.err *= f;
}

// One chunk's share of a row whose keys are split over several blocks.
struct DDPart {
    int32_t R, flag;  // reference exponent (DD_NONE: no key); 0, 1 undecided, 2 domain error
    DD z;
    DD n[EA_MAXDV];
};
constexpr int DD_NONE = -1200000000;

// RN(N / Z) of N = n.hi + n.lo, Z = z.hi + z.lo (Z > 0), each with an error of at most adds 2^-53 mag:
// true and the bits when certain.
__device__ inline bool dd_quotient(const DD& n, const DD& z, double adds, int fp32, uint32_t* bits) {
    const double u = 0x1p-53 * (1.0 + 0x1p-20);
    if (n.hi == 0.0 && n.lo == 0.0 && n.mag == 0.0 && n.err == 0.0) {  // an exact zero
        *bits = 0;
        return true;
    }
    const double en = adds * u * n.mag + n.err * (1.0 + 0x1p-20), ez = adds * u * z.mag + z.err * (1.0 + 0x1p-20);
    const double q = (n.hi + n.lo) / (z.hi + z.lo), aq = fabs(q);
    // the quotient alone: 3 roundings and the two errors; |z.hi + z.lo| >= z.hi (1 - 2^-40)
    const double rad = aq * (0x1p-51 + 2.0 * ez / z.hi) + 2.0 * en / z.hi + 0x1p-1060;
    if (!isfinite(q) || !isfinite(rad)) return false;
    if (certify_round(q, rad, fp32, bits)) return true;
    if (!(aq >= 0x1p-125) || !(aq < 0x1p126) || rad > aq * 0x1p-48) return false;
    // m: the midpoint next to q, a number of p + 1 bits (q is within 2^-47 of one, or no midpoint
    // decides and the residual test below fails to be near it)
    const int S = fp32 ? 29 : 45;  // fp64 fraction bits below the format's
    const uint64_t qb = f64_as_u64(aq), half = 1ull << (S - 1);
    const uint64_t mb = (qb & ~((1ull << S) - 1)) | half;
    const double m = u64_as_f64(mb);
    if (fabs(aq - m) > m * 0x1p-46) return false;
    // r = |N| - m Z: m z.hi = p1 + e1 exactly, n - p1 exact (they agree to 2^-40)
    const double sg = q < 0.0 ? -1.0 : 1.0;
    const double p1 = m * z.hi, e1 = __fma_rn(m, z.hi, -p1);
    const double nh = sg * n.hi, nl = sg * n.lo;
    double e0;
    const double d0 = two_sum(nh, -p1, &e0);
    const double rest = ((nl - m * z.lo) - e1) + e0;
    const double r = d0 + rest;
    // the last term covers products here, and parts of the sums scaled down with a row's reference,
    // that fall below the smallest numbers (2^-1074 each)
    const double err = (fabs(d0) + fabs(rest) + fabs(nl) + fabs(m * z.lo) + fabs(e1) + fabs(e0)) * 0x1p-50 + en + m * ez + 0x1p-1000;
    const bool exact = nl == 0.0 && n.mag == 0.0 && n.err == 0.0 && z.lo == 0.0 && z.mag == 0.0 && z.err == 0.0;
    uint64_t k = mb >> S;  // the format's value below the midpoint
    if (exact && d0 == 0.0 && e0 == 0.0 && e1 == 0.0) k += k & 1;  // a tie: to even
    else if (r > err) ++k;
    else if (!(r < -err)) return false;
    const uint32_t mag = (uint32_t)(k - ((uint64_t)(1023 - 127) << (52 - S)));
    *bits = ((q < 0.0 ? 1u : 0u) << (fp32 ? 31 : 15)) | mag;
    return true;
}

// Data that another block of the same launch reads: stores and loads at agent scope, and the wait that
// completes a wave's stores
__device__ __forceinline__ void agent_store(int32_t* p, int32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int32_t agent_load(int32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void agent_store(DD* p, const DD& v) {
    __hip_atomic_store(&p->hi, v.hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&p->lo, v.lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&p->mag, v.mag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&p->err, v.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ DD agent_load(DD* p) {
    DD v;
    v.hi = __hip_atomic_load(&p->hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v.lo = __hip_atomic_load(&p->lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v.mag = __hip_atomic_load(&p->mag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v.err = __hip_atomic_load(&p->err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return v;
}
__device__ __forceinline__ void agent_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

struct DDSmem {
    double T1[256], T2[256];  // T1 times 2^23
    double q[EA_MAXD];
    int32_t M[EA_DD_KEYS], E[EA_DD_KEYS];
    DD red[EA_DD_WAVES][EA_MAXDV];
    DD zred[EA_DD_WAVES];
    int32_t pR[EA_DD_PARTS];
    DD pz[EA_DD_PARTS];
    int32_t mx, flag, last;
};

// The listed rows, in grid-stride order; C chunks per row (C > 1 only with rows C <= EA_DD_PARTS and
// rows C <= gridDim.x). parts: EA_DD_PARTS partials. Certified rows get their output and flag 0,
// rows with a domain error flag 2; the rest are listed in P.t2left, P.wl_cnt[EA_T2_LEFT] of them.
__device__ inline void dd_rows(const Params& P, DDSmem& S, int cnt, int C, DDPart* parts) {
    const int tid = (int)threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int d = P.g.head_dim, dv = P.g.head_dim_v, Hq = P.g.num_q_heads, T = P.g.num_tokens;
    if (tid < 256) {
        S.T1[tid] = u64_as_f64(EA_T1_BITS[tid]) * 8388608.0;
        S.T2[tid] = u64_as_f64(EA_T2_BITS[tid]);
    }
    const bool k16 = (((uintptr_t)P.k | (uintptr_t)(2 * P.g.k_page_stride) | (uintptr_t)(2 * P.g.k_slot_stride) |
                       (uintptr_t)(2 * P.g.k_head_stride)) & 15) == 0;
    const bool v4 = (((uintptr_t)P.v | (uintptr_t)(2 * P.g.v_page_stride) | (uintptr_t)(2 * P.g.v_slot_stride) |
                      (uintptr_t)(2 * P.g.v_head_stride)) & 3) == 0;  // dv is even
    const int64_t items = (int64_t)cnt * C;
    for (int64_t item = blockIdx.x; item < items; item += gridDim.x) {
        const int slot = (int)(item / C), chunk = (int)(item % C);
        const int64_t row = P.wl[slot];
        const int64_t b = row / ((int64_t)T * Hq);
        const int t = (int)((row / Hq) % T), hq = (int)(row % Hq), hk = hq / P.grp;
        const int64_t tok = b * T + t;
        const int64_t slen = P.seq_len[b], L = vis_prefix(P.kv_len[tok], slen);
        const int64_t tb = P.tree_mask ? P.tree_base[b] : 0;
        const uint64_t mask = P.tree_mask ? vis_tree_bits(P.tree_mask[tok], tb, L, slen) : 0ull;
        const int64_t nkeys = L + __popcll(mask);
        const int64_t csz = (nkeys + C - 1) / C;
        const int64_t jc0 = min(nkeys, (int64_t)chunk * csz), jc1 = min(nkeys, jc0 + csz);
        auto key_n = [&](int64_t j) -> int64_t {
            if (j < L) return j;
            uint64_t m = mask;
            for (int64_t cc = j - L; cc > 0; --cc) m &= m - 1;
            return tb + (__ffsll((long long)m) - 1);
        };
        __syncthreads();  // the previous row's LDS reads are done
        if (tid == 0) {
            S.flag = 0;
            S.mx = DD_NONE;
        }
        __syncthreads();
        // the thread's own flag (0, 1 undecided, 2 domain error): every loop exit is decided by a
        // __syncthreads_or over these, the same in every thread
        int mf = 0;
        if (tid < EA_MAXD) {
            const uint16_t* qr = P.q + b * P.g.q_seq_stride + (int64_t)t * P.g.q_tok_stride + (int64_t)hq * P.g.q_head_stride;
            const uint32_t x = tid < d ? qr[tid] : 0u;
            S.q[tid] = (double)__uint_as_float(x << 16);
            if (((x >> 7) & 0xFF) == 0xFF) mf = 2;
        }
        bool stop = __syncthreads_or(mf) != 0;
        const DD zero = {0.0, 0.0, 0.0, 0.0};
        DD z = zero, n[2] = {zero, zero};
        int R = DD_NONE;  // block-uniform
        for (int64_t j0 = jc0; j0 < jc1 && !stop; j0 += EA_DD_KEYS) {
            // ---- the wave's V rows (keys 16 wv .. of the pass), lane ln channels 2 ln and 2 ln + 1:
            // requested first, so that one memory latency covers K and V
            const int kb = 16 * wv;
            const int nk = (int)max((int64_t)0, min((int64_t)16, jc1 - j0 - kb));
            const int64_t myoff = lane < nk ? kv_off(P, b, key_n(j0 + kb + lane), hk, 1) : 0;
            uint32_t vx[16];
#pragma unroll
            for (int kk = 0; kk < 16; ++kk) {
                const int64_t o = __shfl(myoff, kk, 64);
                vx[kk] = 0;
                if (kk < nk && 2 * lane < dv) {
                    const uint16_t* vp = P.v + o + 2 * lane;
                    vx[kk] = v4 ? *(const uint32_t*)vp : ((uint32_t)vp[0] | ((uint32_t)vp[1] << 16));
                }
            }
            // ---- scores and weights: 4 lanes per key
            const int kq = tid >> 2, part = tid & 3;
            const int64_t j = j0 + kq;
            const bool have = j < jc1;
            double s = 0.0, es = 0.0, ea = 0.0;
            bool bad = false;
            if (have) {
                const uint16_t* kr = P.k + kv_off(P, b, key_n(j), hk, 0);
                uint4 kv[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int c0 = 8 * (4 * i + part);
                    kv[i] = make_uint4(0, 0, 0, 0);
                    if (c0 >= d) continue;  // d is a multiple of 8
                    if (k16) {
                        kv[i] = *(const uint4*)(kr + c0);
                    } else {
                        uint32_t* kw = (uint32_t*)&kv[i];
#pragma unroll
                        for (int h = 0; h < 4; ++h) kw[h] = (uint32_t)kr[c0 + 2 * h] | ((uint32_t)kr[c0 + 2 * h + 1] << 16);
                    }
                }
#pragma unroll 1
                for (int i = 0; i < 4; ++i) {
                    const double* qp = S.q + 8 * (4 * i + part);
                    const uint32_t kw[4] = {kv[0].x, kv[0].y, kv[0].z, kv[0].w};
                    kv[0] = kv[1];
                    kv[1] = kv[2];
                    kv[2] = kv[3];
#pragma unroll
                    for (int h = 0; h < 4; ++h) {
                        bad |= ((kw[h] >> 7) & 0xFF) == 0xFF || ((kw[h] >> 23) & 0xFF) == 0xFF;
                        double e0, e1;
                        s = two_sum(s, qp[2 * h] * bf16lo_f64(kw[h]), &e0);
                        s = two_sum(s, qp[2 * h + 1] * bf16hi_f64(kw[h]), &e1);
                        es += e0 + e1;
                        ea += fabs(e0) + fabs(e1);
                    }
                }
            }
#pragma unroll
            for (int o = 1; o < 4; o <<= 1) {
                const double s2 = __shfl_xor(s, o, 64), es2 = __shfl_xor(es, o, 64), ea2 = __shfl_xor(ea, o, 64);
                double e0;
                // the lower lane first in every lane, so that the four lanes agree
                s = (part & o) ? two_sum(s2, s, &e0) : two_sum(s, s2, &e0);
                es = (es + es2) + e0;
                ea = (ea + ea2) + fabs(e0);
            }
            if (bad) mf = 2;
            int32_t M = 0, E = 0;
            if (have && part == 0 && !bad) {
                uint32_t tbits = 0;
                const int ls = !isfinite(s) ? 3
                               : (s == 0.0 && es == 0.0 && ea == 0.0) ? 1 : logit_cert(P.alpha, s, es, ea * 0x1p-44, &tbits);
                bool ok = false;
                if (ls == 1) tbits = 0;
                if (ls <= 1) {
                    ok = pf::table_weight(tbits, S.T1, S.T2, &M, &E);
                    if (!ok) {
                        int64_t E2 = 0;
                        ok = weight_wide(tbits, &M, &E2) == 0 && E2 > -(1LL << 30) && E2 < (1LL << 30);
                        E = (int32_t)E2;
                    }
                }
                if (!ok) {
                    M = 0;
                    mf = max(mf, ls == 2 ? 2 : 1);  // 2: |alpha s| rounds above fp32 max
                }
            }
            if (part == 0) {
                S.M[kq] = M;
                S.E[kq] = E;
            }
            const int wm = wave_max_dpp(M ? E + 23 : DD_NONE);
            if (lane == 0) atomicMax(&S.mx, wm);
            __syncthreads();
            // the reference exponent, moved when a weight passes it by 2^64
            const int mx = S.mx;
            if (mx > R + 64) {
                if (R != DD_NONE) {
                    if (R - mx < -800) mf = max(mf, 1);
                    const double f = ldexp(1.0, max(R - mx, -800));
                    dd_scale(z, f);
                    dd_scale(n[0], f);
                    dd_scale(n[1], f);
                }
                R = mx;
            }
            if (M) {
                // products stay normal numbers down to 2^-800 (2^-133 the smallest V element)
                if (E - R < -800) mf = max(mf, 1);
                else if (E + 23 - R < DD_WINDOW) z.err += ldexp((double)M, E - R);
                else dd_add(z, ldexp((double)M, E - R));
            }
            // ---- P.V
            double myw = 0.0;
            if (lane < nk) {
                const int de = S.E[kb + lane] - R;
                myw = de < -800 ? 0.0 : ldexp((double)S.M[kb + lane], de);
            }
            bool vbad = false;
#pragma unroll
            for (int kk = 0; kk < 16; ++kk) {
                const double w = __shfl(myw, kk, 64);  // 0 past the last key
                const uint32_t v = vx[kk];
                vbad |= ((v >> 7) & 0xFF) == 0xFF || ((v >> 23) & 0xFF) == 0xFF;
                const double p0 = w * bf16lo_f64(v), p1 = w * bf16hi_f64(v);
                if (w < ldexp(1.0, DD_WINDOW)) {
                    n[0].err += fabs(p0);
                    n[1].err += fabs(p1);
                } else {
                    dd_add(n[0], p0);
                    dd_add(n[1], p1);
                }
            }
            if (vbad) mf = 2;  // NaN/inf in a visible V row
            stop = __syncthreads_or(mf) != 0;  // and S.M, S.E may be rewritten
        }
        if (mf) atomicMax(&S.flag, mf);
        // ---- the block's sums
#pragma unroll 1
        for (int o = 32; o > 0; o >>= 1) {
            const DD a = {__shfl_xor(z.hi, o, 64), __shfl_xor(z.lo, o, 64), __shfl_xor(z.mag, o, 64), __shfl_xor(z.err, o, 64)};
            dd_join(z, a);
        }
        if (lane == 0) S.zred[wv] = z;
        S.red[wv][2 * lane] = n[0];
        S.red[wv][2 * lane + 1] = n[1];
        __syncthreads();
        z = S.zred[0];
#pragma unroll 1
        for (int k = 1; k < EA_DD_WAVES; ++k) dd_join(z, S.zred[k]);
        DD nc = zero;
        if (tid < dv)
#pragma unroll 1
            for (int k = 0; k < EA_DD_WAVES; ++k) dd_join(nc, S.red[k][tid]);
        int fl = S.flag;
        if (C > 1) {
            // this chunk's partial, then the row's last block merges. Partials go past the XCD's L2
            // (agent-scope stores and loads) and are complete before the count moves: a release
            // fence would write back the whole L2 instead (it cost about 40 us after a prefill step)
            DDPart& pt = parts[item];
            if (tid == 0) {
                agent_store(&pt.R, R);
                agent_store(&pt.flag, fl);
                agent_store(&pt.z, z);
            }
            if (tid < dv) agent_store(&pt.n[tid], nc);
            agent_done();
            __syncthreads();
            if (tid == 0) S.last = atomicAdd(&P.wl_cnt[1 + slot], 1) == C - 1;
            __syncthreads();
            if (!S.last) continue;
            asm volatile("" ::: "memory");
            // every partial's head in one round of loads, then the channels by 4 threads each
            DDPart* rp = parts + (int64_t)slot * C;
            if (tid < C) {
                S.pR[tid] = agent_load(&rp[tid].R);
                S.pz[tid] = agent_load(&rp[tid].z);
                const int pf = agent_load(&rp[tid].flag);
                if (pf) atomicMax(&S.flag, pf);
                atomicMax(&S.mx, S.pR[tid]);
            }
            __syncthreads();
            R = S.mx;
            fl = S.flag;
            z = zero;
#pragma unroll 1
            for (int k = 0; k < C; ++k) {
                if (S.pR[k] == DD_NONE) continue;
                const double f = ldexp(1.0, max(S.pR[k] - R, -800));
                if (S.pR[k] - R < -800) fl = max(fl, 1);
                if (S.pR[k] - R < DD_WINDOW) z.err += dd_size(S.pz[k]) * f;
                else dd_join(z, S.pz[k], f);
            }
            const int c = tid & (EA_MAXDV - 1), g = tid / EA_MAXDV;
            nc = zero;
            if (c < dv) {
#pragma unroll 4
                for (int k = g; k < C; k += EA_DD_THREADS / EA_MAXDV) {
                    const DD a = agent_load(&rp[k].n[c]);
                    if (S.pR[k] == DD_NONE) continue;
                    const double f = ldexp(1.0, max(S.pR[k] - R, -800));
                    if (S.pR[k] - R < DD_WINDOW) nc.err += dd_size(a) * f;
                    else dd_join(nc, a, f);
                }
                S.red[g][c] = nc;
            }
            __syncthreads();
            if (tid < dv)
                for (int k = 1; k < EA_DD_THREADS / EA_MAXDV; ++k) dd_join(nc, S.red[k][tid]);
        }
        // ---- RN(N / Z) per channel; a row without keys is +0
        uint32_t bits = 0;
        bool und = false;
        if (fl == 0 && R != DD_NONE && tid < dv) {
            const double adds = (double)(nkeys + 64 + 4 * C + 4 * EA_DD_WAVES);
            und = !dd_quotient(nc, z, adds, P.out_fp32, &bits);
        }
        if (__syncthreads_or(und)) fl = 1;
        if (fl == 1) {
            if (tid == 0) {
                agent_store(&P.t2left[atomicAdd(&P.wl_cnt[EA_T2_LEFT], 1)], (int32_t)row);
                if (P.stats_x) atomicAdd((unsigned long long*)&P.stats_x[1], 1ull);
            }
            continue;
        }
        if (tid < dv) {
            const int64_t o = b * P.g.o_seq_stride + (int64_t)t * P.g.o_tok_stride + (int64_t)hq * P.g.o_head_stride + tid;
            if (P.out_fp32) ((uint32_t*)P.out)[o] = fl ? 0u : bits;
            else ((uint16_t*)P.out)[o] = fl ? (uint16_t)0 : (uint16_t)bits;
        }
        if (tid == 0) {
            P.flags[row] = (uint8_t)fl;
            if (P.stats) atomicAdd((unsigned long long*)&P.stats[fl ? 4 : 2], 1ull);
        }
    }
}

}  // namespace ea
