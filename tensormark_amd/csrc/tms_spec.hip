// tms_spec.hip -- speculative accept/reject (stochastic verify) for gfx950.
//
// Two launches per call, both stream-ordered:
//
//   statistics    one record per row (the k + 1 target rows and the k draft
//                 rows of every sequence): m = max(v / T), the exact integer
//                 sum Z of the row's weights q44(exp64(v / T - m)), and the
//                 weight of the row's draft token.  spec_row_kernel: one
//                 1024-thread workgroup per 32K ids of a row, holding them in
//                 registers (one read), or per fewer ids where the rows are
//                 too few to fill the chip.
//   spec_resolve  B x P workgroups.  Every workgroup of a sequence evaluates
//                 the accept tests u_i < p_t(x_i) / p_d(x_i) from the row
//                 statistics (the same decision in each), then sums the
//                 weights of its 1/P of the vocabulary for the distribution
//                 the final draw uses: the residual max(p_t - p_d, 0) at the
//                 first rejection, else the target row k (the bonus token).
//                 It publishes the partial sums, reads the others', and the
//                 workgroup whose part holds the draw's threshold locates the
//                 token (vocabularies past 262144: the last arriver by ticket
//                 does, recomputing that part's weights).
//
// The weights are build-defined (no reference counterpart): exp64 is the
// table-driven exponential of tms_device.h, q44 rounds to multiples of 2^-44,
// so every sum is an exact int64 and independent of summation order.  The
// greedy limit (one-hot p_t and p_d) is the argmax-match rule of
// spec_generate_greedy (tensormark/llama.h:5127-5131).

#include <float.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "../../include/tmsample_hip.h"
#include "tms_context.h"
#include "tms_device.h"

namespace tms {

__constant__ double kSpecExpTab[64] = {TMS_EXP2_64THS};
constexpr uint64_t kPartReady = 1ull << 63;   // published partial sum is complete
constexpr int kPartPoll = 1 << 20;            // bound on the finisher's wait per part, which has been stored

constexpr int kRowW = kRowT / 64;

// Workgroups that wait on each other, in a grid that need not be resident at
// once, take their places in order from a counter: when one is resident, all
// those before it have been, so the parts of every earlier row are all
// running or done, and only the last row of a group's counter waits for
// workgroups that have still to start, which those rows' ends let in.
// kSpecClaims counters, each with the rows (or sequences) of its residue,
// share the traffic.  The last claim resets its counter.
//
// Other contexts' kernels may hold the places that the last workgroups need,
// and wait themselves.  So no answer depends on a wait: a workgroup polls
// `polls` times (some 0.2 ms, where a call takes 20 to 100 us); then it forms
// a missing maximum from the logits itself, or leaves the draw to the
// sequence's last workgroup, for which every sum is there.  The results are
// the same whoever forms them.
struct SArgs {
    const void* target;
    const void* draft;
    int B, k, V;
    bool fast;   // rows 16-byte aligned and V a multiple of the vector width
    int P, Lp;   // vocabulary parts of the two-launch resolve and their length
    bool lazy;   // the row kernel leaves the bonus rows (target row k) to the resolve
    const int32_t* tokens;
    const tms_row_params* params;
    const uint32_t* draws;
    int32_t* out_acc;
    int32_t* out_tok;
    int32_t* out_status;
    tms_spec_stat* stats;
    uint64_t* parts;
    uint32_t* tickets;   // [B][kCounterStride]: resolve parts
    int S, pv;           // parts of a row in the row kernel, and their length in vectors
    uint64_t* rparts;    // [B * (2k + 1)][S][2]: a part's max word and its share of Z
    uint32_t* claims;    // [2][kSpecClaims][kCounterStride]: row kernel, resolve
    bool claim_rows, claim_parts;   // the grid may not be resident at once
    int polls;           // of a wait for another workgroup
#ifdef TMS_TRACE
    uint64_t* trace;     // trace builds: 8 stamps per workgroup
#endif
};

#ifdef TMS_TRACE
#define SPEC_TR(i)                                                                                         \
    do {                                                                                                   \
        if (threadIdx.x == 0 && a.trace) a.trace[blockIdx.x * 8 + (i)] = __builtin_amdgcn_s_memrealtime(); \
    } while (0)
#else
#define SPEC_TR(i) ((void)0)
#endif

// LDS of a verify workgroup (up to 16 waves).
struct SpecLds {
    double tab[64];
    float shf[kRowW];
    int64_t shl[2 * kRowW];
    int64_t part_w[kSpecParts];
    int64_t part_t[kSpecParts];
    int misc[kRowW];
    tms_spec_stat srow[2 * kSpecMaxK + 1];
    int stok[kSpecMaxK];
    double su[kSpecMaxK];
    int claim;
    uint64_t late;       // the parts a wait ran out for
};

// This workgroup's place in a grid of kSpecClaims x n: (row, part) of rows
// of S parts; claimed when the grid may not be resident at once.
__device__ __forceinline__ void place(int S, bool claimed, uint32_t* counters, SpecLds& L, int& row, int& part) {
    const int c = blockIdx.x & (kSpecClaims - 1);
    int n = blockIdx.x / kSpecClaims;
    if (claimed) {
        if (threadIdx.x == 0) {
            uint32_t* w = counters + c * kCounterStride;
            const uint32_t m = __hip_atomic_fetch_add(w, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (m == gridDim.x / kSpecClaims - 1) st_agent(w, 0u);
            L.claim = (int)m;
        }
        lds_sync();
        n = __builtin_amdgcn_readfirstlane(L.claim);
    }
    row = n / S * kSpecClaims + c;
    part = n % S;
}

__device__ __forceinline__ void load_exp_table(double* tab) {
    if (threadIdx.x < 64) tab[threadIdx.x] = kSpecExpTab[threadIdx.x];
}

// Row i of sequence b: i <= k is target row i, i > k is draft row i - k - 1.
template <typename T>
__device__ __forceinline__ const T* spec_row(const SArgs& a, int b, int i) {
    if (i <= a.k) return (const T*)a.target + ((int64_t)b * (a.k + 1) + i) * a.V;
    return (const T*)a.draft + ((int64_t)b * a.k + (i - a.k - 1)) * a.V;
}

// f(id, value) over ids [lo, hi) of a row, strided over the workgroup.  The
// vector path needs lo and hi multiples of the vector width.
template <typename T, typename F>
__device__ __forceinline__ void for_range(const T* row, int lo, int hi, bool fast, F&& f) {
    constexpr int VEC = Elt<T>::kVec;
    if (fast) {
#pragma unroll 4
        for (int v = lo / VEC + (int)threadIdx.x; v < hi / VEC; v += kBlock) {
            const uint4 q = *(const uint4*)(row + (int64_t)v * VEC);
            float x[VEC];
            Elt<T>::widen(q, x);
#pragma unroll
            for (int e = 0; e < VEC; ++e) f(v * VEC + e, x[e]);
        }
    } else {
        for (int i = lo + (int)threadIdx.x; i < hi; i += kBlock) f(i, Elt<T>::scalar(row + i));
    }
}

// The same over two rows at once: f(id, value of r0, value of r1).
template <typename T, typename F>
__device__ __forceinline__ void for_range2(const T* r0, const T* r1, int lo, int hi, bool fast, F&& f) {
    constexpr int VEC = Elt<T>::kVec;
    if (fast) {
#pragma unroll 2
        for (int v = lo / VEC + (int)threadIdx.x; v < hi / VEC; v += kBlock) {
            const uint4 q0 = *(const uint4*)(r0 + (int64_t)v * VEC);
            const uint4 q1 = *(const uint4*)(r1 + (int64_t)v * VEC);
            float x0[VEC], x1[VEC];
            Elt<T>::widen(q0, x0);
            Elt<T>::widen(q1, x1);
#pragma unroll
            for (int e = 0; e < VEC; ++e) f(v * VEC + e, x0[e], x1[e]);
        }
    } else {
        for (int i = lo + (int)threadIdx.x; i < hi; i += kBlock)
            f(i, Elt<T>::scalar(r0 + i), Elt<T>::scalar(r1 + i));
    }
}

template <int NW = kWaves>
__device__ __forceinline__ float block_max_f32(float v, float* sh) {
    v = wave_max_f32(v);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = sh[0];
#pragma unroll
    for (int i = 1; i < NW; ++i) r = fmaxf(r, sh[i]);
    __syncthreads();
    return r;
}

template <int NW = kWaves>
__device__ __forceinline__ int64_t block_sum_i64(int64_t v, int64_t* sh) {
    v = wave_incl_scan_i64_dpp(v);
    if ((threadIdx.x & 63) == 63) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    int64_t r = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) r += sh[i];
    __syncthreads();
    return r;
}

template <int NW = kWaves>
__device__ __forceinline__ int block_or(int v, int* sh) {
    v = __any(v) ? 1 : 0;
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    int r = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) r |= sh[i];
    __syncthreads();
    return r;
}

// v / T.  The hot loops are instantiated twice, DIV false for T = 1 (where
// the division is the identity) and true otherwise, and pick one per row:
// a per-element test compiles to a select that still divides.
template <bool DIV = true>
__device__ __forceinline__ float scaled(float v, float temp) { return DIV ? v / temp : v; }

// Weight of a scaled logit on the 2^-44 grid: q44(exp64(v / T - m)), where m
// is the maximum of v / T over the row, so the argument is never positive.
template <bool DIV = true>
__device__ __forceinline__ int64_t weight(float v, float temp, double m, const double* tab) {
    return q44_exp_nonpos((double)scaled<DIV>(v, temp) - m, tab);
}

// The same weight as a double holding the whole number.
template <bool DIV = true>
__device__ __forceinline__ double weight_f(float v, float temp, double m, const double* tab) {
    return q44_exp_nonpos_f((double)scaled<DIV>(v, temp) - m, tab);
}

// Residual weight q44(max(p_t - p_d, 0)) from the two rows' weights (whole
// numbers as doubles), p = e / (double)Z.  The divisors' reciprocals are
// formed once (Resid), and div_rn returns the correctly rounded quotients,
// the same as dividing per element.  Z >= 2^44 for a row that reaches here
// (its maximum has weight 2^44), so nothing overflows or is subnormal.
struct Resid {
    double zt, zd, yt, yd;
    __device__ __forceinline__ Resid(int64_t Zt, int64_t Zd)
        : zt((double)Zt), zd((double)Zd), yt(1.0 / (double)Zt), yd(1.0 / (double)Zd) {}
    __device__ __forceinline__ int64_t operator()(double et, double ed) const {
        const double d = div_rn(et, zt, yt) - div_rn(ed, zd, yd);
        return d > 0.0 ? q44(d) : 0;
    }
};

__device__ __forceinline__ int64_t as_i64(double f) {
    return __double_as_longlong(f + 0x1p52) - __double_as_longlong(0x1p52);
}

// Loops over a thread's registers (slot sl holds vector t + sl * NT, in
// while below nv): the max of the logits and the NaN/+inf flag, then the
// share of Z.
//
// Max and flag from the logits' bits, three integer operations a logit (two
// of them to an instruction): a positive NaN is above +inf as a signed
// number, a negative one above -inf as an unsigned one, and the maximum is
// the signed maximum or, with every sign bit set, the unsigned minimum.  A
// slot past nv holds a vector of the row again, which changes none of them.
template <typename T, int NS>
__device__ __forceinline__ void row_max(const uint4 (&q)[NS], float& mx, int& nf) {
    constexpr int VEC = Elt<T>::kVec;
    int hi = INT32_MIN;
    uint32_t hu = 0, lu = UINT32_MAX;
#pragma unroll
    for (int sl = 0; sl < NS; ++sl) {
        float x[VEC];
        Elt<T>::widen(q[sl], x);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const uint32_t u = __float_as_uint(x[e]);
            hi = max(hi, (int)u);
            hu = max(hu, u);
            lu = min(lu, u);
        }
    }
    nf = hi >= 0x7F800000 || hu > 0xFF800000u;   // NaN or +inf
    mx = __uint_as_float(hi >= 0 ? (uint32_t)hi : lu);
}
// DIV: v / T as (float)(v * y), y = RN(1 / T) in double.  The quotient of
// two 24-bit significands is no midpoint of two floats and lies at least
// 2^-49 of itself from one, and the product is within 2^-52 of it, so it
// rounds to the float that the division returns.  (Subnormal quotients can
// be midpoints: there the two may differ by 2^-149, which moves no weight.)
template <typename T, int NS, int NT, bool DIV>
__device__ __forceinline__ int64_t row_z(const uint4 (&q)[NS], int nv, double y, double md, const double* tab) {
    constexpr int VEC = Elt<T>::kVec;
    const int t = threadIdx.x;
    // whole numbers of at most 2^44 each, at most 128 of them: the double
    // sum is exact
    static_assert(NS * VEC <= 128, "exact double sum");
    double z = 0.0;
#pragma unroll
    for (int sl = 0; sl < NS; ++sl) {
        float x[VEC];
        Elt<T>::widen(q[sl], x);
        if (t + sl * NT < nv) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                const double v = (double)x[e];
                z += q44_exp_nonpos_f((DIV ? (double)(float)(v * y) : v) - md, tab);
            }
        }
    }
    return __double_as_longlong(z + 0x1p52) - __double_as_longlong(0x1p52);
}

// The vector with its first n elements (n < the vector width) set to -inf.
template <typename T>
__device__ __forceinline__ uint4 drop_first(uint4 q, int n) {
    constexpr uint32_t kNeg = Elt<T>::kNegInfWord;
    constexpr int PW = 4 / (int)sizeof(T);   // elements a word
    uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (n >= (i + 1) * PW) w[i] = kNeg;
        else if (PW == 2 && n == 2 * i + 1) w[i] = (w[i] & 0xFFFF0000u) | (kNeg & 0xFFFFu);
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// A row of fewer ids than a vector holds: its logits, then -inf.
template <typename T>
__device__ __forceinline__ uint4 short_row(const T* row, int V) {
    uint4 q;
    T* e = (T*)&q;
    uint32_t* w = (uint32_t*)&q;
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = Elt<T>::kNegInfWord;
#pragma unroll
    for (int i = 0; i < Elt<T>::kVec; ++i)
        if (i < V) e[i] = row[i];
    return q;
}

// The sequence's statistics, draft tokens and accept uniforms staged in LDS
// (one load or Philox draw per thread), then the accept tests
// u_i < (e_t * Z_d) / (e_d * Z_t), evaluated identically by every workgroup
// that runs them.  rej < 0: every draft accepted (the bonus draw).
template <typename T>
__device__ void accept_tests(const SArgs& a, int b, SpecLds& L, int& status, int& acc, int& rej) {
    const int t = threadIdx.x;
    const int R = 2 * a.k + 1;
    const tms_row_params P = a.params[b];
    const int g0 = b * R;
    const uint32_t* dw = a.draws ? a.draws + (int64_t)b * (a.k + 1) * 2 : nullptr;
    if (t < R) {
        const uint64_t* w = (const uint64_t*)(a.stats + g0 + t);
        const uint64_t w0 = ld_agent(&w[0]);
        L.srow[t].m = __uint_as_float((uint32_t)w0);
        L.srow[t].status = (int32_t)(w0 >> 32);
        L.srow[t].Z = a.S > 1 ? 0 : (int64_t)ld_agent(&w[1]);
        L.srow[t].ex = (int64_t)ld_agent(&w[2]);
        L.srow[t].pad = 0;
    }
    if (a.S > 1) {   // the shares of Z of a row's parts
        __syncthreads();
        const uint64_t* w = a.rparts + (int64_t)g0 * a.S * 2;
        for (int i = t; i < R * a.S; i += kBlock)
            if (!(a.lazy && i / a.S == a.k))
                atomicAdd((unsigned long long*)&L.srow[i / a.S].Z, (unsigned long long)ld_agent(&w[2 * i + 1]));
    }
    if (t < a.k) {
        L.stok[t] = a.tokens[(int64_t)b * a.k + t];
        uint32_t w0, w1;
        if (dw) { w0 = dw[2 * t]; w1 = dw[2 * t + 1]; }
        else row_words(P.seed, P.offset, (uint32_t)t, w0, w1);
        L.su[t] = canonical(w0, w1);
    }
    __syncthreads();
    status = TMS_ROW_OK;
    acc = 0;
    rej = -1;
    if (!(P.temperature > 0.0f && P.temperature <= FLT_MAX)) {
        status = TMS_ROW_BAD_PARAMS;
        return;
    }
    acc = a.k;
    // Lane i < k of every wave evaluates position i (the same operations as
    // a loop over i would); the lowest position that is not an accept
    // decides, as the first exit of that loop would.
    const int lane = t & 63;
    int code = 0;   // 0: accepted, 1: rejected, 2: the row's status sv
    int sv = TMS_ROW_OK;
    if (lane < a.k) {
        const tms_spec_stat ts = L.srow[lane], ds = L.srow[a.k + 1 + lane];
        const int x = L.stok[lane];
        if (ts.status) {
            code = 2;
            sv = ts.status;
        } else if (ds.status) {
            code = 2;
            sv = ds.status;
        } else if (x < 0 || x >= a.V) {
            code = 2;
            sv = TMS_ROW_BAD_PARAMS;
        } else {
            double r;
            if (ds.ex == 0) r = ts.ex > 0 ? 1.0 : 0.0;
            else r = ((double)ts.ex * (double)ds.Z) / ((double)ds.ex * (double)ts.Z);
            code = L.su[lane] < r ? 0 : 1;
        }
    }
    const uint64_t stop = __ballot(lane < a.k && code != 0);
    if (stop) {
        const int i = __builtin_ctzll(stop);
        const int ci = __shfl(code, i, 64);
        if (ci == 2) {
            status = __shfl(sv, i, 64);
            return;
        }
        acc = i;
        rej = i;
    }
    if (rej < 0 && !a.lazy && L.srow[a.k].status) status = L.srow[a.k].status;
}

// Part p of sequence b's resolution.
// WAIT (up to kSpecParts parts of runs of at most kRunMax ids): every
// workgroup keeps its part's weights in registers, reads every part's sums
// (bounded wait), and the one whose part holds the draw's threshold locates
// the token from its registers (from the logits again for a residual of no
// mass, which is drawn by the target's weights).  One whose wait ran out says so and is gone.
// The last of the P to count itself (each after its words are stored and its
// loads returned) zeroes the parts, and locates the token if its workgroup is
// gone, from that part's weights again.
// Otherwise the last arriver by ticket gathers the parts and recomputes the
// weights of the part holding the threshold.
template <typename T, bool WAIT>
__device__ void resolve_part(const SArgs& a, int b, int p, SpecLds& L) {
    const double* tab = L.tab;
    int64_t* shl = L.shl;
    int64_t* part_w = L.part_w;
    int64_t* part_t = L.part_t;
    int* misc = L.misc;
    const tms_spec_stat* srow = L.srow;
    const int t = threadIdx.x;
    const tms_row_params P = a.params[b];
    const uint32_t* dw = a.draws ? a.draws + (int64_t)b * (a.k + 1) * 2 : nullptr;
    int status, acc, rej;
    SPEC_TR(0);
    // the rows' part maxima, ready for the next call (their readers, the
    // statistics' workgroups, have ended)
    if (a.S > 1 && p == 0)
        for (int i = t; i < (2 * a.k + 1) * a.S; i += kBlock)
            st_agent(a.rparts + ((int64_t)b * (2 * a.k + 1) * a.S + i) * 2, (uint64_t)0);
    accept_tests<T>(a, b, L, status, acc, rej);
    SPEC_TR(1);
    if (status != TMS_ROW_OK) {
        if (p == 0 && t == 0) {
            a.out_acc[b] = 0;
            a.out_tok[b] = -1;
            a.out_status[b] = status;
        }
        return;   // every workgroup of the sequence returns here: no ticket
    }

    // ---- this part's sums: the draw's weights (w) and the target's (et).
    const int ti = rej < 0 ? a.k : rej;
    const T* rt = spec_row<T>(a, b, ti);
    const T* rd = spec_row<T>(a, b, rej < 0 ? ti : a.k + 1 + rej);
    const tms_spec_stat ts = srow[ti];
    const tms_spec_stat ds = rej < 0 ? ts : srow[a.k + 1 + rej];
    const float temp = P.temperature;
    const double mt = (double)ts.m, md = (double)ds.m;
    const Resid res(ts.Z, ds.Z);
    __syncthreads();   // exp table in LDS
    const int lo = p * a.Lp, hi = min(a.V, lo + a.Lp);
    int64_t wsum = 0, tsum = 0;
    int64_t wr[kRunMax];                // a run's weights
    double mtu = mt;                    // the target row's maximum of v / T
    if constexpr (WAIT) {
        // a contiguous run of ids per thread, every load issued at once
        const int E = a.Lp / kBlock;   // a multiple of the vector width
        const int r_lo = min(hi, lo + t * E), r_hi = min(hi, r_lo + E);
        float xt[kRunMax], xd[kRunMax];
#pragma unroll
        for (int j = 0; j < kRunMax; ++j) xt[j] = xd[j] = 0.0f;
        if (r_hi - r_lo == E) {
            constexpr int VEC = Elt<T>::kVec;
#pragma unroll
            for (int j = 0; j < kRunMax; j += VEC) {
                if (j >= E) break;
                const uint4 qt = ld_any(rt + r_lo + j);
                uint4 qd = qt;
                if (rej >= 0) qd = ld_any(rd + r_lo + j);
                float x[VEC];
                Elt<T>::widen(qt, x);
#pragma unroll
                for (int e = 0; e < VEC; ++e) xt[j + e] = x[e];
                Elt<T>::widen(qd, x);
#pragma unroll
                for (int e = 0; e < VEC; ++e) xd[j + e] = x[e];
            }
        } else {   // the row's last run
#pragma unroll
            for (int j = 0; j < kRunMax; ++j) {
                if (r_lo + j < r_hi) {
                    xt[j] = Elt<T>::scalar(rt + r_lo + j);
                    if (rej >= 0) xd[j] = Elt<T>::scalar(rd + r_lo + j);
                }
            }
        }
        if (a.lazy && rej < 0) {
            // The bonus row's statistics (the row kernel left them): each
            // part's max of v / T and NaN / +inf flag, exchanged between the
            // sequence's workgroups; the status rules of the statistics
            // kernels (tmo_spec_weights).
            float pm = -__builtin_huge_valf();
            int pnf = 0;
#pragma unroll
            for (int j = 0; j < kRunMax; ++j) {
                if (r_lo + j < r_hi) {
                    const float v = xt[j];
                    pnf |= (__builtin_isnan(v) || v == __builtin_huge_valf()) ? 1 : 0;
                    pm = fmaxf(pm, scaled(v, temp));
                }
            }
            pm = block_max_f32(pm, L.shf);
            pnf = block_or(pnf, misc);
            uint64_t* mw = a.parts + ((int64_t)b * kSpecParts + p) * kPartWords + 2;
            if (t == 0) st_agent(mw, kPartReady | ((uint64_t)pnf << 32) | okey(pm));
            uint32_t km = 0;
            int knf = 0;
            if (t < 64) {
                bool late = false;
                if (t < a.P) {
                    const uint64_t* q = a.parts + ((int64_t)b * kSpecParts + t) * kPartWords + 2;
                    uint64_t h = 0;
                    for (int it = 0; it < a.polls; ++it) {
                        h = ld_agent(q);
                        if (h & kPartReady) break;
                        __builtin_amdgcn_s_sleep(1);
                    }
                    late = !(h & kPartReady);
                    km = (uint32_t)h;
                    knf = (int)((h >> 32) & 1u);
                }
                const uint64_t all = __ballot(late);
                if (t == 0) L.late = all;
            }
            // the bonus maxima's readers: the last zeroes the words and its
            // counter.  The waves' maxima meet in part_w, whose next writes
            // (the part sums' gather) come after the sums' barriers; shl is
            // the sums' own scratch.
            km = (uint32_t)wave_max_u64(km);
            if ((t & 63) == 0) part_w[t >> 6] = (int64_t)km;
            knf = block_or(knf, misc);
            if (t == 0) {
                __builtin_amdgcn_s_waitcnt(0);   // this workgroup's word is stored
                const uint32_t done = __hip_atomic_fetch_add(&a.tickets[b * kCounterStride + 1], 1u,
                                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                misc[2] = done == (uint32_t)(a.P - 1) ? 1 : 0;
            }
            __syncthreads();
            uint32_t kmax = (uint32_t)part_w[0];
            for (int w = 1; w < kWaves; ++w) kmax = max(kmax, (uint32_t)part_w[w]);
            if (misc[2]) {
                if (t < a.P) st_agent(a.parts + ((int64_t)b * kSpecParts + t) * kPartWords + 2, (uint64_t)0);
                if (t == 0) st_agent(&a.tickets[b * kCounterStride + 1], 0u);
            }
            const uint64_t late = (uint64_t)readlane_i64((int64_t)L.late, 0);
            if (late) {   // those parts' maxima, from the row
                __syncthreads();
                pm = -__builtin_huge_valf();
                pnf = 0;
                for (uint64_t m = late; m; m &= m - 1) {
                    const int j0 = __builtin_ctzll(m) * a.Lp, j1 = min(a.V, j0 + a.Lp);
#pragma unroll 1
                    for (int id = j0 + t; id < j1; id += kBlock) {
                        const float v = Elt<T>::scalar(rt + id);
                        pnf |= (__builtin_isnan(v) || v == __builtin_huge_valf()) ? 1 : 0;
                        pm = fmaxf(pm, scaled(v, temp));
                    }
                }
                kmax = max(kmax, okey(block_max_f32(pm, L.shf)));
                knf |= block_or(pnf, misc);
            }
            const float gm = okey_inv(kmax);
            int st = TMS_ROW_OK;
            if (knf) st = TMS_ROW_NONFINITE;
            else if (gm == -__builtin_huge_valf()) st = TMS_ROW_ALL_MASKED;
            else if (gm == __builtin_huge_valf()) st = TMS_ROW_NONFINITE;
            if (st != TMS_ROW_OK) {
                if (p == 0 && t == 0) {
                    a.out_acc[b] = 0;
                    a.out_tok[b] = -1;
                    a.out_status[b] = st;
                }
                return;   // every workgroup of the sequence: no parts published
            }
            mtu = (double)gm;
        }
#pragma unroll
        for (int j = 0; j < kRunMax; ++j) {
            wr[j] = 0;
            if (r_lo + j < r_hi) {
                const double etf = weight_f(xt[j], temp, mtu, tab);
                const int64_t et = as_i64(etf);
                wr[j] = rej < 0 ? et : res(etf, weight_f(xd[j], temp, md, tab));
                tsum += et;
            }
            wsum += wr[j];
        }
    } else if (rej < 0) {
        for_range(rt, lo, hi, a.fast, [&](int, float v) { tsum += weight(v, temp, mt, tab); });
        wsum = tsum;
    } else {
        for_range2(rt, rd, lo, hi, a.fast, [&](int, float vt, float vd) {
            const double et = weight_f(vt, temp, mt, tab);
            tsum += as_i64(et);
            wsum += res(et, weight_f(vd, temp, md, tab));
        });
    }
    wsum = block_sum_i64(wsum, shl);
    tsum = block_sum_i64(tsum, shl + kWaves);
    SPEC_TR(2);
    uint64_t* pw = a.parts + ((int64_t)b * kSpecParts + p) * kPartWords;
    if constexpr (WAIT) {
        if (t == 0) {
            st_agent(&pw[0], kPartReady | (uint64_t)wsum);
            st_agent(&pw[1], kPartReady | (uint64_t)tsum);
        }
    } else {
        uint32_t ticket = 0;
        if (t == 0) {
            st_agent(&pw[0], kPartReady | (uint64_t)wsum);
            st_agent(&pw[1], kPartReady | (uint64_t)tsum);
            ticket = __hip_atomic_fetch_add(&a.tickets[b * kCounterStride], 1u, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
            misc[0] = (int)ticket;
        }
        __syncthreads();
        SPEC_TR(3);
        if (misc[0] != a.P - 1) return;
        // the last arriver: its ticket for the next call
        if (t == 0) st_agent(&a.tickets[b * kCounterStride], 0u);
    }

    // ---- gather the parts (bounded wait on their ready bits); the reader
    //      that is last zeroes them for the next call.
    int timed_out = 0;
    if (t < a.P) {
        uint64_t* q = a.parts + ((int64_t)b * kSpecParts + t) * kPartWords;
        uint64_t w = 0, u = 0;
        for (int it = 0; it < (WAIT ? a.polls : kPartPoll); ++it) {
            w = ld_agent(&q[0]);
            u = ld_agent(&q[1]);
            if ((w & kPartReady) && (u & kPartReady)) break;
            __builtin_amdgcn_s_sleep(1);
        }
        timed_out = !((w & kPartReady) && (u & kPartReady));
        part_w[t] = (int64_t)(w & ~kPartReady);
        part_t[t] = (int64_t)(u & ~kPartReady);
        if (!WAIT) {
            st_agent(&q[0], (uint64_t)0);
            st_agent(&q[1], (uint64_t)0);
        }
    }
    uint64_t gone = 0;   // WAIT, in the last workgroup: the parts whose workgroup's wait ran out
    if constexpr (WAIT) {
        static_assert(kSpecParts <= 64, "the parts in one wave");
        uint32_t* done = a.tickets + b * kCounterStride;
        uint64_t* left = (uint64_t*)(done + 2);
        const bool leave = __ballot(timed_out != 0) != 0;   // (the first wave)
        if (t == 0) {
            if (leave) __hip_atomic_fetch_or(left, 1ull << p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __builtin_amdgcn_s_waitcnt(0);
            const uint32_t n = __hip_atomic_fetch_add(done, leave ? 0x10001u : 1u, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT);
            const bool last = (n & 0xFFFFu) == (uint32_t)(a.P - 1);
            L.late = last && ((n >> 16) || leave) ? ld_agent(left) : 0ull;
            misc[1] = last ? 1 : leave ? 2 : 0;
        }
        __syncthreads();
        const int role = __builtin_amdgcn_readfirstlane(misc[1]);
        if (role == 2) return;
        gone = (uint64_t)readlane_i64((int64_t)L.late, 0);
        if (role == 1) {
            if (t < a.P) {
                uint64_t* q = a.parts + ((int64_t)b * kSpecParts + t) * kPartWords;
                if (gone) {
                    part_w[t] = (int64_t)(ld_agent(&q[0]) & ~kPartReady);
                    part_t[t] = (int64_t)(ld_agent(&q[1]) & ~kPartReady);
                }
                st_agent(&q[0], (uint64_t)0);
                st_agent(&q[1], (uint64_t)0);
            }
            if (t == 0) {
                st_agent(done, 0u);
                st_agent(left, (uint64_t)0);
            }
            if (gone) __syncthreads();
        }
    } else if (block_or(timed_out, misc)) {
        if (t == 0) {
            a.out_acc[b] = 0;
            a.out_tok[b] = -1;
            a.out_status[b] = TMS_ROW_INTERNAL;
        }
        return;
    }
    SPEC_TR(4);
    // The parts' sums across the lanes of each wave (P <= 64), by integer
    // scans: exact, so W, the threshold's part and the sum before it equal
    // the sequential sums.  Residual mass 0 (p_t <= p_d everywhere on the
    // grid): draw from p_t.
    static_assert(kSpecParts <= 64, "one part per lane");
    const int pl = t & 63;
    const int64_t sw = wave_incl_scan_i64_dpp(pl < a.P ? part_w[pl] : 0);
    const int64_t st = wave_incl_scan_i64_dpp(pl < a.P ? part_t[pl] : 0);
    int64_t W = readlane_i64(sw, 63);
    const bool use_t = rej < 0 || W == 0;
    if (use_t) W = readlane_i64(st, 63);
    uint32_t w0, w1;
    if (dw) { w0 = dw[2 * a.k]; w1 = dw[2 * a.k + 1]; }
    else row_words(P.seed, P.offset, (uint32_t)a.k, w0, w1);
    const double uf = canonical(w0, w1);
    int64_t thr = (int64_t)floor(uf * (double)W);
    if (thr > W - 1) thr = W - 1;
    // the first part whose inclusive sum exceeds thr (the last one does:
    // thr < W), and the sum of the parts before it
    const int64_t sc = use_t ? st : sw;
    const uint64_t over = __ballot(pl < a.P && sc > thr);
    const int ps = over ? __ffsll((unsigned long long)over) - 1 : a.P - 1;
    const int64_t base = ps > 0 ? readlane_i64(sc, ps - 1) : 0;
    if (WAIT && ps != p && !((gone >> ps) & 1)) return;   // another workgroup holds the threshold's part
    SPEC_TR(6);
    // The part's weights, a contiguous run of ids per thread.
    const int plo = ps * a.Lp, phi = min(a.V, plo + a.Lp);
    const int E = WAIT ? a.Lp / kBlock : (phi - plo + kBlock - 1) / kBlock;
    const int my_lo = min(phi, plo + t * E), my_hi = min(phi, my_lo + E);
    auto w_at = [&](int id) -> int64_t {
        const double et = weight_f(Elt<T>::scalar(rt + id), temp, mtu, tab);
        if (use_t) return as_i64(et);
        return res(et, weight_f(Elt<T>::scalar(rd + id), temp, md, tab));
    };
    // The threads' sums `mine`, scanned; the thread that holds the threshold
    // walks its run from the sum before it.
    auto locate = [&](int64_t mine, auto&& walk) {
        const int lane = t & 63, wv = t >> 6;
        const int64_t inc = wave_incl_scan_i64(mine);
        if (lane == 63) shl[wv] = inc;
        __syncthreads();
        SPEC_TR(5);
        int64_t pre = base;
        for (int i = 0; i < wv; ++i) pre += shl[i];
        pre += inc - mine;
        if (mine > 0 && pre <= thr && thr < pre + mine) {
            a.out_acc[b] = acc;
            a.out_tok[b] = walk(pre);
            a.out_status[b] = TMS_ROW_OK;
        }
    };
    auto walk_ids = [&](int64_t sum) {
#pragma unroll 1
        for (int id = my_lo; id < my_hi; ++id) {
            sum += w_at(id);
            if (sum > thr) return id;
        }
        return my_hi - 1;
    };
    // Runs of up to kRunMax ids: every load issued at once (clamped
    // addresses), the weights kept in registers for the scan and the search;
    // longer runs walk the ids one by one.  WAIT: this workgroup's own run
    // weights, still in registers; others one by one.
    const bool cached = WAIT ? ps == p && (rej < 0 || !use_t) : E <= kRunMax;
    int64_t mine = 0;
    if (!cached) {
#pragma unroll 1
        for (int id = my_lo; id < my_hi; ++id) mine += w_at(id);
        SPEC_TR(7);
        locate(mine, walk_ids);
        return;
    }
    if constexpr (!WAIT) {
        float xt[kRunMax], xd[kRunMax];
#pragma unroll
        for (int j = 0; j < kRunMax; ++j) {
            const int id = min(my_lo + j, phi - 1);
            xt[j] = Elt<T>::scalar(rt + id);
            xd[j] = use_t ? 0.0f : Elt<T>::scalar(rd + id);
        }
#pragma unroll
        for (int j = 0; j < kRunMax; ++j) {
            wr[j] = 0;
            if (my_lo + j < my_hi) {
                const double et = weight_f(xt[j], temp, mt, tab);
                wr[j] = use_t ? as_i64(et) : res(et, weight_f(xd[j], temp, md, tab));
            }
        }
    }
#pragma unroll
    for (int j = 0; j < kRunMax; ++j) mine += wr[j];
    SPEC_TR(7);
    locate(mine, [&](int64_t sum) {
        int tok = my_hi - 1;
        bool found = false;
#pragma unroll
        for (int j = 0; j < kRunMax; ++j) {
            sum += wr[j];
            if (!found && my_lo + j < my_hi && sum > thr) {
                tok = my_lo + j;
                found = true;
            }
        }
        return tok;
    });
}


#ifdef TMS_TRACE
static uint64_t* g_spec_trace;
extern "C" int tms_spec_trace_set(uint64_t* buf) {
    g_spec_trace = buf;
    return 0;
}
#endif

template <typename T, bool WAIT>
__global__ __launch_bounds__(kBlock) void spec_resolve_kernel(SArgs a) {
    __shared__ SpecLds L;
    load_exp_table(L.tab);
    int b, p;
    place(a.P, WAIT && a.claim_parts, a.claims + kSpecClaims * kCounterStride, L, b, p);
    if (b < a.B) resolve_part<T, WAIT>(a, b, p, L);
}

// Row statistics: S workgroups a row (a.S), each holding its part of the row
// in registers (one read), in at most NS vectors a thread.  With more than
// one part, each publishes its maximum and waits for the others' (place()
// has the order that lets it).  Part 0 writes the row's record: m = max(v /
// T) = max(v) / T (a correctly rounded division by T > 0 is monotone), the
// status and the draft token's weight; every part adds its share of
// Z = sum of q44(exp64(v / T - m)), whole numbers, so any split sums to the
// same.  64 registers a thread: 32 waves a CU.
//
// Bound by the exponentials: 110 cycles of a SIMD for 64 of them, 34 us of
// the 63 that B = 32, k = 5, V = 151936 bf16 takes (as two passes by one
// 256-thread workgroup a row: 125); the rest is the loads and the exchange
// that a part's exponentials wait for, under the other workgroup's of its CU.
// Parts of 16K ids in 512-thread workgroups measured alike (88 us a call
// against 92, but 42 against 41 at B = 32, k = 8, V = 32000 fp32).  B = 1, k
// = 4, V = 128256 bf16: 9 rows in 16 parts each take 8.3 us (59).
template <typename T, int NS, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(8, 8)))
void spec_row_kernel(SArgs a) {
    constexpr int VEC = Elt<T>::kVec;
    constexpr int NW = NT / 64;
    __shared__ SpecLds L;
    load_exp_table(L.tab);
    const int t = threadIdx.x;
    // lazy: 2k rows a sequence (the bonus row k left to the resolve)
    const int R = a.lazy ? 2 * a.k : 2 * a.k + 1;
    int g = blockIdx.x, p = 0;
    if (a.S > 1) {
        place(a.S, a.claim_rows, a.claims, L, g, p);
        if (g >= a.B * R) return;
    }
    const int b = g / R;
    int i = g - b * R;
    if (a.lazy && i >= a.k) ++i;
    const T* row = spec_row<T>(a, b, i);
    const int V = a.V;
    const int v0 = p * a.pv;
    const int nv = min((V + VEC - 1) / VEC - v0, a.pv);   // this part's vectors
    uint4 q[NS];
    if (V >= VEC) {
        // a ragged row's last vector ends at the row's end
#pragma unroll
        for (int sl = 0; sl < NS; ++sl)
            q[sl] = ld_any(row + min((v0 + min(t + sl * NT, nv - 1)) * VEC, V - VEC));
        if (!a.fast) {   // ... and begins with ids of the vector before it
#pragma unroll
            for (int sl = 0; sl < NS; ++sl) {
                const int dup = (v0 + t + sl * NT) * VEC - (V - VEC);
                if (dup > 0 && dup < VEC) q[sl] = drop_first<T>(q[sl], dup);
            }
        }
    } else {
#pragma unroll
        for (int sl = 0; sl < NS; ++sl) q[sl] = short_row(row, V);
    }
    // The draft token's logit (draft rows; target row i takes draft i's
    // token), loaded now, after the stream's loads: it is in flight under
    // the max and the sums, and its weight is formed at the end.
    const int di = i < a.k ? i : (i > a.k ? i - a.k - 1 : -1);
    bool xin = false;
    float xv = 0.0f;
    if (t == 0 && p == 0 && di >= 0) {
        const int x = a.tokens[(int64_t)b * a.k + di];
        xin = x >= 0 && x < V;
        if (xin) xv = Elt<T>::scalar(row + x);
    }
    float mx;
    int nf;
    row_max<T, NS>(q, mx, nf);
    if constexpr (VEC == 8) {   // not the max's widened logits, which take twice the registers, kept for the sums
#pragma unroll
        for (int sl = 0; sl < NS; ++sl) asm("" : "+v"(q[sl].x), "+v"(q[sl].y), "+v"(q[sl].z), "+v"(q[sl].w));
    }
    // The part's maximum and NaN/+inf flag in one exchange: each wave's pair
    // in LDS words written once, so one barrier (which also orders the
    // table's LDS writes) and none after the reads.
    {
        const float wm = wave_max_f32(mx);
        const int wn = __any(nf) ? 1 : 0;
        if ((t & 63) == 0) {
            L.shf[t >> 6] = wm;
            L.misc[t >> 6] = wn;
        }
        lds_sync();
        mx = L.shf[0];
        nf = L.misc[0];
#pragma unroll
        for (int j = 1; j < NW; ++j) {
            mx = fmaxf(mx, L.shf[j]);
            nf |= L.misc[j];
        }
    }
    uint64_t* rp = a.rparts + ((int64_t)b * (2 * a.k + 1) + i) * a.S * 2;
    if (a.S > 1) {   // the row's, from every part's word
        if (t == 0) st_agent(rp + 2 * p, kPartReady | ((uint64_t)nf << 32) | okey(mx));
        if (t < 64) {
            uint32_t km = okey(mx);
            bool late = false;
            if (t < a.S && t != p) {
                uint64_t h = 0;
                for (int it = 0; it < a.polls; ++it) {
                    h = ld_agent(rp + 2 * t);
                    if (h & kPartReady) break;
                    __builtin_amdgcn_s_sleep(1);
                }
                late = !(h & kPartReady);
                nf |= (int)((h >> 32) & 1u);
                km = max(km, (uint32_t)h);
            }
            km = (uint32_t)wave_max_u64(km);
            nf = __any(nf) ? 1 : 0;
            const uint64_t all = __ballot(late);
            if (t == 0) {
                L.stok[0] = (int)km;
                L.stok[1] = nf;
                L.late = all;
            }
        }
        lds_sync();
        mx = okey_inv((uint32_t)L.stok[0]);
        nf = L.stok[1];
        const uint64_t late = (uint64_t)readlane_i64((int64_t)L.late, 0);
        if (late) {   // those parts' maxima, from the row
            for (uint64_t m = late; m; m &= m - 1) {
                const int j0 = __builtin_ctzll(m) * a.pv * VEC, j1 = min(j0 + a.pv * VEC, V);
#pragma unroll 1
                for (int id = j0 + t; id < j1; id += NT) {
                    const float v = Elt<T>::scalar(row + id);
                    nf |= __builtin_amdgcn_class(v, 0x203);   // NaN or +inf
                    mx = fmaxf(mx, v);
                }
            }
            mx = wave_max_f32(mx);
            nf = __any(nf) ? 1 : 0;
            if ((t & 63) == 0) {
                L.shf[t >> 6] = mx;
                L.misc[t >> 6] = nf;
            }
            lds_sync();
#pragma unroll
            for (int j = 0; j < NW; ++j) {
                mx = fmaxf(mx, L.shf[j]);
                nf |= L.misc[j];
            }
        }
    }
    const float temp = a.params[b].temperature;
    const bool div = temp != 1.0f;
    mx = scaled(mx, temp);
    int st = TMS_ROW_OK;
    if (nf) st = TMS_ROW_NONFINITE;
    else if (mx == -__builtin_huge_valf()) st = TMS_ROW_ALL_MASKED;
    else if (mx == __builtin_huge_valf()) st = TMS_ROW_NONFINITE;
    const double md = (double)mx;
    int64_t z = 0;
    if (st == TMS_ROW_OK)
        z = div ? row_z<T, NS, NT, true>(q, nv, 1.0 / (double)temp, md, L.tab)
                : row_z<T, NS, NT, false>(q, nv, 1.0, md, L.tab);
    {   // Z: each wave's share in LDS words written once (one barrier)
        const int64_t wz = wave_incl_scan_i64_dpp(z);
        if ((t & 63) == 63) L.shl[t >> 6] = wz;
        lds_sync();
        z = 0;
        if (t == 0)
#pragma unroll
            for (int j = 0; j < NW; ++j) z += L.shl[j];
    }
    if (t == 0 && a.S > 1) st_agent(rp + 2 * p + 1, (uint64_t)z);
    if (t == 0 && p == 0) {
        const int64_t ex = (st == TMS_ROW_OK && xin) ? weight(xv, temp, md, L.tab) : 0;
        uint64_t* w = (uint64_t*)(a.stats + (int64_t)b * (2 * a.k + 1) + i);
        st_agent(&w[0], (uint64_t)__float_as_uint(mx) | ((uint64_t)(uint32_t)st << 32));
        st_agent(&w[1], (uint64_t)z);
        st_agent(&w[2], (uint64_t)ex);
        st_agent(&w[3], (uint64_t)0);
    }
}

}  // namespace tms

// Workgroups of a kernel that are resident at once on the current device
// (occupancy x compute units, looked up once per device and kernel); 0 if
// it cannot be told.
template <auto Kernel, int NT>
static int resident_cap() {
    constexpr int kMaxDevices = 64;
    static std::atomic<int> cap[kMaxDevices];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 0;
    int c = cap[dev].load(std::memory_order_relaxed);
    if (c == 0) {
        int per_cu = 0, cus = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, Kernel, NT, 0) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        c = per_cu * cus;
        cap[dev].store(c, std::memory_order_relaxed);
    }
    return c;
}

template <typename T>
static int launch_verify(tms::SArgs s, hipStream_t stream) {
    constexpr int VEC = tms::Elt<T>::kVec;
    constexpr int NSMAX = tms::kSpecPartIds / VEC / tms::kRowT;
    static_assert(tms::kSpecBlock == tms::kBlock, "the plan's resolve block");
    const tms::SpecPlan p = tms::spec_plan(
        s.B, s.k, s.V, VEC, resident_cap<tms::spec_row_kernel<T, NSMAX, tms::kRowT>, tms::kRowT>(),
        resident_cap<tms::spec_resolve_kernel<T, true>, tms::kBlock>());
    s.P = p.P;
    s.Lp = p.Lp;
    s.claim_parts = p.claim_parts;
    s.S = p.S;
    s.pv = p.pv;
    s.lazy = p.lazy;
    s.claim_rows = p.claim_rows;
    const dim3 g1((unsigned)p.n1), b1(tms::kRowT), g2((unsigned)p.n2), b2(tms::kBlock);
    if (p.ns == 1)
        hipLaunchKernelGGL((tms::spec_row_kernel<T, 1, tms::kRowT>), g1, b1, 0, stream, s);
    else if (p.ns == NSMAX / 2)
        hipLaunchKernelGGL((tms::spec_row_kernel<T, NSMAX / 2, tms::kRowT>), g1, b1, 0, stream, s);
    else
        hipLaunchKernelGGL((tms::spec_row_kernel<T, NSMAX, tms::kRowT>), g1, b1, 0, stream, s);
    if (p.wait)
        hipLaunchKernelGGL((tms::spec_resolve_kernel<T, true>), g2, b2, 0, stream, s);
    else
        hipLaunchKernelGGL((tms::spec_resolve_kernel<T, false>), g2, b2, 0, stream, s);
    return hipGetLastError() == hipSuccess ? TMS_OK : TMS_ERR_HIP;
}

// Test hook: polls of a wait for another workgroup (negative: the default).
extern "C" int tms_debug_spec_polls(tms_context* ctx, int polls) {
    if (!ctx) return TMS_ERR_INVALID_ARG;
    ctx->spec_polls = polls < 0 ? tms::kSpecPolls : polls;
    return TMS_OK;
}

extern "C" int tms_spec_verify(tms_context* ctx, const tms_spec_args* a, hipStream_t stream) {
    if (!ctx || !a || !a->target_logits || !a->draft_logits || !a->draft_tokens || !a->params ||
        !a->out_accepted || !a->out_token || !a->out_status)
        return TMS_ERR_INVALID_ARG;
    if (a->batch <= 0 || a->k < 1 || a->k > tms::kSpecMaxK || a->vocab <= 0)
        return TMS_ERR_INVALID_ARG;
    if (a->batch > ctx->max_batch || a->vocab > ctx->max_vocab) return TMS_ERR_CAPACITY;
    int esz;
    switch (a->dtype) {
        case TMS_DTYPE_F32: esz = 4; break;
        case TMS_DTYPE_F16:
        case TMS_DTYPE_BF16: esz = 2; break;
        default: return TMS_ERR_INVALID_ARG;
    }
    const int vec = 16 / esz;
    tms::SArgs s{};
    s.target = a->target_logits;
    s.draft = a->draft_logits;
    s.B = a->batch;
    s.k = a->k;
    s.V = a->vocab;
    s.fast = ((uintptr_t)a->target_logits % 16 == 0) && ((uintptr_t)a->draft_logits % 16 == 0) &&
             (a->vocab % vec == 0);
    s.tokens = a->draft_tokens;
    s.params = a->params;
    s.draws = a->draws;
    s.out_acc = a->out_accepted;
    s.out_tok = a->out_token;
    s.out_status = a->out_status;
    s.stats = ctx->spec_stats;
    s.parts = ctx->spec_parts;
    s.tickets = ctx->spec_tickets;
#ifdef TMS_TRACE
    s.trace = tms::g_spec_trace;
#endif
    s.rparts = ctx->spec_rparts;
    s.claims = ctx->spec_claims;
    s.polls = ctx->spec_polls;
    switch (a->dtype) {
        case TMS_DTYPE_F32: return launch_verify<float>(s, stream);
        case TMS_DTYPE_F16: return launch_verify<_Float16>(s, stream);
        default: return launch_verify<tms::Bf16>(s, stream);
    }
}
