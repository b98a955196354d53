// tms_topp.hip -- the whole-vocabulary kernel: top-p rows with thousands of
// significant entries (nucleus sampling without a top-k, and sampling from
// the plain softmax), exactly as tmsample::sample (tensormark/tmsample.h:
// 177-200) samples them.  It follows the general kernel (tms_sample.hip),
// which marks such rows.
//
// A row is not sorted.  Its workgroups first describe it chunk by chunk
// (record, tms_topp.h): per 1/25-wide bucket of lg, how many entries lie above
// it, their softmax mass, and the ids in bucket order.  That places the
// top-p cut, the min-p cut and the draw in a bucket each (`plan`, `select`);
// the few thousand entries of those buckets (runs of the chunks' ids in bucket
// order) are fetched and ordered in LDS, and the decisions are taken from prefix sums
// within a proven margin of the reference's left-to-right sums.  What the
// margin does not decide, and rows outside the limits below, take the exact
// full-row form (tms_dense.h).
//
// top_p = 1 is never decided by a margin: the reference stops at the first
// entry whose running sum of rounded quotients reaches 1.0.  Those rows run
// the reference's own additions, bit for bit but in parallel.  While a
// running sum s stays in one binade it is a whole multiple S of its ulp U, and
// one rounded addition is S += round(x / U): the increment depends on S only
// through its parity, and only when x / U is a tie.  So an entry is a function
// of the parity of S (SeqFn), functions compose associatively, and the row's
// workgroups each order one range of buckets in LDS and compose its
// functions, leaving out the few entries at which s may change its binade;
// the row's first workgroup composes the ranges.  Twice: z, then the sums of
// pr / z.  The serial loop that this replaces took about 290 ns an entry: a
// call of B = 32, V = 256000 fp16 with six such rows 79.0 ms, now 0.15.
//
// Bound by latency, not by bytes: a nucleus row of V = 128256 takes 50.6 us
// (2294 sorted whole) as a chain of the general kernel's lists (10), the
// records (9: LDS atomics), the plan (7), the bucket search and fetch (7), the
// ordering (4) and the sums and pick (5 to 14); 64 of them 72.2 us (3422).
//
// The first workgroups of the launch take a row each, the rest, up to one a CU
// in all, help them.  A chunk or a range is claimed by an atomic counter, so no
// workgroup waits for one that has not started: whoever runs takes what is
// left.
//
// A row's records and items are a slot of the workspace: the row's place among
// the call's rows while those have a slot each.  More rows than slots (as many
// as CUs, each of which holds one workgroup) take theirs by a lock and give
// them back, and have no helpers, which could still be reading one.

#include "tms_dense.h"
#include "tms_topp.h"

namespace tms {
namespace topp {

__constant__ double kExpTab[64] = {TMS_EXP2_64THS};

constexpr int kT = 1024;         // threads: one workgroup a CU, by LDS
constexpr int kW = kT / 64;
constexpr int kPer = 11;         // entries of a range a thread (odd: its LDS words fall on distinct banks)
constexpr int kRange = kPer * kT;
constexpr int kSel = 4096;       // keys of a selection
constexpr int kSelPer = kSel / kT;
constexpr int kSelBuckets = 2 * kT;
constexpr int kSub = 16 * kT;    // sub-buckets of a range
constexpr int kItems = 512;      // items of a row's ranges, composed in LDS
constexpr int kNone = 0x7FFFFFFF;
constexpr int kWindow = 32767;   // window positions of a row, at most: 15-bit counts
constexpr int kMaxSeg = 64;        // (interval, chunk) runs of a fetch
constexpr int kGrace = 1 << 8;   // polls before the first workgroup takes over unclaimed ranges
// Shared words of a row (u32 index; the general kernel zeroed them).
enum { kCtlState = 0, kCtlClaim = 1, kCtlDone1 = 2, kCtlPhase = 3, kCtlDone2 = 4, kCtlTaken = 6, kCtlZ = 8,
       kCtlSum = 10, kCtlAt = 12, kCtlReach = 13, kCtlKeep = 14, kCtlChunk = 16, kCtlChunks = 17, kCtlForm = kToppForm };

struct Lds {
    union {
        struct {
            uint32_t k[kRange];      // ~okey(lg): lg descending
            uint32_t cnt[kSub];
            uint32_t mixed[kSub / 32];
        } r;
        double x[kRange];   // a range's ordered weights
        struct {            // record(): a chunk
            uint32_t win[kHistIds / 2];   // window counts, 16 bits an id: bit 15 once an owner has it
            double mass[kHistBuckets];
            uint32_t cnt[kHistBuckets];
            uint64_t ext[kHistExtra];
            uint16_t ids[kHistIds + kHistExtra];
        } h;
        struct {
            uint64_t keys[kSel], srt[kSel];
            int cnt[kSelBuckets];
            uint32_t mixed[kSelBuckets / 32];
        } s;
        DenseLds d;
    } u;
    double pm[kHistBuckets];             // mass above bucket J (in units of the maximum's)
    int pc[kHistBuckets];                // entries above bucket J
    double tab[64];
    uint64_t items[3 * kItems];
    uint8_t item_r[kItems];
    uint64_t head[kMaxChunks];
    double cw[32];          // plan(): the chunks' scales
    int shift[32], lost;
    int seg_at[kMaxSeg], seg_src[kMaxSeg];
    double wd[kW];
    int wi[2 * kW];
    int64_t sw[2][kW][2];
    int raw[kToppRawMax], se[kToppRawMax + 1];   // emit(): raw entries, the runs' binades
    int mine[kToppRanges];
    int off[kToppRanges + 1];
    int misc[8];
    double dm[4];
    int at_j[3], at_n[3];   // select(): an interval's first bucket, its first rank less its first entry
    int64_t res[4];
};

// What every workgroup of a row knows after plan().
struct Row {
    int row, slot, V, K, S, CE, words;   // CE ids a chunk, `words` a record
    float mx;        // the row's maximum of lg
    int top;         // its bucket
    int n;           // entries within the histogram's span
    double z;        // their mass, up to rounding
    double rel;      // margin of prefix sums against the reference's, relative
    float temp;
    bool divide, window;
    int from, nrec;  // the window's positions
};

// A value every thread holds, as the scalar it is.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double uni(double v) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    return __longlong_as_double((long long)((uint64_t)(uint32_t)uni((int)(u >> 32)) << 32 | (uint32_t)uni((int)u)));
}

// f() in thread 0, and every thread's value of f().  Every branch on thread 0
// in this file is one of these: where two of them meet around a loop's backedge
// with no barrier between, the compiler may otherwise merge them, and take the
// other threads round the loop, and through its barriers, without thread 0.
// (The wave barrier is a convergent no-op.)
template <typename F>
__device__ __forceinline__ void once(F&& f) {
    if (threadIdx.x == 0) f();
    __builtin_amdgcn_wave_barrier();
}
template <typename F>
__device__ __forceinline__ uint32_t from_first(int& word, F&& f) {
    once([&] { word = (int)f(); });
    lds_sync();
    const uint32_t v = (uint32_t)uni(word);
    lds_sync();
    return v;
}

__device__ __forceinline__ int excl_i(int v, int& total, Lds& L) {
    const int w = threadIdx.x >> 6;
    const int inc = wave_incl_scan_i32(v);
    if ((threadIdx.x & 63) == 63) L.wi[w] = inc;
    lds_sync();
    int base = 0;
    total = 0;
#pragma unroll
    for (int i = 0; i < kW; ++i) {
        const int x = L.wi[i];
        base += i < w ? x : 0;
        total += x;
    }
    lds_sync();
    total = uni(total);
    return base + inc - v;
}

// Exclusive prefix of non-negative doubles in thread order.
__device__ __forceinline__ double excl_d(double v, double& total, Lds& L) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const double inc = wave_incl_scan_f64(v);
    if (lane == 63) L.wd[w] = inc;
    lds_sync();
    double base = 0.0;
    total = 0.0;
#pragma unroll
    for (int i = 0; i < kW; ++i) {
        const double x = L.wd[i];
        base += i < w ? x : 0.0;
        total += x;
    }
    lds_sync();
    total = uni(total);
    const uint64_t up = __shfl_up((unsigned long long)__double_as_longlong(inc), 1, 64);
    return base + (lane ? __longlong_as_double((long long)up) : 0.0);
}

__device__ __forceinline__ int block_min2(int v, int v2, int& r2, Lds& L) {   // both >= 0
    v = wave_min_nonneg(v);
    v2 = wave_min_nonneg(v2);
    if ((threadIdx.x & 63) == 0) {
        L.wi[threadIdx.x >> 6] = v;
        L.wi[kW + (threadIdx.x >> 6)] = v2;
    }
    lds_sync();
    int r = L.wi[0];
    r2 = L.wi[kW];
#pragma unroll
    for (int i = 1; i < kW; ++i) {
        r = min(r, L.wi[i]);
        r2 = min(r2, L.wi[kW + i]);
    }
    lds_sync();
    r2 = uni(r2);
    return uni(r);
}

__device__ __forceinline__ int block_min(int v, Lds& L) {   // v >= 0
    v = wave_min_nonneg(v);
    if ((threadIdx.x & 63) == 0) L.wi[threadIdx.x >> 6] = v;
    lds_sync();
    int r = L.wi[0];
#pragma unroll
    for (int i = 1; i < kW; ++i) r = min(r, L.wi[i]);
    lds_sync();
    return uni(r);
}

__device__ __forceinline__ void write_row(const KArgs& a, int row, int tok, int keep) {
    once([&] {
        a.out_tokens[row] = tok;
        a.out_status[row] = TMS_ROW_OK;
        if (a.out_keep) a.out_keep[row] = keep;
    });
}

// put(i, v, id) for the entries i in [0, m) of the buckets [j0, j1] of nI
// intervals, interval by interval: each chunk holds an interval's ids as
// one run, so a thread's entries are found by index, U in flight.  Returns
// m; put is called for i < most only, a thread's U at a time.
template <typename T, int U, typename F>
__device__ __forceinline__ int fetch(const KArgs& a, const Row& R, int3 j0, int3 j1, int nI, int most, Lds& L, F&& put) {
    const int t = threadIdx.x;
    const uint64_t* rec = a.hist + (int64_t)R.slot * R.S * R.words;
    const T* base = (const T*)a.logits + (int64_t)R.row * a.row_stride;
    if (t < 64) {   // the runs, in one wave
        int len = 0, src = 0;
        if (t < nI * R.S) {
            const int k = t / R.S, c = t - k * R.S;
            const float cm = __uint_as_float((uint32_t)L.head[c]);
            const int b0 = k == 0 ? j0.x : k == 1 ? j0.y : j0.z, b1 = k == 0 ? j1.x : k == 1 ? j1.y : j1.z;
            const int shift = R.top - topp_bucket(cm);
            const int lo = min(max(b0 - shift, 0), kHistBuckets - 1), hi = min(max(b1 + 1 - shift, 0), kHistBuckets - 1);
            if (hi > lo && (L.head[c] >> 32)) {
                const uint32_t* cnt = (const uint32_t*)(rec + (int64_t)c * R.words + kHistCnt);
                src = (int)ld_agent(&cnt[lo]);
                len = (int)ld_agent(&cnt[hi]) - src;
            }
        }
        const int inc = wave_incl_scan_i32(len);
        L.seg_at[t] = inc - len;
        L.seg_src[t] = src;
        if (t == 63) L.misc[0] = inc;
    }
    lds_sync();
    const int m = uni(L.misc[0]), n = min(m, most);
    const int nseg = nI * R.S;
    for (int i0 = t; i0 < n; i0 += U * kT) {
        const uint64_t* rc[U];
        int lid[U], ch[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = min(i0 + u * kT, n - 1);
            int s = 0;   // the last run that starts at or below i
#pragma unroll
            for (int step = 32; step >= 1; step >>= 1)
                if (s + step < nseg && L.seg_at[s + step] <= i) s += step;
            ch[u] = s % R.S;
            rc[u] = rec + (int64_t)ch[u] * R.words;
            lid[u] = (int)ld_agent(&((const uint16_t*)(rc[u] + kHistId))[L.seg_src[s] + (i - L.seg_at[s])]);
        }
        float v[U];
        int id[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool pen = lid[u] >= kHistIds;   // a penalised entry
            id[u] = ch[u] * R.CE + lid[u];
            v[u] = Elt<T>::scalar(base + (pen ? 0 : id[u]));
            if (pen) {
                const uint64_t x = ld_agent(&rc[u][kHistExt + lid[u] - kHistIds]);
                v[u] = __uint_as_float((uint32_t)(x >> 32));
                id[u] = (int)(uint32_t)x;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i0 + u * kT < n) put(i0 + u * kT, v[u], id[u]);
    }
    return m;
}

// The record of the row's chunk c (tms_topp.h).  The chunk's entries stay in
// registers, 16 a thread: the window's ids leave the stream and come back
// penalised (apply_pen) from the first position to count them, then one pass
// adds every entry's mass and count to its bucket (LDS atomics, four
// exponentials in flight; the count before is its place there) and one
// writes its id.
template <typename T>
__device__ __forceinline__ void record(const KArgs& a, const Row& R, const tms_row_params& P, int c, Lds& L) {
    constexpr int VEC = Elt<T>::kVec, NV = kHistIds / kT, NVT = NV / VEC;
    const int t = threadIdx.x;
    auto& H = L.u.h;
    const int e0 = c * R.CE, len = min(R.CE, R.V - e0);
    const T* base = (const T*)a.logits + (int64_t)R.row * a.row_stride + e0;
    const uint32_t* mrow = a.mask + (int64_t)R.row * a.mask_stride;
    uint64_t* rec = a.hist + ((int64_t)R.slot * R.S + c) * R.words;
    const int nv = len / VEC;   // whole vectors; the row's last ids one by one
    uint4 q[NVT];
    uint32_t mw[NVT];
#pragma unroll
    for (int j = 0; j < NVT; ++j) {
        const int v = min(t + j * kT, max(nv - 1, 0));
        q[j] = nv > 0 ? ld_any(base + v * VEC) : make_uint4(0, 0, 0, 0);
        mw[j] = mrow[(e0 + v * VEC) >> 5];
    }
    lds_sync();   // (the previous use of L.u)
    for (int i = t; i < kHistBuckets; i += kT) {
        H.mass[i] = 0.0;
        H.cnt[i] = 0u;
    }
    if (t < 4) L.misc[t] = 0;
    if (R.window)
        for (int i = t; i < kHistIds / 8; i += kT) ((uint4*)H.win)[i] = make_uint4(0, 0, 0, 0);
    lds_sync();
    if (R.window) {
        const int32_t* hist = a.recent + (int64_t)R.row * a.recent_stride;
        const bool ovm = a.ov_vals != nullptr;
        for (int p = R.from + t; p < R.nrec; p += kT) {
            const int o = hist[p] - e0;
            if (o >= 0 && o < len) atomicAdd(&H.win[o >> 1], 1u << ((o & 1) * 16));
        }
        lds_sync();
        Pen pn;
        pn.on = true;
        pn.rep_on = !(P.repeat_penalty <= 1.0f);
        pn.fp_on = P.frequency_penalty != 0.0f || P.presence_penalty != 0.0f;
        pn.rep = P.repeat_penalty;
        pn.freq = P.frequency_penalty;
        pn.pres = P.presence_penalty;
        if (ovm) pn.ov = a.ov_vals + (int64_t)R.row * kHistMax;
        for (int p = R.from + t; p < R.nrec; p += kT) {
            const int o = hist[p] - e0;
            if (o < 0 || o >= len) continue;
            const int sh = (o & 1) * 16;
            const uint32_t w = (atomicOr(&H.win[o >> 1], 0x8000u << sh) >> sh) & 0xFFFFu;
            if (w & 0x8000u) continue;   // another position of the id has it
            if (!((mrow[(e0 + o) >> 5] >> ((e0 + o) & 31)) & 1u)) continue;
            // (with the history pre-pass: the value of list position p)
            const float v = apply_pen<true>(Elt<T>::scalar(base + o), ovm ? (uint32_t)(p + 1) : w, pn);
            const int x = atomicAdd(&L.misc[0], 1);
            if (x < kHistExtra) H.ext[x] = (uint64_t)__float_as_uint(v) << 32 | (uint32_t)(e0 + o);
        }
        lds_sync();
    }
    const int nxt = uni(L.misc[0]), nx = min(nxt, kHistExtra);
    const bool lost = nxt > kHistExtra;
    // the entries, -inf where masked, penalised or past the row
    const float NEG = -__builtin_huge_valf();
    float x[NV], mxv = NEG;
#pragma unroll
    for (int j = 0; j < NVT; ++j) {
        const int v = t + j * kT;
        float f[VEC];
        Elt<T>::widen(q[j], f);
        uint32_t m = v < nv ? mw[j] >> ((e0 + v * VEC) & 31) : 0u;
        if (R.window && v < nv) {
#pragma unroll
            for (int e = 0; e < VEC; e += 2) {
                const uint32_t w = H.win[(v * VEC + e) >> 1];
                m &= ~((w & 0xFFFFu ? 1u : 0u) << e | (w >> 16 ? 2u : 0u) << e);
            }
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            x[j * VEC + e] = (m >> e) & 1u ? f[e] : NEG;
            mxv = fmaxf(mxv, x[j * VEC + e]);
        }
    }
    // the ids past the last whole vector (fewer than VEC, in the row's last
    // chunk) and the penalised entries: one value a thread and turn
    const int tail = len - nv * VEC;
    auto odd = [&](int i, int& local) {   // the i-th of them
        if (i < tail) {
            const int o = nv * VEC + i;
            const bool on = (mrow[(e0 + o) >> 5] >> ((e0 + o) & 31)) & 1u;
            const bool w = R.window && ((H.win[o >> 1] >> ((o & 1) * 16)) & 0xFFFFu);
            local = o;
            return on && !w ? Elt<T>::scalar(base + o) : NEG;
        }
        local = kHistIds + i - tail;
        return __uint_as_float((uint32_t)(H.ext[i - tail] >> 32));
    };
    for (int i = t; i < tail + nx; i += kT) {
        int local;
        mxv = fmaxf(mxv, odd(i, local));
    }
    mxv = wave_max_f32_dpp(mxv);
    if ((t & 63) == 0) L.wi[t >> 6] = (int)okey(mxv);
    lds_sync();
    uint32_t ko = (uint32_t)L.wi[0];
#pragma unroll
    for (int w = 1; w < kW; ++w) ko = max(ko, (uint32_t)L.wi[w]);
    mxv = okey_inv((uint32_t)uni((int)ko));
    const float lmax = R.divide ? mxv / R.temp : mxv;
    const int top = topp_bucket(lmax);
    auto bucket = [&](float v, float& lg) {
        lg = R.divide ? v / R.temp : v;
        return v == NEG ? kHistBuckets - 1 : min(top - topp_bucket(lg), kHistBuckets - 1);
    };
    // jb: the bucket, with the entry's place in it (the count before) above
    static_assert(kHistBuckets == 1024 && kHistIds + kHistExtra < 1 << 21, "bucket and place in 31 bits");
    auto add = [&](int& jb, double w) {
        if (jb < kHistBuckets - 1) {
            __hip_atomic_fetch_add(&H.mass[jb], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            jb |= (int)atomicAdd(&H.cnt[jb], 1u) << 10;
        }
    };
    auto place = [&](int jb, int local) {
        if (jb != kHistBuckets - 1) H.ids[H.cnt[jb & (kHistBuckets - 1)] + (jb >> 10)] = (uint16_t)local;
    };
    int jb[NV];
#pragma unroll
    for (int g = 0; g < NV; g += 4) {
        if (g / VEC * kT * VEC >= len) {   // a small chunk's empty slots
#pragma unroll
            for (int u = 0; u < 4; ++u) jb[g + u] = kHistBuckets - 1;
            continue;
        }
        double w[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            float lg;
            jb[g + u] = bucket(x[g + u], lg);
            w[u] = exp_span(fmax((double)lg - (double)lmax, -42.0), L.tab);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) add(jb[g + u], w[u]);
        __builtin_amdgcn_sched_barrier(0);
    }
    static_assert(VEC + kHistExtra <= 2 * kT, "two odd entries a thread");
    int jo[2], lo[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int i = t + u * kT;
        jo[u] = kHistBuckets - 1;
        if (i < tail + nx) {
            float lg;
            jo[u] = bucket(odd(i, lo[u]), lg);
            add(jo[u], exp_span(fmax((double)lg - (double)lmax, -42.0), L.tab));
        }
    }
    lds_sync();
    int total;
    const int above = excl_i((int)H.cnt[t], total, L);
    st_agent(&rec[t], (uint64_t)__double_as_longlong(H.mass[t]));
    H.cnt[t] = (uint32_t)above;
    lds_sync();
    if (t < kHistBuckets / 2) st_agent(&rec[kHistCnt + t], ((const uint64_t*)H.cnt)[t]);
    for (int i = t; i < nx; i += kT) st_agent(&rec[kHistExt + i], H.ext[i]);
    lds_sync();
#pragma unroll
    for (int g = 0; g < NV; ++g) place(jb[g], (t + g / VEC * kT) * VEC + g % VEC);
#pragma unroll
    for (int u = 0; u < 2; ++u) place(jo[u], lo[u]);
    lds_sync();
    for (int i = t; i < (total + 3) / 4; i += kT) st_agent(&rec[kHistId + i], ((const uint64_t*)H.ids)[i]);
    once([&] { st_agent(&rec[kHistHead], (uint64_t)(lost ? 0 : 1) << 32 | __float_as_uint(lmax)); });
}

// The row, as every workgroup of it sees it before its records are read.
// False: outside this kernel's limits.
__device__ __forceinline__ bool describe(const KArgs& a, int row, const tms_row_params& P, Row& R) {
    R.row = row;
    R.V = a.V;
    R.S = a.S;
    R.CE = a.CE;
    R.words = hist_words(a.CE);
    R.K = (P.top_k <= 0 || P.top_k > a.V) ? a.V : P.top_k;
    R.temp = P.temperature;
    R.divide = P.temperature != 1.0f;
    int nrec = 0;
    if (a.recent) {
        nrec = a.n_recent ? a.n_recent[row] : (int)a.recent_stride;
        nrec = min(nrec, (int)a.recent_stride);
    }
    const bool ovm = a.ov_vals != nullptr;
    R.window = nrec > 0 && (ovm || (P.repeat_last_n > 0 && (!(P.repeat_penalty <= 1.0f) ||
                                                            P.frequency_penalty != 0.0f || P.presence_penalty != 0.0f)));
    R.nrec = nrec;
    R.from = !ovm && nrec > P.repeat_last_n ? nrec - P.repeat_last_n : 0;
    return !R.window || nrec - R.from <= kWindow;
}

// Merges the row's chunk records: counts and masses above every bucket.
// False: outside this kernel's limits.  Counts are the same in every
// workgroup of the row.
__device__ __forceinline__ bool plan(const KArgs& a, Row& R, Lds& L) {
    const int t = threadIdx.x;
    const uint64_t* rec = a.hist + (int64_t)R.slot * R.S * R.words;
    if (t < a.S) L.head[t] = ld_agent(&rec[(int64_t)t * R.words + kHistHead]);
    once([&] { L.lost = 0; });
    lds_sync();
    float mx = -__builtin_huge_valf();
    for (int c = 0; c < a.S; ++c) mx = fmaxf(mx, __uint_as_float((uint32_t)L.head[c]));
    mx = __uint_as_float((uint32_t)uni((int)__float_as_uint(mx)));
    R.mx = mx;
    R.top = topp_bucket(mx);
    if (t < a.S) {
        // a chunk's scale and the shift of its buckets; 0: nothing of it is
        // within the span
        const float cm = __uint_as_float((uint32_t)L.head[t]);
        const double d = (double)cm - (double)mx;
        const bool in = d >= -41.5;
        L.cw[t] = in ? exp_span(fmax(d, -42.0), L.tab) : 0.0;
        L.shift[t] = in ? R.top - topp_bucket(cm) : kHistBuckets;
        // (entries that a record lost may lie above its maximum, and above the row's)
        if (!(L.head[t] >> 32)) L.lost = 1;
    }
    lds_sync();
    double m = 0.0;
    int n = 0;
    const bool lost = uni(L.lost) != 0;
    for (int c0 = 0; c0 < a.S; c0 += 8) {   // eight chunks' words in flight
        double hm[8];
        int h0[8], h1[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int c = min(c0 + u, a.S - 1);
            const int j = max(t - L.shift[c], 0);   // at most kHistBuckets - 1
            const uint64_t* h = rec + (int64_t)c * R.words;
            const uint32_t* cnt = (const uint32_t*)(h + kHistCnt);
            hm[u] = __longlong_as_double((long long)ld_agent(&h[j]));
            h0[u] = (int)ld_agent(&cnt[j]);
            h1[u] = (int)ld_agent(&cnt[min(j + 1, kHistBuckets - 1)]);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int c = min(c0 + u, a.S - 1);
            if (c0 + u < a.S && t >= L.shift[c] && t < kHistBuckets - 1) {
                m += L.cw[c] * hm[u];
                n += h1[u] - h0[u];
            }
        }
    }
    if (lost) return false;   // (more penalised entries than a record holds)
    double z;
    int tot;
    L.pm[t] = excl_d(m, z, L);
    L.pc[t] = excl_i(n, tot, L);
    R.z = z;
    R.n = tot;
    // A prefix sum of masses against the reference's left-to-right sums of
    // rounded quotients: at most 2n + 1 roundings there, n + 64 here and n +
    // 64 in the divisor, 2^-50 a mass, and n e^-40.9 left out.
    R.rel = (4.0 * (double)tot + 256.0) * 0x1p-53 + 0x1p-40;
    lds_sync();
    return true;
}

// The first buckets whose entries bring the mass to at least x0 and x1 (the
// count to at least n); kHistBuckets - 1 where none does.
__device__ __forceinline__ void buckets_of(double x0, double x1, int n, int& b0, int& b1, int& bn, Lds& L) {
    const int t = threadIdx.x;
    const bool in = t < kHistBuckets - 1;
    const double m = in ? L.pm[t + 1] : 0.0;
    b0 = block_min2(in && m >= x0 ? t : kHistBuckets - 1, in && m >= x1 ? t : kHistBuckets - 1, b1, L);
    bn = kHistBuckets - 1;
    if (n > 0) bn = block_min(in && L.pc[t + 1] >= n ? t : kHistBuckets - 1, L);
}

enum : int { SEL_DONE = 0, SEL_EXACT = 1, SEL_WHOLE = 2 };

// The row's cut and draw from the histogram and the entries of the buckets
// they fall in.  SEL_DONE: the row is written.  SEL_EXACT: top_p = 1 decides
// the kept prefix; tok / rank then hold the draw's entry (from the whole
// mass) and the id lists are written.  SEL_WHOLE: the full-row form.
template <typename T>
__device__ __forceinline__ int select(const KArgs& a, const tms_row_params& P, const Row& R, Lds& L, int& tok, int& rank) {
    const int t = threadIdx.x;
    constexpr int kEnd = kHistBuckets - 1;
    const double z = R.z, thr = (double)P.top_p * z;
    const bool minp = P.min_p > 0.0f;
    if (P.top_p != P.top_p || P.min_p != P.min_p) return SEL_WHOLE;
    // The cut's buckets.
    int32_t* ids = a.out_topk_ids ? a.out_topk_ids + (int64_t)R.row * a.topk_cap : nullptr;
    float* probs = a.out_topk_probs ? a.out_topk_probs + (int64_t)R.row * a.topk_cap : nullptr;
    const int cap = (ids || probs) ? a.topk_cap : 0;
    if (R.n < R.K && cap > R.n) return SEL_WHOLE;
    int p0, p1, t1;
    buckets_of(thr - z * R.rel * 4.0, thr + z * R.rel * 4.0, min(cap, R.n), p0, p1, t1, L);
    if (!cap) t1 = -1;
    bool cut_p = false, exact = false;
    if (P.top_p <= 1.0f) {
        cut_p = p1 < kEnd;
        exact = !cut_p;   // the threshold is within the margin of the whole mass
    } else {
        p0 = p1 = kEnd;
    }
    int m0 = kEnd, m1 = kEnd;
    if (minp) {
        const double lm = (double)R.mx + log((double)P.min_p);
        const double slack = 1e-5 + 1e-6 * fabs(lm);
        m0 = max(0, R.top - topp_bucket((float)(lm + slack)));
        m1 = max(0, R.top - topp_bucket((float)(lm - slack)));
        if (m1 >= kEnd) return SEL_WHOLE;
    }
    bool use_p = cut_p, use_m = minp;
    if (minp && m1 < p0) {
        use_p = exact = false;
    } else if (minp && m0 > p1) {
        use_m = false;
    }
    if (exact && P.top_p != 1.0f) return SEL_WHOLE;
    if (exact && use_m) return SEL_WHOLE;
    int k0 = kEnd, k1 = -1;   // the interval that decides the kept prefix
    if (use_p) {
        k0 = min(k0, p0);
        k1 = max(k1, p1);
    }
    if (use_m) {
        k0 = min(k0, m0);
        k1 = max(k1, m1);
    }
    // The draw's buckets, for every sum the cut may leave.
    const double s0 = k1 >= 0 ? uni(L.pm[k0]) : z, s1 = k1 >= 0 ? uni(L.pm[k1 + 1]) : z;
    uint32_t w0, w1;
    row_uniform(a, R.row, P, w0, w1);
    const double u = canonical(w0, w1);
    int d0, d1, none;
    buckets_of(u * s0 - z * R.rel * 4.0, u * s1 + z * R.rel * 4.0, 0, d0, d1, none, L);
    if (k1 >= 0) d1 = min(d1, k1);
    if (d0 >= kEnd || d1 >= kEnd) return SEL_WHOLE;
    // The intervals [g0, g1], ascending and disjoint: the id list's from 0,
    // the draw's, the cut's (d0 <= k1).
    int3 g0 = make_int3(0, d0, k0), g1 = make_int3(t1, d1, k1);
    if (g1.y >= g0.z - 1 && k1 >= 0) {   // draw and cut touch
        g0.y = min(g0.y, g0.z);
        g1.y = max(g1.y, g1.z);
        g1.z = -1;
    }
    if (g1.x >= 0 && g1.x >= g0.y - 1) {
        g0.y = 0;
        g1.y = max(g1.y, g1.x);
        g1.x = -1;
        if (g1.z >= 0 && g1.y >= g0.z - 1) {
            g1.y = max(g1.y, g1.z);
            g1.z = -1;
        }
    }
    if (g1.x < 0) {   // the empty ones last (the draw's is not)
        g0 = make_int3(g0.y, g0.z, 0);
        g1 = make_int3(g1.y, g1.z, -1);
    }
    auto held = [&](int b0, int b1) { return b1 < 0 ? 0 : uni(L.pc[b1 + 1]) - uni(L.pc[b0]); };
    const int n0 = held(g0.x, g1.x), n1 = held(g0.y, g1.y), n2 = held(g0.z, g1.z);
    const int m = n0 + n1 + n2, nI = 1 + (g1.y >= 0) + (g1.z >= 0);
    const int last = g1.z >= 0 ? g1.z : g1.y >= 0 ? g1.y : g1.x;
    const int st1 = g1.y >= 0 ? n0 : kNone, st2 = g1.z >= 0 ? n0 + n1 : kNone;   // their first entries
    if (m > kSel) return SEL_WHOLE;
    // ---- their keys, unordered
    for (int i = t; i < kSelBuckets; i += kT) L.u.s.cnt[i] = 0;
    const int found = fetch<T, kSelPer>(a, R, g0, g1, nI, kSel, L, [&](int i, float v, int id) {
        L.u.s.keys[i] = ckey(R.divide ? v / R.temp : v, (uint32_t)id);
    });
    if (found != m) return SEL_WHOLE;   // not what the histogram counted
    lds_sync();
    // ---- ordered: sub-buckets by a monotone function of lg, then each key
    //      against its own sub-bucket.  16-bit logits tie by the hundreds: a
    //      large sub-bucket of one value is left in any order (its prefix sums
    //      do not depend on it) unless the id list reaches into it.
    constexpr int kBig = 48;
    const float qlo = (float)(R.top - last) / kHistScale;
    const float span = (float)(R.top - g0.x + 1) / kHistScale - qlo;
    const float scale = span > 0.0f ? (float)(kSelBuckets - 1) / span : 0.0f;
    auto sub = [&](uint64_t k) {
        const float f = (ckey_val(k) - qlo) * scale;
        return f >= (float)(kSelBuckets - 1) ? kSelBuckets - 1 : (f >= 1.0f ? (int)f : 0);
    };
    {
        uint64_t k[kSelPer];
        int b[kSelPer], slot[kSelPer];
#pragma unroll
        for (int s = 0; s < kSelPer; ++s) {
            const int i = t + s * kT;
            k[s] = i < m ? L.u.s.keys[i] : 0ull;
            b[s] = slot[s] = 0;
            if (k[s]) {
                b[s] = sub(k[s]);
                slot[s] = atomicAdd(&L.u.s.cnt[b[s]], 1);
            }
        }
        lds_sync();
        const int c0 = L.u.s.cnt[kSelBuckets - 1 - 2 * t], c1 = L.u.s.cnt[kSelBuckets - 2 - 2 * t];
        int tot;
        const int at = excl_i(c0 + c1, tot, L);
        L.u.s.cnt[kSelBuckets - 1 - 2 * t] = at;
        L.u.s.cnt[kSelBuckets - 2 - 2 * t] = at + c0;
        for (int i = t; i < kSelBuckets / 32; i += kT) L.u.s.mixed[i] = 0u;
        lds_sync();
#pragma unroll
        for (int s = 0; s < kSelPer; ++s)
            if (k[s]) L.u.s.keys[L.u.s.cnt[b[s]] + slot[s]] = k[s];
        lds_sync();
#pragma unroll
        for (int s = 0; s < kSelPer; ++s)
            if (k[s] && (uint32_t)(L.u.s.keys[L.u.s.cnt[b[s]]] >> 32) != (uint32_t)(k[s] >> 32))
                atomicOr(&L.u.s.mixed[b[s] >> 5], 1u << (b[s] & 31));
        lds_sync();
#pragma unroll
        for (int s = 0; s < kSelPer; ++s) {
            if (!k[s]) continue;
            const int lo = L.u.s.cnt[b[s]], hi = b[s] > 0 ? L.u.s.cnt[b[s] - 1] : m;
            int r = lo;
            if (hi - lo <= kBig || lo < cap || ((L.u.s.mixed[b[s] >> 5] >> (b[s] & 31)) & 1u))
                for (int j = lo; j < hi; ++j) r += L.u.s.keys[j] > k[s] ? 1 : 0;
            else
                r += slot[s];
            L.u.s.srt[r] = k[s];
        }
        lds_sync();
    }
    // ---- their prefix sums: entry i of interval k has global rank
    //      pc[its first bucket] + i - its first entry, and the mass above the
    //      interval in front
    const double mxd = (double)R.mx;
    double pr[kSelPer], pre[kSelPer];
    int rk[kSelPer];
    double loc = 0.0;
#pragma unroll
    for (int s = 0; s < kSelPer; ++s) {
        const int i = t * kSelPer + s;
        pr[s] = i < m ? exp((double)ckey_val(L.u.s.srt[i]) - mxd) : 0.0;
        loc += pr[s];
        pre[s] = loc;
        __builtin_amdgcn_sched_barrier(0);
    }
    double all;
    const double ex = excl_d(loc, all, L);
#pragma unroll
    for (int s = 0; s < kSelPer; ++s) {
        const int i = t * kSelPer + s;
        const double before = ex + (s ? pre[s > 0 ? s - 1 : 0] : 0.0);
        if (i == 0 || i == st1 || i == st2) {
            const int k = (i >= st1 ? 1 : 0) + (i >= st2 ? 1 : 0), b = k == 0 ? g0.x : k == 1 ? g0.y : g0.z;
            L.dm[k] = before;
            L.at_j[k] = b;
            L.at_n[k] = L.pc[b] - i;
        }
    }
    lds_sync();
#pragma unroll
    for (int s = 0; s < kSelPer; ++s) {
        const int i = t * kSelPer + s;
        const int k = (i >= st1 ? 1 : 0) + (i >= st2 ? 1 : 0);
        rk[s] = i < m ? L.at_n[k] + i : kNone;
        pre[s] = L.pm[L.at_j[k]] + ((ex + pre[s]) - L.dm[k]);
    }
    // The first rank below lim whose prefix / D is >= th: definitely (fd) or
    // within the margin (fm).
    auto first_ge = [&](double D, double th, int lim, int& fd, int& fm) {
        int d = kNone, q = kNone;
        const double rD = 1.0 / D, slack = R.rel * z * rD * 0x1p-6;
#pragma unroll
        for (int s = kSelPer - 1; s >= 0; --s) {
            if (rk[s] >= lim) continue;
            const double v = pre[s] * rD;
            const double mg = (v + fabs(th)) * R.rel + slack;
            if (v > th + mg) d = rk[s];
            else if (!(v < th - mg)) q = rk[s];
        }
        fd = block_min2(d, q, fm, L);
    };
    int keep = R.K;
    if (use_p) {
        int fd, fm;
        first_ge(z, (double)P.top_p, R.n, fd, fm);
        if (fd == kNone || fm < fd) return SEL_WHOLE;
        keep = min(keep, fd + 1);
    }
    if (use_m) {
        int fl = kNone;
        const double mp = (double)P.min_p;
#pragma unroll
        for (int s = kSelPer - 1; s >= 0; --s)
            if (rk[s] >= 1 && rk[s] < R.n && pr[s] < mp) fl = rk[s];
        fl = block_min(fl, L);
        if (fl == kNone) fl = L.pc[m1 + 1];   // every entry below the interval is below min_p
        keep = min(keep, max(fl, 1));
    }
    // ---- the draw
    int pick = 0;
    if (keep >= 2) {
        // the sum over the kept prefix: the prefix at rank keep - 1
        once([&] { L.misc[1] = 0; });
        lds_sync();
#pragma unroll
        for (int s = 0; s < kSelPer; ++s)
            if (rk[s] == keep - 1) {
                L.dm[3] = pre[s];
                L.misc[1] = 1;
            }
        lds_sync();
        double sum = z;
        if (k1 >= 0 && keep < R.n) {
            if (uni(L.misc[1])) sum = uni(L.dm[3]);
            else if (keep == L.pc[k0]) sum = uni(L.pm[k0]);   // the cut takes the whole bucket above
            else return SEL_WHOLE;
        }
        int gd, gm;
        const int dl = min(R.n, keep - 1);
        first_ge(sum, u, dl, gd, gm);
        if (gm < gd) return SEL_WHOLE;
        pick = gd < dl ? gd : keep - 1;
    }
    if (t < 2) L.misc[1 + t] = -1;
    lds_sync();
#pragma unroll
    for (int s = 0; s < kSelPer; ++s)
        if (rk[s] == pick) L.misc[1] = t * kSelPer + s;
    lds_sync();
    const int pi = uni(L.misc[1]);
    if (pi < 0) return SEL_WHOLE;
    {
        // the drawn entry's sub-bucket may be in any order: its entry with
        // pi - lo larger keys
        const int b = sub(L.u.s.srt[pi]), lo = L.u.s.cnt[b], hi = b > 0 ? L.u.s.cnt[b - 1] : m;
        for (int i = lo + t; i < hi; i += kT) {
            const uint64_t k = L.u.s.srt[i];
            int r = lo;
            for (int j = lo; j < hi; ++j) r += L.u.s.srt[j] > k ? 1 : 0;
            if (r == pi) L.misc[2] = (int)ckey_id(k);
        }
    }
    lds_sync();
    tok = uni(L.misc[2]);
    rank = pick;
    // (A bucket's mass is added up in no fixed order, so z differs by some 2^-50
    // of itself from call to call, and a probability by its last bit where that
    // moves its rounding, about once in 10^7.  The decisions above do not depend
    // on it: within the margin they are the full-row form's.)
    for (int i = t; i < cap; i += kT) {
        const bool have = i < R.n && i < R.K;
        const uint64_t k = have ? L.u.s.srt[i] : 0ull;
        if (ids) ids[i] = have ? (int)ckey_id(k) : -1;
        if (probs) probs[i] = have ? (float)(exp((double)ckey_val(k) - mxd) / z) : 0.0f;
    }
    if (exact) return SEL_EXACT;
    write_row(a, R.row, tok, keep);
    return SEL_DONE;
}

// ---- rows with top_p = 1: the reference's sums

// One rounded addition to a sum of either parity, in ulps of the sum.
struct SeqFn {
    int64_t a0, a1;   // increment of an even, of an odd sum
    __device__ __forceinline__ int64_t at(int64_t s) const { return a0 + ((a1 - a0) & -(s & 1)); }
};
__device__ __forceinline__ SeqFn then(const SeqFn& f, const SeqFn& g) {
    return {f.a0 + g.at(f.a0), f.a1 + g.at(1 + f.a1)};
}
__device__ __forceinline__ SeqFn seq_fn(double y) {   // y = x / U, below 2^53; ties go to the even sum
    const double m = floor(y);
    const int64_t f = (int64_t)m;
    const bool tie = y - m == 0.5;
    const int64_t up = y - m > 0.5 ? 1 : 0;
    return {f + (tie ? f & 1 : up), f + (tie ? ~f & 1 : up)};
}
__device__ __forceinline__ SeqFn shfl_down(const SeqFn& f, int d) {
    return {(int64_t)__shfl_down((long long)f.a0, d, 64), (int64_t)__shfl_down((long long)f.a1, d, 64)};
}
__device__ __forceinline__ SeqFn shfl_up(const SeqFn& f, int d) {
    return {(int64_t)__shfl_up((long long)f.a0, d, 64), (int64_t)__shfl_up((long long)f.a1, d, 64)};
}
__device__ __forceinline__ int expo(double v) { return (int)((uint64_t)__double_as_longlong(v) >> 52) - 1023; }
__device__ __forceinline__ double pow2(int e) { return __longlong_as_double((long long)(e + 1023) << 52); }
constexpr int64_t kTop = (int64_t)1 << 53;

// Range r's buckets [j0, j1) of a row cut into ranges of about Q entries.
__device__ __forceinline__ int range_begin(int x, const Lds& L) {   // first J with pc[J] >= x
    int lo = 0, hi = kHistBuckets - 1;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (uni(L.pc[mid]) >= x) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}

// The weights exp(lg - mx) of the entries of the buckets [j0, j1), ordered,
// in L.u.x, their count in n; false when the row does not hold what the
// histogram counted.  Ordered by sub-buckets of lg, then each key against its
// own sub-bucket (a large sub-bucket of one value stays in any order: its
// weights are equal).
template <typename T>
__device__ __forceinline__ bool load_range(const KArgs& a, const Row& R, int j0, int j1, int& n, Lds& L) {
    const int t = threadIdx.x, lane = t & 63;
    n = uni(L.pc[j1]) - uni(L.pc[j0]);
    lds_sync();
    for (int i = t; i < kSub; i += kT) L.u.r.cnt[i] = 0u;
    for (int i = t; i < kSub / 32; i += kT) L.u.r.mixed[i] = 0u;
    const int found = fetch<T, kPer>(a, R, make_int3(j0, 0, 0), make_int3(j1 - 1, 0, 0), 1, kRange, L, [&](int i, float v, int) {
        L.u.r.k[i] = ~okey(R.divide ? v / R.temp : v);
    });
    if (found != n || n > kRange) return false;
    lds_sync();
    const float hi_q = (float)(R.top - j0 + 1) / kHistScale, span = hi_q - (float)(R.top - j1 + 1) / kHistScale;
    const float scale = span > 0.0f ? (float)(kSub - 1) / span : 0.0f;
    uint32_t k[kPer], at[kPer];   // at: sub-bucket << 16 | place in it
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = t + j * kT;
        k[j] = i < n ? L.u.r.k[i] : 0u;
        const float f = (hi_q - okey_inv(~k[j])) * scale;
        const int b = f >= (float)(kSub - 1) ? kSub - 1 : (f >= 1.0f ? (int)f : 0);
        // Neighbouring lanes hold one bucket's entries, which tie in 16 bits:
        // the first lanes' sub-buckets are counted by ballot, one atomic for
        // all their lanes, and only what is left lane by lane.
        uint64_t todo = __ballot(i < n);
        uint32_t place = 0u;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            if (!todo) break;
            const int first = __ffsll((unsigned long long)todo) - 1;
            const int fb = __builtin_amdgcn_readlane(b, first);
            const uint64_t same = __ballot(b == fb) & todo;
            uint32_t base = 0u;
            if (lane == first) base = atomicAdd(&L.u.r.cnt[fb], (uint32_t)__popcll(same));
            base = (uint32_t)__builtin_amdgcn_readlane((int)base, first);
            if ((same >> lane) & 1ull) place = base + (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
            todo &= ~same;
        }
        if ((todo >> lane) & 1ull) place = atomicAdd(&L.u.r.cnt[b], 1u);
        at[j] = (uint32_t)b << 16 | place;
    }
    lds_sync();
    {   // counts to starts (16 words a thread, skewed over the banks)
        uint32_t c[16];
        int sum = 0, tot;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint4 w = ((const uint4*)L.u.r.cnt)[4 * t + q];
            c[4 * q] = w.x;
            c[4 * q + 1] = w.y;
            c[4 * q + 2] = w.z;
            c[4 * q + 3] = w.w;
            sum += (int)(w.x + w.y + w.z + w.w);
        }
        uint32_t b = (uint32_t)excl_i(sum, tot, L);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint4 w;
            w.x = b;
            w.y = w.x + c[4 * q];
            w.z = w.y + c[4 * q + 1];
            w.w = w.z + c[4 * q + 2];
            b = w.w + c[4 * q + 3];
            ((uint4*)L.u.r.cnt)[4 * t + q] = w;
        }
    }
    lds_sync();
#pragma unroll
    for (int j = 0; j < kPer; ++j)
        if (t + j * kT < n) L.u.r.k[L.u.r.cnt[at[j] >> 16] + (at[j] & 0xFFFFu)] = k[j];
    lds_sync();
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int b = (int)(at[j] >> 16);
        if (t + j * kT < n && L.u.r.k[L.u.r.cnt[b]] != k[j]) atomicOr(&L.u.r.mixed[b >> 5], 1u << (b & 31));
    }
    lds_sync();
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        if (t + j * kT >= n) continue;
        const int b = (int)(at[j] >> 16);
        const int lo = (int)L.u.r.cnt[b], hi = b + 1 < kSub ? (int)L.u.r.cnt[b + 1] : n;
        int r = lo + (int)(at[j] & 0xFFFFu);
        if ((L.u.r.mixed[b >> 5] >> (b & 31)) & 1u) {
            // smaller keys, and equal ones placed before it
            const int me = r;
            r = lo;
            for (int q = lo; q < hi; ++q) {
                const uint32_t o = L.u.r.k[q];
                r += o < k[j] || (o == k[j] && q < me) ? 1 : 0;
            }
        }
        at[j] = (uint32_t)r;
    }
    lds_sync();
#pragma unroll
    for (int j = 0; j < kPer; ++j)
        if (t + j * kT < n) L.u.r.k[at[j]] = k[j];
    lds_sync();
#pragma unroll
    for (int j = 0; j < kPer; ++j) k[j] = L.u.r.k[t * kPer + j];
    lds_sync();
#pragma unroll 1
    for (int j = 0; j < kPer; ++j) {   // (unrolled, the exponentials spill)
        uint32_t q = k[0];
#pragma unroll
        for (int i = 1; i < kPer; ++i) q = j == i ? k[i] : q;
        L.u.x[t * kPer + j] = t * kPer + j < n ? exp((double)okey_inv(~q) - (double)R.mx) : 0.0;
    }
    lds_sync();
    return true;
}

// Range r's items into items[]: runs of entries that stay in one binade as
// one function, the entries between them raw.  With `second` the sums are of
// quotients, and the last binade's upper end, 1.0, is the row's threshold: no
// entry is raw for it.  Items: [0] kind << 40 | (binade + 2048) << 20 | first
// entry, [1] [2] the function (kind 0) or the term (kind 1; kind 2 is empty).
__device__ __forceinline__ void emit(const Row& R, int n, double base, bool first, bool second, uint64_t* items, Lds& L) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    // the sum before the thread's first entry, up to rounding
    double s0 = 0.0, tot;
#pragma unroll 1
    for (int j = 0; j < kPer; ++j) s0 += L.u.x[t * kPer + j];
    s0 = base + excl_d(s0, tot, L);
    const double lo_f = 1.0 - 4.0 * R.rel, hi_f = 1.0 + 4.0 * R.rel;
    uint32_t rawm = 0;   // the raw entries
    {
        double s = s0;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int i = t * kPer + j;
            const double lo = s * lo_f;
            s += L.u.x[i];
            const bool last = second && lo >= 0.5;
            bool raw = !(lo > 0.0) || expo(lo) != expo(s * hi_f);
            if (last) raw = false;
            if (first && i == 0) raw = true;
            if (raw && i < n) rawm |= 1u << j;
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    int nraw;
    int at = excl_i(__popc(rawm), nraw, L);
    if (nraw > kToppRawMax) {
        once([&] { st_agent(&items[0], ~(uint64_t)0); });
        return;
    }
    once([&] { L.se[0] = second && s0 * lo_f >= 0.5 ? -1 : expo(s0 * lo_f); });
    if (rawm) {
        double s = s0;
#pragma unroll 1
        for (int j = 0; j < kPer; ++j) {
            const double x = L.u.x[t * kPer + j];
            s += x;
            if (!((rawm >> j) & 1u)) continue;
            uint64_t* q = items + 1 + 3 * (2 * at + 1);
            st_agent(&q[0], (uint64_t)1 << 40 | (uint64_t)(t * kPer + j));
            st_agent(&q[1], (uint64_t)__double_as_longlong(x));
            L.raw[at++] = t * kPer + j;
            L.se[at] = second && s * lo_f >= 0.5 ? -1 : expo(s * lo_f);   // the run after it
        }
    }
    lds_sync();
#pragma unroll 1
    for (int k = 0; k <= nraw; ++k) {
        const int lo = k ? uni(L.raw[k - 1]) + 1 : 0, hi = k < nraw ? uni(L.raw[k]) : n;
        SeqFn f{0, 0};
        // A wave's entries fall in few runs; the others it leaves out.  (An
        // entry's function is formed in its run, of whose binade it is, and not
        // kept from one run to the next: 22 registers.)
        const int w0 = (t & ~63) * kPer;
        if (hi > w0 && lo < w0 + 64 * kPer) {
            const double scale = pow2(52 - uni(L.se[k]));
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const int i = t * kPer + j;
                if (i >= lo && i < hi) f = then(f, seq_fn(L.u.x[i] * scale));
            }
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const SeqFn o = shfl_down(f, d);
                if ((lane & (2 * d - 1)) == 0) f = then(f, o);
            }
        }
        if (lane == 0) {
            L.sw[k & 1][w][0] = f.a0;
            L.sw[k & 1][w][1] = f.a1;
        }
        lds_sync();
        once([&] {
            SeqFn g{0, 0};
            for (int q = 0; q < kW; ++q) g = then(g, SeqFn{L.sw[k & 1][q][0], L.sw[k & 1][q][1]});
            uint64_t* q = items + 1 + 3 * (2 * k);
            st_agent(&q[0], lo < hi ? (uint64_t)(L.se[k] + 2048) << 20 | (uint64_t)lo : (uint64_t)2 << 40);
            st_agent(&q[1], (uint64_t)g.a0);
            st_agent(&q[2], (uint64_t)g.a1);
        });
    }
    once([&] { st_agent(&items[0], (uint64_t)(2 * nraw + 1)); });
}

// Composes the row's items in order.  res[0]: 0 the sum never reached the
// threshold (res[1] its bits), 1 it does at raw entry res[3] of range
// res[2], 2 in the run of range res[2] that starts at entry res[3] with S =
// res[1], 3 the items do not fit together.
__device__ __forceinline__ void compose(const uint64_t* items, int nr, bool second, Lds& L) {
    const int t = threadIdx.x;
    int c = 0;
    if (t < nr) {
        const uint64_t h = ld_agent(&items[(int64_t)t * kToppItemWords]);
        c = h > (uint64_t)(2 * kToppRawMax + 1) ? kItems + 1 : (int)h;
    }
    int total;
    const int at = excl_i(c, total, L);
    if (t < nr) L.off[t] = at;
    once([&] { L.off[nr] = total; });
    lds_sync();
    if (total > kItems || total < 0) {
        once([&] { L.res[0] = 3; });
        lds_sync();
        return;
    }
    if (t < total) {
        int r = 0;
        while (r + 1 < nr && L.off[r + 1] <= t) ++r;
        const uint64_t* q = items + (int64_t)r * kToppItemWords + 1 + 3 * (t - L.off[r]);
        L.items[3 * t] = ld_agent(&q[0]);
        L.items[3 * t + 1] = ld_agent(&q[1]);
        L.items[3 * t + 2] = ld_agent(&q[2]);
        L.item_r[t] = (uint8_t)r;
    }
    lds_sync();
    if (t < 64) {
        // s = S ulps of binade e.  One wave, a lane an item, the running sum
        // uniform.
        int e = 0;
        int64_t S = 0, r0 = 0, r1 = 0, r2 = 0, r3 = 0;
        auto value = [&] { return (double)S * pow2(e - 52); };
        bool stop = false;
        for (int i0 = 0; i0 < total && !stop; i0 += 64) {
            const int mine = min(i0 + t, total - 1), c = min(64, total - i0);
            const int64_t vh = (int64_t)L.items[3 * mine], v0 = (int64_t)L.items[3 * mine + 1],
                          v1 = (int64_t)L.items[3 * mine + 2];
#pragma unroll 1
            for (int i = 0; i < c; ++i) {
                const uint64_t h = (uint64_t)readlane_i64(vh, i);
                const SeqFn f{readlane_i64(v0, i), readlane_i64(v1, i)};
                const int kind = (int)(h >> 40);
                if (kind == 2) continue;
                if (kind == 0) {
                    if (S == 0 || (int)((h >> 20) & 0xFFFFF) - 2048 != e) {
                        r0 = 3;
                        stop = true;
                        break;
                    }
                    const int64_t N = S + f.at(S);
                    if (N < kTop) {
                        S = N;
                        continue;
                    }
                    r0 = second && e == -1 ? 2 : 3;
                    r1 = S;
                } else {
                    const double s = value() + __longlong_as_double((long long)f.a0);
                    e = expo(s);
                    S = (int64_t)(s * pow2(52 - e));
                    if (!(second && s >= 1.0)) continue;
                    r0 = 1;
                }
                r2 = L.item_r[i0 + i];
                r3 = (int64_t)(h & 0xFFFFF);
                stop = true;
                break;
            }
        }
        const double s = value();
        if (r0 == 0) r1 = (int64_t)__double_as_longlong(s);
        once([&] {
            L.res[0] = r0;
            L.res[1] = r1;
            L.res[2] = r2;
            L.res[3] = r3;
        });
    }
    lds_sync();
}

// The first entry at or after `lo` of a range (in LDS) whose sum reaches
// 1.0, starting from S ulps of the binade below it.
__device__ __forceinline__ int reach_one(int n, int lo, int64_t S0, Lds& L) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    SeqFn f{0, 0};
#pragma unroll 1
    for (int j = 0; j < kPer; ++j) {
        const int i = t * kPer + j;
        if (i >= lo && i < n) f = then(f, seq_fn(L.u.x[i] * pow2(53)));
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const SeqFn o = shfl_up(f, d);
        if (lane >= d) f = then(o, f);
    }
    SeqFn ex = shfl_up(f, 1);
    if (lane == 0) ex = {0, 0};
    if (lane == 63) {
        L.sw[0][w][0] = f.a0;
        L.sw[0][w][1] = f.a1;
    }
    lds_sync();
    SeqFn before{0, 0};
    for (int q = 0; q < w; ++q) before = then(before, SeqFn{L.sw[0][q][0], L.sw[0][q][1]});
    int64_t S = S0 + then(before, ex).at(S0);
    int hit = kNone;
#pragma unroll 1
    for (int j = 0; j < kPer; ++j) {
        const int i = t * kPer + j;
        if (i >= lo && i < n) S += seq_fn(L.u.x[i] * pow2(53)).at(S);
        if (hit == kNone && S >= kTop) hit = i;
    }
    return block_min(hit, L);
}

__device__ __forceinline__ uint32_t add_agent(uint32_t* p, uint32_t v) {
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Thread 0 polls until *p >= want (bounded); the result is uniform.
__device__ __forceinline__ bool wait_ge(const uint32_t* p, uint32_t want, int polls, Lds& L) {
    return from_first(L.misc[7], [&] {
        uint32_t ok = 0;
        for (int i = 0; i < polls && !ok; ++i) {
            ok = ld_agent(p) >= want ? 1u : 0u;
            if (!ok) __builtin_amdgcn_s_sleep(2);
        }
        return ok;
    }) != 0;
}

// The kept prefix of a top_p = 1 row (leader: the row's first workgroup), or
// -1 for the full-row form.  Helpers return -1.
template <typename T>
__device__ __forceinline__ int exact_keep(const KArgs& a, const Row& R, bool leader, Lds& L) {
    const int t = threadIdx.x;
    uint32_t* ctl = a.topp_ctl + (int64_t)R.row * kToppCtl;
    uint64_t* items = a.topp_items + (int64_t)R.slot * kToppRanges * kToppItemWords;
    // Ranges of at most kRange entries: whole buckets, about Q entries each.
    int big = t < kHistBuckets - 1 ? L.pc[t + 1] - L.pc[t] : 0;
    big = kRange - block_min(kRange - min(big, kRange), L);
    const int Q = kRange - big;
    const int nr = Q > 0 ? (R.n + Q - 1) / Q : 0;
    if (2 * big > kRange || nr > kToppRanges) {
        // (the leader tells nobody: no workgroup takes a range)
        return -1;
    }
    auto begin = [&](int r) { return range_begin(r * Q, L); };
    auto end = [&](int r) { return r + 1 < nr ? range_begin((r + 1) * Q, L) : kHistBuckets - 1; };
    auto take = [&](int r) {   // a range's second pass, unless another workgroup has it
        return from_first(L.misc[7], [&] {
            return (uint32_t)!((__hip_atomic_fetch_or((unsigned long long*)&ctl[kCtlTaken], 1ull << r, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT) >> r) & 1ull);
        }) != 0;
    };
    // Stages (one place does a range's work): 0 the ranges this workgroup
    // claims, for z; 1 the same ranges again, the one in LDS first, for the
    // sums of pr / z; 2 (leader) what is left of those; 3 (leader) the entry
    // at which they reach 1.0.
    enum { CLAIM, AGAIN, REST, REACH };
    int stage = CLAIM, held = -1, held_n = 0, nmine = 0, next = 0, at = 0;
    bool divided = false;   // the weights in LDS are quotients by z
    int64_t S1 = 0;
    double z = 1.0;
    bool have = false;
    for (;;) {
        int r = -1;
        if (stage == CLAIM) {
            const uint32_t q = from_first(L.misc[7], [&] { return add_agent(&ctl[kCtlClaim], 1u); });
            if (q < (uint32_t)nr) {
                r = (int)q;
                once([&] { L.mine[nmine] = r; });
                ++nmine;
            } else {
                uint64_t zb = 0;
                if (leader) {
                    // every range is claimed, by a workgroup that runs
                    const bool in = wait_ge(&ctl[kCtlDone1], (uint32_t)nr, kPollCap, L);
                    if (in) compose(items, nr, false, L);
                    zb = in && uni((int)L.res[0]) == 0 ? (uint64_t)readlane_i64(L.res[1], 0) : 0ull;
                    once([&] {
                        st_agent((uint64_t*)&ctl[kCtlZ], zb);
                        __builtin_amdgcn_s_waitcnt(0);
                        st_agent(&ctl[kCtlPhase], 1u);
                    });
                } else {
                    if (nmine == 0 || !wait_ge(&ctl[kCtlPhase], 1u, 1 << 12, L)) return -1;
                    once([&] { L.res[1] = (int64_t)ld_agent((uint64_t*)&ctl[kCtlZ]); });
                    lds_sync();
                    zb = (uint64_t)readlane_i64(L.res[1], 0);
                }
                if (zb == 0) return -1;
                z = __longlong_as_double((long long)zb);
                stage = AGAIN;
                next = nmine;
                lds_sync();
            }
        }
        if (stage == AGAIN) {
            while (next > 0 && r < 0) {
                const int q = uni(L.mine[--next]);
                if (take(q)) r = q;
            }
            if (r < 0 && !leader) {
                // The last ranges' helpers stay for the row's answer: the
                // sums reach 1.0 in one of them, if at all.
                if (!(have && divided && uni(L.pm[end(held)]) > z * (1.0 - 1e-6))) return -1;
                if (!wait_ge(&ctl[kCtlPhase], 2u, 1 << 12, L)) return -1;
                once([&] {
                    L.res[1] = (int64_t)ld_agent((uint64_t*)&ctl[kCtlSum]);
                    L.res[2] = (int64_t)ld_agent(&ctl[kCtlReach]) - 1;
                    L.res[3] = (int64_t)ld_agent(&ctl[kCtlAt]);
                });
                lds_sync();
                S1 = readlane_i64(L.res[1], 0);
                at = uni((int)L.res[3]);
                const bool here = uni((int)L.res[2]) == held;
                lds_sync();
                if (!here) return -1;
                r = held;
                stage = REACH;
            } else if (r < 0) {
                stage = REST;
                if (wait_ge(&ctl[kCtlDone2], (uint32_t)nr, kGrace, L)) next = nr;
            }
        }
        if (stage == REST) {
            while (next < nr && r < 0) {
                if (take(next)) r = next;
                ++next;
            }
            if (r < 0) {
                if (!wait_ge(&ctl[kCtlDone2], (uint32_t)nr, kPollCap, L)) return -1;
                compose(items, nr, true, L);
                const int kind = uni((int)L.res[0]);
                S1 = readlane_i64(L.res[1], 0);
                r = uni((int)L.res[2]);
                at = uni((int)L.res[3]);
                lds_sync();
                once([&] {
                    st_agent((uint64_t*)&ctl[kCtlSum], (uint64_t)S1);
                    st_agent(&ctl[kCtlAt], (uint32_t)at);
                    st_agent(&ctl[kCtlReach], kind == 2 && held != r ? (uint32_t)r + 1u : 0u);
                    __builtin_amdgcn_s_waitcnt(0);
                    st_agent(&ctl[kCtlPhase], 2u);
                });
                if (kind == 3) return -1;
                if (kind == 0) return R.K;
                if (kind == 1) return L.pc[begin(r)] + at + 1;
                if (held != r && wait_ge(&ctl[kCtlKeep], 1u, kGrace, L))
                    return (int)from_first(L.misc[7], [&] { return ld_agent(&ctl[kCtlKeep]); });
                stage = REACH;
            }
        }
        const int j0 = begin(r);
        const bool second = stage != CLAIM;
        if (held != r) {
            have = load_range<T>(a, R, j0, end(r), held_n, L);
            held = r;
            divided = false;
        }
        uint64_t* out = items + (int64_t)r * kToppItemWords;
        if (have) {
            if (second && !divided) {
#pragma unroll 2
                for (int j = 0; j < kPer; ++j) L.u.x[t * kPer + j] /= z;
                divided = true;
            }
            if (stage == REACH) {
                const int i = reach_one(held_n, at, S1, L);
                const int keep = i == kNone ? -1 : L.pc[j0] + i + 1;
                if (!leader && keep > 0) once([&] { st_agent(&ctl[kCtlKeep], (uint32_t)keep); });
                return keep;
            }
            emit(R, held_n, second ? L.pm[j0] / z : L.pm[j0], r == 0, second, out, L);
        } else {
            if (stage == REACH) return -1;
            once([&] { st_agent(&out[0], ~(uint64_t)0); });
        }
        // the items are stored; then the range's done count
        __builtin_amdgcn_s_waitcnt(0);   // this wave's stores
        lds_sync();
        once([&] { add_agent(&ctl[second ? kCtlDone2 : kCtlDone1], 1u); });
    }
}

// The k-th row (k modulo their number n) of those the general kernel left to
// this launch; with `exact`, of the top_p = 1 rows among them (less those with
// a min-p: their cut may not need the exact sums, and the row's first
// workgroup goes on alone).  -1: there is none.
__device__ __forceinline__ int pick_row(const KArgs& a, int B, int k, bool exact, int& n, Lds& L) {
    const int t = threadIdx.x;
    n = 0;
    for (int pass = 0; pass < 2; ++pass) {   // counts, then the row
        int base = 0;
        for (int b0 = 0; b0 < B; b0 += kT) {
            bool in = false;
            if (b0 + t < B) {
                const uint32_t state = a.topp_ctl[(int64_t)(b0 + t) * kToppCtl];
                in = exact ? state == TOPP_SELECT && a.params[b0 + t].top_p == 1.0f && !(a.params[b0 + t].min_p > 0.0f)
                           : state != TOPP_NONE;
            }
            int c;
            const int at = base + excl_i(in ? 1 : 0, c, L);
            if (pass == 1 && in && at == k % n) L.misc[0] = b0 + t;
            base += c;
        }
        n = base;
        if (n == 0) return -1;
    }
    lds_sync();
    const int row = uni(L.misc[0]);
    lds_sync();
    return row;
}

// The row's chunk records: claimed one by one, until none is left.
template <typename T>
__device__ __forceinline__ void records(const KArgs& a, const Row& R, const tms_row_params& P, uint32_t* ctl, Lds& L) {
    const int t = threadIdx.x;
    for (;;) {
        const uint32_t c = from_first(L.misc[7], [&] { return add_agent(&ctl[kCtlChunk], 1u); });
        if (c >= (uint32_t)R.S) break;
        record<T>(a, R, P, (int)c, L);
        __builtin_amdgcn_s_waitcnt(0);   // this wave's stores
        lds_sync();
        once([&] { add_agent(&ctl[kCtlChunks], 1u); });
    }
}

// The rows before `row` that the general kernel left to this launch.
__device__ __forceinline__ int rows_before(const KArgs& a, int row, Lds& L) {
    int n = 0;
    for (int b0 = 0; b0 < row; b0 += kT) {
        const int b = b0 + (int)threadIdx.x;
        int c;
        excl_i(b < row && a.topp_ctl[(int64_t)b * kToppCtl] != TOPP_NONE ? 1 : 0, c, L);
        n += c;
    }
    return n;
}

// Workgroup g takes the g-th of the rows, if there are so many; the others
// help: with a row's records, then with a top_p = 1 row's ranges.
//
// A call that left no row waits for one load: `any` and `call` are the first
// arguments, which the hardware puts in registers (the build preloads four
// words).  B = 1, V = 32000: 15.2 us a call, 15.5 with the word's address
// loaded first, 13.7 without this launch; B = 64, V = 128256: 17.8, 18.1 and
// 16.3.  The rest is the launch's: an empty kernel in its place costs the same.
template <typename T>
__global__ __launch_bounds__(kT) void topp_kernel(const uint32_t* any, uint32_t call, int B, KArgs a) {
    __shared__ Lds L;
    const int g = (int)blockIdx.x, t = threadIdx.x;
    // No row was left by this call.  (A captured call's replays share one
    // number: an earlier one's rows then only cost the look at the states.)
    if (*any != call) return;
    int n, ne;
    int row = pick_row(a, B, g, false, n, L);
    if (row < 0) return;
    const bool leader = g < n, shared = n > a.topp_slots;
    if (shared && !leader) return;
    if (t < 64) L.tab[t] = kExpTab[t];
    // state words and parameters were written before this launch
    Row R;
    R.slot = g % n;   // pick_row's row
    if (shared) R.slot = (int)from_first(L.misc[7], [&] { return take_dense_slot(a.topp_locks, a.topp_slots, g); });
    bool whole = R.slot < 0;
    int how = SEL_WHOLE, tok = -1, rank = 0;
    for (int turn = leader ? 1 : 0; turn < 2 && !whole; ++turn) {
        if (!leader && turn == 1) {
            row = pick_row(a, B, g - n, true, ne, L);
            if (row < 0) return;
            R.slot = rows_before(a, row, L);
        }
        const tms_row_params P = a.params[row];
        uint32_t* ctl = a.topp_ctl + (int64_t)row * kToppCtl;
        whole = ctl[kCtlState] == TOPP_WHOLE || !describe(a, row, P, R);
        if (!whole) records<T>(a, R, P, ctl, L);
        if (turn == 0) {
            whole = false;
            continue;
        }
        if (!whole) whole = !wait_ge(&ctl[kCtlChunks], (uint32_t)R.S, kPollCap, L) || !plan(a, R, L);
    }
    const tms_row_params P = a.params[row];
    const bool inf = !whole && R.mx == __builtin_huge_valf();   // v / T overflowed (the reference's maximum is +inf)
    if (!whole && !inf && R.K < R.n) whole = true;
    if (!whole && !inf && leader) {
        how = select<T>(a, P, R, L, tok, rank);
        whole = how == SEL_WHOLE;
        lds_sync();
    }
    if (!whole && !inf && (!leader || how == SEL_EXACT)) {
        const int keep = exact_keep<T>(a, R, leader, L);
        whole = !(keep >= 2 && rank < keep - 1);
        if (leader && !whole) write_row(a, row, tok, keep);
    }
    if (!leader) return;
    if (shared && R.slot >= 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        lds_sync();
        once([&] { __hip_atomic_store(&a.topp_locks[R.slot], 0u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT); });
    }
    once([&] {
        a.topp_ctl[(int64_t)row * kToppCtl + kCtlForm] =
            whole ? TOPP_BY_ROW : inf ? TOPP_NOT_FINITE : how == SEL_EXACT ? TOPP_BY_SUMS : TOPP_BY_BUCKETS;
    });
    if (inf) write_row_error(a, row, TMS_ROW_NONFINITE);
    if (inf || !whole) return;
    lds_sync();
    if (t >= kBlock) return;
    [[clang::always_inline]] dense_inline<T>(a, row, L.u.d);
}

}  // namespace topp
}  // namespace tms

int tms_launch_topp(const tms::KArgs& k0, int dtype, int batch, int cus, hipStream_t stream) {
    // A workgroup for every CU (one is resident on a CU) and for every row.
    // Small chunks while the CUs outnumber them: the records of a row are then
    // formed in one turn.
    tms::KArgs k = k0;
    const int small = (k.V + tms::kHistIdsSmall - 1) / tms::kHistIdsSmall;
    const bool few = batch <= tms::kHistSmallRows && batch * small <= cus && 3 * small <= tms::topp::kMaxSeg;
    k.CE = few ? tms::kHistIdsSmall : tms::kHistIds;
    k.S = (k.V + k.CE - 1) / k.CE;
    const dim3 grid((unsigned)(batch < cus ? cus : batch)), block(tms::topp::kT);
    auto launch = [&](auto* kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, stream, k.topp_any, k.topp_call, batch, k);
    };
    switch (dtype) {
        case TMS_DTYPE_F32: launch(&tms::topp::topp_kernel<float>); break;
        case TMS_DTYPE_F16: launch(&tms::topp::topp_kernel<_Float16>); break;
        default: launch(&tms::topp::topp_kernel<tms::Bf16>); break;
    }
    return hipGetLastError() == hipSuccess ? TMS_OK : TMS_ERR_HIP;
}
