// tms_spec_plan.h -- how a verify call is cut into workgroups (host
// arithmetic only: tms_spec.hip launches it, tests/test_spec_plan.py compiles
// it by itself).
#ifndef TMS_SPEC_PLAN_H
#define TMS_SPEC_PLAN_H

#include <stddef.h>

#include <algorithm>

namespace tms {
constexpr int kSpecMaxK = 16;        // draft tokens per sequence
constexpr int kSpecParts = 64;       // vocabulary parts of the residual draw
constexpr int kSpecPartIds = 32768;  // ids of a statistics part, where the rows fill the chip
constexpr int kSpecFill = 1024;      // most statistics parts of a call with fewer rows than that
constexpr int kSpecClaims = 8;       // claim counters of a verify launch
constexpr int kSpecShare = 4;        // contexts that may verify at once
constexpr int kRowT = 1024;          // threads of the row kernel
constexpr int kSpecBlock = 256;      // threads of the resolve
constexpr int kRunMax = 16;          // most ids of a thread in the waiting resolve

// Words of spec_rparts: two for each part of each row of the largest call.
constexpr size_t spec_rpart_words(size_t max_batch, int max_vocab) {
    return 2 * (max_batch * (2 * kSpecMaxK + 1) * (((size_t)max_vocab + kSpecPartIds - 1) / kSpecPartIds) + kSpecFill);
}

struct SpecPlan {
    // the resolve: P parts of Lp ids a sequence
    int P, Lp, n2;
    bool wait, claim_parts;
    // the statistics: S parts of pv vectors a row, ns vectors a thread
    int S, pv, ns, n1;
    bool lazy, claim_rows;
};

// B sequences of k drafts over V ids, vec ids to a 16-byte vector; cap1 and
// cap2 workgroups of the row kernel and of the waiting resolve are resident at
// once.
inline SpecPlan spec_plan(int B, int k, int V, int vec, int cap1, int cap2) {
    SpecPlan s{};
    const int nsmax = kSpecPartIds / vec / kRowT;
    const int R = 2 * k + 1;
    const int nv = (V + vec - 1) / vec;
    // The resolve: the waiting form for up to kSpecParts parts of kRunMax ids
    // a thread, in parts of half that length where its grid is resident at
    // once (B = 1, V = 128256: 10 us).  B = 32, V = 151936 bf16: 27 us, where
    // the ticket form, which reads the threshold's part again, takes 35.
    const int most = kSpecBlock * kRunMax;
    s.Lp = most / 2;
    s.P = (V + s.Lp - 1) / s.Lp;
    if (s.P > kSpecParts || B * s.P > cap2) {
        s.Lp = most;
        s.P = (V + s.Lp - 1) / s.Lp;
    }
    s.wait = s.P <= kSpecParts && s.P <= cap2 / kSpecClaims;
    if (!s.wait) {
        s.P = std::min((V + 2047) / 2048, kSpecParts);
        s.Lp = ((V + s.P - 1) / s.P + 7) / 8 * 8;
        s.P = (V + s.Lp - 1) / s.Lp;
    }
    s.n2 = (B + kSpecClaims - 1) / kSpecClaims * kSpecClaims * s.P;
    s.claim_parts = s.wait && s.n2 > cap2;   // (an XCD holds the sequences of one residue)
    // The statistics: as few parts a row as registers allow, more where the
    // rows would leave compute units idle.  Where the grid takes more than
    // one round of the chip, the waiting resolve takes the bonus rows'
    // statistics itself: 2k rows a sequence in place of 2k + 1, for an
    // exchange more (B = 32, k = 8, V = 32000 fp32: 512 rows, one round of
    // two workgroups a CU, in place of 544).
    s.S = (nv + nsmax * kRowT - 1) / (nsmax * kRowT);
    // A row's parts wait for each other and have one residue of kSpecClaims,
    // hence one XCD: at most a kSpecShare-th of its places each, so that as
    // many contexts (the hardware queues of a process) may verify at once
    // and none waits for a place that another's waiting parts hold.  (Past
    // 524288 ids the registers ask for more parts, 32 of 64 places at most.)
    const int room = std::max(1, cap1 / kSpecClaims / kSpecShare);
    const int fill = std::min(std::min(cap1 / 2, kSpecFill) / (B * R), room);
    s.S = std::max(s.S, std::min(fill, (nv + kRowT - 1) / kRowT));
    s.pv = (nv + s.S - 1) / s.S;
    s.S = (nv + s.pv - 1) / s.pv;
    s.ns = s.pv <= kRowT ? 1 : s.pv <= nsmax / 2 * kRowT ? nsmax / 2 : nsmax;
    s.lazy = s.wait && B * R * s.S > cap1;
    const int rows = B * (s.lazy ? R - 1 : R);
    s.n1 = s.S == 1 ? rows : (rows + kSpecClaims - 1) / kSpecClaims * kSpecClaims * s.S;
    s.claim_rows = s.n1 > cap1;
    return s;
}
}  // namespace tms

#endif  // TMS_SPEC_PLAN_H
