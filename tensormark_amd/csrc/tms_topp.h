// tms_topp.h -- the workspace that the general kernel (tms_sample.hip), which
// marks the dense top-p rows of a call, and the whole-vocabulary kernel
// (tms_topp.hip), which samples them, share.
#pragma once

#include "tms_sample_common.h"

namespace tms {

// A record describes one chunk of a row over buckets of lg = penalised value
// / T, 1/25 wide: each bucket's softmax mass, the number of entries above it,
// and the chunk's ids in bucket order (a counting sort), so that any interval
// of buckets is one run of ids a chunk.
//
// Buckets run from the one holding the chunk's maximum downwards: 1023 x 1/25
// spans 40.9, more than kSigSpan, so every entry that can change a sum has
// one.  The fullest bucket of a normal row holds about 0.016 V / d entries, d the
// standard deviation of lg: 1,640 of 256,000 at d = 2.5.  So a cut and a draw
// are settled by ordering a few thousand keys (kSel at most) where a row is not
// flat.  Rows that took the full-row form, of 64 normal rows at top_p 0.9, 0.95
// and 0.98: V = 256000 none or one at d >= 2.5, 3 to 5 at 2.0, 12 to 16 at 1.67,
// 31 to 44 at 1.25; V = 128256 none at 1.67, up to 8 at 1.25, 4 to 11 at 1.0; V =
// 32000 none at 0.5.  With top_p = 1 (kRange): V = 256000 none at 1.25, two at
// 1.0; V = 128256 none at 0.75, seven at 0.5.
constexpr int kHistBuckets = 1024;
constexpr float kHistScale = 25.0f;
constexpr int kHistExtra = 1024;        // penalised entries of a chunk, at most
constexpr int kHistIds = 16384;         // ids of a chunk, at most: 16 a thread
constexpr int kHistIdsSmall = 8192;     // ... where that gives more workgroups work
constexpr int kToppMaxVocab = 262144;
// u64 words of a record: masses, then u32 counts of the entries above bucket
// 0..1023, the penalised entries (value bits << 32 | id), the head (valid << 32
// | bits of the chunk's maximum of lg), and u16 ids in bucket order (below the
// chunk's length: id - its first id; else kHistIds + the index of a penalised
// entry).
constexpr int kHistCnt = kHistBuckets;
constexpr int kHistExt = kHistCnt + kHistBuckets / 2;
constexpr int kHistHead = kHistExt + kHistExtra;
constexpr int kHistId = kHistHead + 2;
static_assert(kHistIds + kHistExtra < 65536, "16-bit ids of a chunk");
constexpr int hist_words(int chunk_ids) { return kHistId + chunk_ids / 4 + 2; }
// Slots of records and items in a workspace, at most: as many as workgroups of
// that kernel run at once, one a CU.  A row of 256,000 ids takes 0.93 MB.
constexpr int kToppSlotsMax = 256;
// Rows in small chunks at most, so that their records fit those of as many
// slots in large ones.
constexpr int kHistSmallRows = 32;
inline size_t topp_hist_words(size_t rows, int vocab) {
    if (vocab > kToppMaxVocab) vocab = kToppMaxVocab;
    const size_t large = rows * (size_t)((vocab + kHistIds - 1) / kHistIds) * hist_words(kHistIds);
    const size_t few = rows < (size_t)kHistSmallRows ? rows : (size_t)kHistSmallRows;
    const size_t small = few * (size_t)((vocab + kHistIdsSmall - 1) / kHistIdsSmall) * hist_words(kHistIdsSmall);
    return (large > small ? large : small) + 32;
}
// Row states the general kernel leaves for the whole-vocabulary kernel.
enum : uint32_t { TOPP_NONE = 0, TOPP_SELECT = 1, TOPP_WHOLE = 2 };
// How that kernel decided a row (word kToppForm of the row's shared words): by
// the buckets of the cut and the draw, by the composed sums of top_p = 1, or
// by the full-row form.
enum : uint32_t { TOPP_BY_BUCKETS = 1, TOPP_BY_SUMS = 2, TOPP_BY_ROW = 3, TOPP_NOT_FINITE = 4 };
constexpr int kToppForm = 18;
// u32 words per row shared by the workgroups of a row (zeroed by the general
// kernel's merger): see tms_topp.hip.
constexpr int kToppCtl = 64;
constexpr int kToppRanges = 64;       // most ranges of a row
constexpr int kToppRawMax = 24;       // raw entries of a range
constexpr int kToppItemWords = 160;   // u64 words of a range's items: count, then 3 an item
static_assert(1 + 3 * (2 * kToppRawMax + 1) <= kToppItemWords, "a range's items");

// The bucket of lg, on a grid common to every chunk: floor(25 lg), clamped so
// that differences of two buckets do not overflow (monotone in lg).
__device__ __forceinline__ int topp_bucket(float lg) {
    const float y = fminf(fmaxf(lg * kHistScale, -5e8f), 5e8f);
    return (int)floorf(y);
}

// e^x for x in [-42, 0] within 2 ulp (exp64 without its special cases).
__device__ __forceinline__ double exp_span(double x, const double* tab) {
    const double kd = rint(x * 0x1.71547652b82fep+6);
    double r = fma(-kd, 0x1.62e42fefa39efp-7, x);
    r = fma(-kd, 0x1.abc9e3b39803fp-62, r);
    double p = 1.0 / 120;
    p = fma(p, r, 1.0 / 24);
    p = fma(p, r, 1.0 / 6);
    p = fma(p, r, 0.5);
    p = fma(p, r, 1.0);
    p = fma(p, r, 1.0);
    const int ki = (int)kd;
    return ldexp(tab[ki & 63] * p, ki >> 6);
}

}  // namespace tms

// Launches the whole-vocabulary kernel over `batch` rows (tms_topp.hip).
int tms_launch_topp(const tms::KArgs& k, int dtype, int batch, int cus, hipStream_t stream);
