"""GPU parity of the history pre-pass (tms_sample_args.history): the n-gram
ban and DRY after the penalties, on the device, against the oracle's
composition of the reference's steps (tmo_sample_batch_h: mask, repetition
penalty, frequency/presence, apply_no_repeat_ngram, apply_dry, sample).
Tokens, keep counts and top-k ids bit-exact; top-k probabilities within
1e-6 relative.

DRY's scale base^k comes from the caller's table of the reference's powf
values (Sampler.sample builds it with tms_dry_scale_table); without a table
the device uses its own correctly rounded power, which is one ulp off glibc's
powf at (1.75, 83), (1.1, 56) and (1.1, 294) among the pairs sampled
(test_history.py).  test_dry_scale_table_decides_ties pins both forms at
exactly those pairs."""
from __future__ import annotations

import numpy as np
import pytest

from tensormark_amd import make_history, workloads
from tests.helpers import params_array
from tests.test_gpu_sample import check

pytestmark = pytest.mark.gpu


def _run(sampler, x, p, *, recent, n_recent=None, mask=None, history=None, breaker=None,
         topk_cap=0, dtype="f32", noalloc=False, dry_scale=None):
    import torch

    if dtype == "f32":
        t = torch.from_numpy(np.ascontiguousarray(x, np.float32)).to("cuda:0")
    elif dtype == "f16":
        t = torch.from_numpy(np.ascontiguousarray(x, np.float16)).to("cuda:0")
    else:
        t = torch.from_numpy(np.ascontiguousarray(x)).view(torch.bfloat16).to("cuda:0")
    dev = lambda a, dt: None if a is None else torch.from_numpy(np.ascontiguousarray(a, dt)).to("cuda:0")
    out = sampler.sample(t, p, recent=dev(recent, np.int32), n_recent=dev(n_recent, np.int32),
                         mask=None if mask is None else dev(mask.astype(np.uint32).view(np.int32), np.int32),
                         topk_cap=topk_cap, history=history, dry_breaker=dev(breaker, np.uint8),
                         noalloc=noalloc, dry_scale=dry_scale)
    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in out.items()}


def _repeating(rng, B, n, alpha, flip=0.03):
    """Histories that loop: a short period over a small alphabet, a few
    random flips, drawn from ids spread over the vocabulary."""
    h = np.zeros((B, n), np.int32)
    for b in range(B):
        ids = rng.choice(50000, size=alpha, replace=False)
        period = int(rng.integers(2, 9))
        pat = ids[rng.integers(0, alpha, period)]
        row = np.resize(pat, n)
        f = rng.random(n) < flip
        row[f] = ids[rng.integers(0, alpha, int(f.sum()))]
        h[b] = row
    return h


def _boost(x, recent, V, by=6.0):
    """Lift the logits of each row's history ids so the ban and DRY decide
    the draws (random logits would rarely put them in the top k)."""
    for b in range(x.shape[0]):
        ids = np.unique(recent[b][(recent[b] >= 0) & (recent[b] < V)])
        x[b, ids] += np.float32(by)


def _row_mix(rng, B):
    p = params_array(B, temperature=0.8, top_k=40, top_p=0.95, seed=np.arange(B) + 100)
    kind = np.arange(B) % 4
    p["greedy"] = (kind == 0).astype(np.int32)
    p["top_k"] = np.where(kind == 2, 0, np.where(kind == 3, 200, 40))
    p["top_p"] = rng.choice([0.8, 0.95, 1.0], size=B)
    p["min_p"] = rng.choice([0.0, 0.05], size=B)
    p["repeat_penalty"] = rng.choice([1.0, 1.1, 1.3], size=B)
    p["repeat_last_n"] = rng.choice([16, 64, 256], size=B)
    p["frequency_penalty"] = rng.choice([0.0, 0.2], size=B)
    p["presence_penalty"] = rng.choice([0.0, 0.1], size=B)
    return p


def _hist_mix(rng, B):
    h = make_history(B)
    k = np.arange(B) % 3
    h["no_repeat_ngram"] = np.where(k != 1, rng.choice([2, 3, 4], size=B), 0)
    h["dry_multiplier"] = np.where(k != 0, rng.choice([0.5, 0.8], size=B), 0.0)
    h["dry_base"] = rng.choice([1.5, 2.0], size=B)
    h["dry_allowed_length"] = rng.choice([1, 2, 3], size=B)
    h["dry_penalty_last_n"] = rng.choice([32, 256, 1000], size=B)
    return h


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
def test_history_rows_vs_oracle(sampler, orc, dtype):
    rng = np.random.default_rng({"f32": 1, "f16": 2, "bf16": 3}[dtype])
    B, V, n = 48, 50000, 400
    x = rng.normal(0.0, 2.0, (B, V)).astype(np.float32)
    recent = _repeating(rng, B, n, alpha=12)
    _boost(x, recent, V)
    if dtype == "f16":
        x = x.astype(np.float16)
        x32 = x.astype(np.float32)
    elif dtype == "bf16":
        x = workloads.to_bf16_bits(x)
        x32 = workloads.bf16_bits_to_f32(x)
    else:
        x32 = x
    n_recent = rng.integers(n // 2, n + 1, B).astype(np.int32)
    bits = rng.random((B, ((V + 31) // 32) * 32)) < 0.7
    bits[: B // 2] = True
    mask = workloads.pack_bits(bits)
    p = _row_mix(rng, B)
    h = _hist_mix(rng, B)
    want = orc.sample_batch(x32, p, recent=recent, n_recent=n_recent, mask=mask, topk_cap=20,
                            history=h)
    g = _run(sampler, x, p, recent=recent, n_recent=n_recent, mask=mask, history=h, topk_cap=20,
             dtype=dtype)
    check(g, want, 20)
    # the ban and DRY moved the answer on many rows
    plain = orc.sample_batch(x32, p, recent=recent, n_recent=n_recent, mask=mask, topk_cap=20)
    assert (plain["tokens"] != want["tokens"]).sum() >= B // 8


def test_ngram_restore_rule(sampler, orc):
    """The ban would leave nothing above -inf: the banned ids keep their
    values (tmsample.h:105-112).  Row 0: the grammar allows only the banned
    id; row 1: no mask, every logit -inf but the banned id's (the pre-pass
    scans the row); row 2: one more allowed id far down the row stays, so
    the ban holds and that id is sampled."""
    V = 70000
    rng = np.random.default_rng(9)
    x = rng.normal(0.0, 1.0, (3, V)).astype(np.float32)
    recent = np.array([[5, 6, 7, 5, 6]] * 3, np.int32)   # ngram 3: context (5, 6) -> 7 banned
    bits = np.zeros((3, ((V + 31) // 32) * 32), bool)
    bits[0, 7] = True
    bits[1] = True
    bits[2, 7] = bits[2, 65001] = True
    x[1, :] = -np.inf
    x[1, 7] = 0.5
    mask = workloads.pack_bits(bits)
    p = params_array(3, temperature=1.0, top_k=40, top_p=1.0, seed=np.arange(3))
    h = make_history(3, no_repeat_ngram=3)
    want = orc.sample_batch(x, p, recent=recent, mask=mask, topk_cap=4, history=h)
    assert want["tokens"].tolist() == [7, 7, 65001]
    g = _run(sampler, x, p, recent=recent, mask=mask, history=h, topk_cap=4)
    check(g, want, 4)


def test_dry_breakers_and_out_of_range_ids(sampler, orc):
    rng = np.random.default_rng(11)
    B, V, n = 16, 32000, 300
    x = rng.normal(0.0, 2.0, (B, V)).astype(np.float32)
    recent = _repeating(rng, B, n, alpha=6, flip=0.01) % V
    _boost(x, recent, V)
    recent[:, ::37] = -5          # out of range: skipped by every step
    recent[:, 5::41] = V + 3
    breaker = np.zeros(V, np.uint8)
    breaker[np.unique(recent[recent >= 0][::7] % V)[:4]] = 1
    p = _row_mix(rng, B)
    h = make_history(B, no_repeat_ngram=3, dry_multiplier=0.8, dry_base=1.5, dry_allowed_length=2,
                     dry_penalty_last_n=256)
    want = orc.sample_batch(x, p, recent=recent, topk_cap=8, history=h, dry_breaker=breaker)
    g = _run(sampler, x, p, recent=recent, history=h, breaker=breaker, topk_cap=8)
    check(g, want, 8)


def test_long_history_lists(sampler, orc):
    """Lists longer than the general kernel's owned window (1024 entries):
    3000 distinct ids in the repetition window, plus bans and DRY targets."""
    rng = np.random.default_rng(13)
    B, V, n = 8, 128256, 3600
    x = rng.normal(0.0, 2.0, (B, V)).astype(np.float32)
    recent = np.zeros((B, n), np.int32)
    for b in range(B):
        recent[b, :3000] = rng.choice(V, 3000, replace=False)
        recent[b, 3000:] = np.resize(recent[b, 100:140], 600)   # a loop at the end
    _boost(x, recent[:, 3000:], V)
    p = _row_mix(rng, B)
    p["repeat_last_n"] = 3600
    p["repeat_penalty"] = 1.2
    h = make_history(B, no_repeat_ngram=4, dry_multiplier=0.8, dry_base=2.0, dry_penalty_last_n=700)
    want = orc.sample_batch(x, p, recent=recent, topk_cap=16, history=h)
    g = _run(sampler, x, p, recent=recent, history=h, topk_cap=16)
    check(g, want, 16)


def test_history_list_overflow_reports_unsupported(sampler, orc):
    """A row whose history touches more than TMS_HISTORY_MAX_IDS (4096)
    distinct ids reports TMS_ROW_UNSUPPORTED; the other rows are sampled."""
    rng = np.random.default_rng(17)
    B, V, n = 4, 60000, 5000
    x = rng.normal(0.0, 2.0, (B, V)).astype(np.float32)
    recent = np.tile(rng.integers(0, 50, n).astype(np.int32), (B, 1))
    recent[1] = rng.choice(V, n, replace=False)
    p = _row_mix(rng, B)
    p["repeat_last_n"] = n
    p["repeat_penalty"] = 1.1
    h = make_history(B, no_repeat_ngram=3)
    want = orc.sample_batch(x, p, recent=recent, history=h)
    g = _run(sampler, x, p, recent=recent, history=h)
    assert g["status"][1] == 4 and g["tokens"][1] == -1
    check(g, want, 0, rows=[0, 2, 3])


def test_history_noalloc_matches_context(sampler, orc):
    rng = np.random.default_rng(19)
    B, V, n = 32, 40000, 256
    x = rng.normal(0.0, 2.0, (B, V)).astype(np.float32)
    recent = _repeating(rng, B, n, alpha=10)
    _boost(x, recent, V)
    p = _row_mix(rng, B)
    h = _hist_mix(rng, B)
    a = _run(sampler, x, p, recent=recent, history=h, topk_cap=10)
    b = _run(sampler, x, p, recent=recent, history=h, topk_cap=10, noalloc=True)
    for k in a:
        assert np.array_equal(a[k], b[k]), k
    want = orc.sample_batch(x, p, recent=recent, topk_cap=10, history=h)
    check(a, want, 10)


def test_history_without_ngram_or_dry_equals_plain(sampler, orc):
    """History params that switch both steps off leave the answers of the
    plain call (the pre-pass still forms the repetition-penalty values)."""
    w = workloads.cfg2(B=16, V=40000, seed=23)
    h = make_history(16)
    a = _run(sampler, w["logits"], w["params"], recent=w["recent"], history=h, topk_cap=40)
    want = orc.sample_batch(w["logits"], w["params"], recent=w["recent"], topk_cap=40)
    check(a, want, 40)


def _ties_at(pairs, allowed=2):
    """Two greedy rows per (base, k): the history `1 t 2 t` (t = k + allowed
    distinct ids) gives id 2 exactly one DRY hit of length k + allowed, so
    its logit 0 becomes -(2^-60 * s), s = powf(base, k) as the reference
    computes it; a twin id holds exactly that value, below id 2 (id 0) in
    one row and above it (id 400) in the other.  Equal values go to the
    lower id, so the reference answers 0 and then 2, and a scale one ulp
    off either way changes one of the two answers."""
    from tensormark_amd.sampler import dry_scale_table

    V = 512
    B = 2 * len(pairs)
    n = max(2 * (k + allowed) + 2 for _, k in pairs)
    x = np.full((B, V), -1e30, np.float32)
    recent = np.zeros((B, n), np.int32)
    n_recent = np.zeros(B, np.int32)
    h = make_history(B, dry_multiplier=2.0 ** -60, dry_allowed_length=allowed, dry_penalty_last_n=n)
    for i, (base, k) in enumerate(pairs):
        L = k + allowed
        t = np.arange(10, 10 + L, dtype=np.int32)
        hist = np.concatenate([[1], t, [2], t]).astype(np.int32)
        s = dry_scale_table(make_history(1, dry_multiplier=1.0, dry_base=base, dry_penalty_last_n=k + 1))[0][k]
        v = np.float32(0.0) - np.float32(2.0 ** -60) * s
        for j, twin in ((2 * i, 0), (2 * i + 1, 400)):
            recent[j, : hist.size] = hist
            n_recent[j] = hist.size
            h["dry_base"][j] = base
            x[j, 2] = 0.0
            x[j, twin] = v
    p = params_array(B, temperature=1.0, top_k=40, top_p=1.0, seed=np.arange(B))
    p["greedy"] = 1
    return x, p, recent, n_recent, h


# where glibc's powf and the correctly rounded power differ, and pairs where they agree
POWF_DIFFER = [(1.75, 83), (1.1, 56), (1.1, 294)]
POWF_AGREE = [(1.75, 82), (1.5, 40), (2.0, 100)]


def test_dry_scale_table_decides_ties(sampler, orc):
    """With the table the device reproduces the reference's scale bit for
    bit (the oracle applies the reference's powf): every twin row answers as
    the oracle does, 0 then 2."""
    x, p, recent, n_recent, h = _ties_at(POWF_DIFFER + POWF_AGREE)
    want = orc.sample_batch(x, p, recent=recent, n_recent=n_recent, history=h)
    assert list(want["tokens"]) == [0, 2] * (len(want["tokens"]) // 2)
    g = _run(sampler, x, p, recent=recent, n_recent=n_recent, history=h)
    check(g, want)


def test_dry_without_table_is_the_correctly_rounded_power(sampler):
    """Without a table the device's own power is the correctly rounded one:
    at the pairs where glibc's powf is one ulp off, one twin row of each pair
    changes its answer in the direction the exact power gives; where they
    agree both rows keep the reference's answers."""
    from fractions import Fraction

    from tests.test_history import _round_f32

    pairs = POWF_DIFFER + POWF_AGREE
    x, p, recent, n_recent, h = _ties_at(pairs)
    g = _run(sampler, x, p, recent=recent, n_recent=n_recent, history=h, dry_scale=False)
    assert (g["status"] == 0).all()
    for i, (base, k) in enumerate(pairs):
        cr = _round_f32(Fraction(float(np.float32(base))) ** k)
        ref = x[2 * i, 0] / np.float32(-(2.0 ** -60))   # the table's value
        if cr > ref:     # a larger penalty: id 2 falls below its twins
            want = [0, 400]
        elif cr < ref:   # smaller: id 2 rises above them
            want = [2, 2]
        else:
            want = [0, 2]
        assert list(g["tokens"][2 * i: 2 * i + 2]) == want, (base, k, cr, ref)


def test_dry_long_repetitive_windows(sampler, orc):
    """Windows of TMS_DRY_MAX_WINDOW ids that repeat one id, or a period of 2
    or 5: every position matches far back, so the pre-pass takes its linear
    Z-function pass; the rows match the oracle, and one call stays well
    under a second.  A DRY window longer than the bound reports
    TMS_ROW_UNSUPPORTED."""
    import time

    import torch

    from tensormark_amd.sampler import DRY_MAX_WINDOW

    rng = np.random.default_rng(41)
    B, V, n = 4, 30000, DRY_MAX_WINDOW
    x = rng.normal(0.0, 2.0, (B, V)).astype(np.float32)
    recent = np.zeros((B, n + 10), np.int32)
    recent[0, :n] = 7
    recent[1, :n] = np.resize([11, 12], n)
    recent[2, :n] = np.resize([20, 21, 22, 23, 24], n)
    recent[3] = 5
    n_recent = np.array([n, n, n, n + 10], np.int32)
    x[:, :30] += 9.0
    p = params_array(B, temperature=0.9, top_k=40, top_p=0.95, seed=np.arange(B) + 3)
    h = make_history(B, dry_multiplier=0.01, dry_base=1.001, dry_allowed_length=2,
                     dry_penalty_last_n=n + 10)
    want = orc.sample_batch(x, p, recent=recent, n_recent=n_recent, history=h, topk_cap=8)
    _run(sampler, x, p, recent=recent, n_recent=n_recent, history=h, topk_cap=8)   # warm
    t0 = time.perf_counter()
    g = _run(sampler, x, p, recent=recent, n_recent=n_recent, history=h, topk_cap=8)
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    assert dt < 1.0, dt
    assert g["status"][3] == 4 and g["tokens"][3] == -1
    check(g, want, 8, rows=[0, 1, 2])


@pytest.mark.parametrize("n,last_n", [(1, 1), (3, 3), (1023, 1023), (1025, 1025), (4096, 4096),
                                      (4097, 4096), (4097, 4097), (6001, 300), (8200, 8192)])
def test_history_window_edges(sampler, orc, n, last_n):
    """Histories and DRY windows around one pass of the workgroup and around
    the ids it holds in LDS: older ids are read where they are needed, and a
    DRY window of more of them is staged elsewhere."""
    rng = np.random.default_rng(n + last_n)
    B, V = 4, 50000
    recent = _repeating(rng, B, n, 12, flip=0.2)
    recent[:, rng.integers(0, n)] = [-1, V, 3, 4]
    x = rng.normal(0.0, 2.0, (B, V)).astype(np.float32)
    _boost(x, recent, V)
    breaker = np.zeros(V, np.uint8)
    breaker[recent[2, 0]] = 1
    p = params_array(B, temperature=0.9, top_k=40, top_p=0.95, seed=np.arange(B) + 17)
    p["repeat_penalty"] = 1.1
    p["repeat_last_n"] = [n, 5000, 64, 4097]
    h = make_history(B, no_repeat_ngram=3, dry_multiplier=0.3, dry_base=1.01,
                     dry_penalty_last_n=last_n)
    want = orc.sample_batch(x, p, recent=recent, history=h, dry_breaker=breaker, topk_cap=8)
    g = _run(sampler, x, p, recent=recent, history=h, breaker=breaker, topk_cap=8)
    check(g, want, 8)


@pytest.mark.parametrize("n,match", [(33, 8), (33, 16), (1024, 56), (4096, 8), (4097, 64), (8192, 1), (8192, 7),
                                     (8192, 8), (8192, 56), (8192, 63), (8192, 64), (8192, 72)])
def test_dry_match_reaches_the_windows_start(sampler, orc, n, match):
    """The window begins with the `match` ids that it ends with: their
    comparison, eight positions a round, ends at the window's start."""
    V = 20000
    rng = np.random.default_rng(n + match)
    recent = np.stack([rng.choice(V, n, replace=False) for _ in range(4)])
    recent[:, :match] = recent[:, n - match:]
    x = rng.normal(0, 1, (4, V)).astype(np.float32)
    x[np.arange(4), recent[:, match]] += 30.0
    p = params_array(4, temperature=0.8, top_k=40, top_p=0.95, seed=np.arange(4))
    h = make_history(4, dry_multiplier=0.5, dry_base=1.1, dry_allowed_length=1, dry_penalty_last_n=n)
    breaker = np.zeros(V, np.uint8)
    got = _run(sampler, x, p, recent=recent, history=h, breaker=breaker, topk_cap=5)
    check(got, orc.sample_batch(x, p, recent=recent, history=h, dry_breaker=breaker, topk_cap=5), 5)


@pytest.mark.parametrize("n", [7, 8, 11, 12, 300, 1500])
@pytest.mark.parametrize("pre_pass", [False, True])
def test_long_repetition_chains(sampler, orc, n, pre_pass):
    """An id that occurs n times is divided n times, each quotient rounded:
    around the count from which products stand in for the divisions, and
    through the end of the normal range (2.0 / 1.1^1500 is subnormal), with
    and without the history pre-pass."""
    rng = np.random.default_rng(n)
    B, V = 6, 20000
    x = rng.normal(0.0, 1.0, (B, V)).astype(np.float32)
    x[:, 5] = [1e30, 7.3, 2.0, -0.7, 1e-37, 0.0]
    x[:, 6] = [8.0, 1.9, 0.3, 0.2, 2.0, 2.0]
    recent = np.full((B, n + 3), 5, np.int32)
    recent[:, ::7] = rng.integers(0, V, recent[:, ::7].shape)
    p = params_array(B, temperature=0.8, top_k=20, top_p=0.95, seed=np.arange(B) + 5)
    p["repeat_penalty"] = [1.3, 1.01, 1.1, 1.001, 1.1, 2.0]
    p["repeat_last_n"] = n + 3
    h = make_history(B, no_repeat_ngram=4) if pre_pass else None
    want = orc.sample_batch(x, p, recent=recent, history=h, topk_cap=20)
    g = _run(sampler, x, p, recent=recent, history=h, topk_cap=20)
    check(g, want, 20)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("V", [3, 7, 8, 9, 4099, 16385, 32771, 65549])
def test_ragged_rows_with_windows(sampler, orc, dtype, V):
    """Rows at any element's address and a last vector of 1 to 7 ids, whose
    maximum is the row's last id: top-k rows with a window and a mask."""
    rng = np.random.default_rng(V)
    B = 3
    x = rng.normal(0.0, 2.0, (B, V)).astype(np.float32)
    x[:, V - 1] = [20.0, 12.0, 9.0]
    x[:, V - 2] = [3.0, 12.0, 9.5]
    if dtype == "bf16":
        gx = workloads.to_bf16_bits(x)
        x = workloads.bf16_bits_to_f32(gx)
    else:
        gx = x
        x = x.astype(np.float16).astype(np.float32) if dtype == "f16" else x
    recent = rng.integers(0, V, (B, 64)).astype(np.int32)
    recent[1] = V - 1
    mask = np.full((B, (V + 31) // 32), 0xFFFFFFFF, np.uint32)
    mask[2, (V - 1) >> 5] &= ~np.uint32(1 << ((V - 1) & 31))
    p = params_array(B, temperature=0.9, top_k=20, top_p=0.95, seed=np.arange(B) + 7)
    p["repeat_penalty"] = 1.1
    p["greedy"] = [1, 0, 0]
    want = orc.sample_batch(x, p, recent=recent, mask=mask, topk_cap=8)
    g = _run(sampler, gx, p, recent=recent, mask=mask, topk_cap=8, dtype=dtype)
    check(g, want, 8)
