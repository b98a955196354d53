"""GPU parity of the whole-vocabulary kernel (tms_topp.hip): top-p rows with
thousands of significant entries, against the oracle.  Tokens, keep counts and
id lists bit-exact; probabilities within 1e-6 relative (fp32 roundings of the
same fp64 quotients).  The full-row form gives the same answers, so the tests
also look at which form decided each row."""
from __future__ import annotations

import numpy as np
import pytest

from tensormark_amd import workloads
from tests.helpers import params_array
from tests.test_gpu_sample import check, run_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from tensormark_amd import Sampler

    s = Sampler(max_batch=320, max_vocab=262144)
    yield s
    s.close()


LISTS, BUCKETS, SUMS, ROW = 0, 1, 2, 3   # tms_debug_row_forms


def forms(s, B):
    import ctypes

    a = (ctypes.c_int32 * B)()
    assert s.lib.tms_debug_row_forms(s.handle, B, a) == 0
    return list(a)


def _rows(rng, B, V, dtype, std, grid=0.0):
    x = rng.normal(0.0, std, (B, V)).astype(np.float32)
    x[np.arange(B)[:, None], rng.integers(0, V, (B, 6))] += rng.uniform(0, 12, (B, 6)).astype(np.float32)
    if grid:
        x = (np.round(x / grid) * grid).astype(np.float32)
    if dtype == "bf16":
        b = workloads.to_bf16_bits(x)
        return b, workloads.bf16_bits_to_f32(b)
    if dtype == "f16":
        x = x.astype(np.float16)
    return x, x.astype(np.float32)


def _mixed(B, seed):
    p = params_array(B, top_k=0, seed=np.arange(B) + seed)
    p["temperature"] = np.resize([1.0, 0.7, 1.3, 1.0, 0.9, 1.0, 0.8, 1.0], B)
    p["top_p"] = np.resize([1.0, 0.95, 0.999, 0.0, 1.0, 2.0, 0.5, 1.0], B)
    p["min_p"] = np.resize([0.0, 0.0, 0.02, 0.0, 0.001, 0.0, 0.3, 0.0], B)
    return p


# _mixed rows: top_p = 1 (with a min-p that cuts earlier, the fifth)
MIXED_FORMS = [SUMS, BUCKETS, BUCKETS, BUCKETS, BUCKETS, BUCKETS, BUCKETS, SUMS]


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("V", [1300, 16384, 16385, 40963, 151936, 262144])
def test_whole_vocabulary_rows(ctx, orc, dtype, V):
    """Every way a row is decided (a cut, a min-p cut, top_p = 1's exact sums,
    neither), with penalties, a mask and an id list, over one chunk to sixteen,
    aligned and not."""
    rng = np.random.default_rng(V)
    B = 8
    x, wide = _rows(rng, B, V, dtype, 1.5)
    p = _mixed(B, V)
    recent = mask = None
    if V != 151936:   # (that one without a window: the packed stream)
        p["repeat_penalty"], p["repeat_last_n"], p["frequency_penalty"] = 1.1, 100, 0.1
        recent = rng.integers(0, V, (B, 120))
        mask = workloads.mask_dense(rng, B, V, 0.8)
    got = run_gpu(ctx, x, p, recent=recent, mask=mask, topk_cap=20, dtype=dtype)
    want = orc.sample_batch(wide, p, recent=recent, mask=mask, topk_cap=20)
    check(got, want, topk_cap=20)
    assert forms(ctx, B) == MIXED_FORMS


@pytest.mark.parametrize("grid", [0.125, 1.0, 64.0])
def test_ties(ctx, orc, grid):
    """Hundreds to all of a row's entries on one value: a cut or a draw inside
    a run of equal logits, and rows whose buckets hold too many keys (the
    full-row form)."""
    B, V = 8, 50000
    rng = np.random.default_rng(int(grid * 8))
    x, wide = _rows(rng, B, V, "bf16", 1.5, grid)
    p = _mixed(B, 5)
    check(run_gpu(ctx, x, p, topk_cap=3, dtype="bf16"), orc.sample_batch(wide, p, topk_cap=3), topk_cap=3)
    f = forms(ctx, B)
    assert f == MIXED_FORMS if grid < 1 else f == [ROW] * B if grid > 1 else ROW in f and BUCKETS in f, f


def test_draws_at_the_ends(ctx, orc):
    """Uniforms at 0, next to 1 and in between, so that the drawn entry is the
    first, the last kept and far down the row."""
    B, V = 12, 30011
    rng = np.random.default_rng(3)
    x, wide = _rows(rng, B, V, "f32", 2.0)
    p = params_array(B, temperature=1.0, top_k=0, seed=1)
    p["top_p"] = np.resize([1.0, 0.9], B)
    hi = np.resize(np.repeat([0, 0xFFFFFFFF, 0xFFFFFF00, 0x80000000, 0xF0000000, 1], 2), B)
    draws = np.stack([np.full(B, 0xFFFFFFFF), hi], axis=1).astype(np.uint32)
    check(run_gpu(ctx, x, p, draws=draws), orc.sample_batch(wide, p, draws=draws))
    f = forms(ctx, B)
    assert f[1::2] == [BUCKETS] * 6 and f[2] == ROW and f[0] == SUMS and f[4::2] == [SUMS] * 4, f


def test_more_rows_than_cus(ctx, orc):
    """300 rows: no workgroups are left to help, each row's own takes every
    range."""
    B, V = 300, 6000
    rng = np.random.default_rng(9)
    x, wide = _rows(rng, B, V, "f16", 1.0)
    p = _mixed(B, 11)
    check(run_gpu(ctx, x, p, dtype="f16"), orc.sample_batch(wide, p))
    assert forms(ctx, B) == list(np.resize(MIXED_FORMS, B))


def test_calls_in_a_row_and_a_captured_graph(ctx):
    """The row states and shared words of one call do not reach the next, and
    a captured call replays to the eager result."""
    import torch

    B, V = 6, 70000
    rng = np.random.default_rng(21)
    x = torch.from_numpy(_rows(rng, B, V, "f32", 2.0)[0]).to("cuda:0")
    p = ctx.params_tensor(_mixed(B, 2))
    want = {k: v.clone() for k, v in ctx.sample(x, p).items()}
    out = {k: torch.zeros_like(v) for k, v in want.items()}
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ctx.sample(x, p, out=out)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            ctx.sample(x, p, out=out)
    torch.cuda.synchronize()
    for _ in range(4):
        for v in out.values():
            v.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(out[k], want[k]) for k in want)
        again = ctx.sample(x.flip(0).contiguous(), p)   # the program's own work between replays
        torch.cuda.synchronize()
        assert int(again["status"].abs().sum()) == 0


@pytest.mark.parametrize("high", [0, 1, 2000])
def test_more_penalised_ids_than_a_record_holds(ctx, orc, high):
    """3000 of the first chunk's ids in the window, the only ones allowed there:
    a record holds 1024 of them, in any order.  None, one or most of them are
    among the row's likely ids."""
    B, V = 16, 20000
    rng = np.random.default_rng(high)
    x = rng.normal(0.0, 0.5, (B, V)).astype(np.float32)
    x[:, :8192] = -200.0
    recent = np.stack([rng.choice(8192, 3000, replace=False) for _ in range(B)])
    for b in range(B):
        x[b, rng.choice(recent[b], high, replace=False)] = 10.0 if high == 1 else 1.0
    allowed = np.ones((B, (V + 31) // 32 * 32), bool)
    allowed[:, V:] = False
    allowed[:, :8192] = False
    allowed[np.arange(B)[:, None], recent] = True
    mask = np.packbits(allowed, axis=1, bitorder="little").view(np.uint32)
    p = params_array(B, top_k=0, temperature=1.0, top_p=0.9, repeat_penalty=1.1, repeat_last_n=4000, seed=np.arange(B))
    check(run_gpu(ctx, x, p, recent=recent, mask=mask), orc.sample_batch(x, p, recent=recent, mask=mask))
    assert forms(ctx, B) == [ROW] * B


@pytest.mark.parametrize("dense", [20, 270])
def test_slots_of_a_large_batch(ctx, orc, dense):
    """A batch of more rows than slots: the rows left to the kernel have a slot
    each, with helpers, or share them."""
    B, V = 320, 9001
    rng = np.random.default_rng(dense)
    x, wide = _rows(rng, B, V, "bf16", 1.5)
    p = _mixed(B, 3)
    p["greedy"] = 1
    p["greedy"][rng.choice(B, dense, replace=False)] = 0
    want = orc.sample_batch(wide, p)
    for _ in range(2):   # (the second on the locks that the first left)
        check(run_gpu(ctx, x, p, dtype="bf16"), want)
        assert forms(ctx, B) == list(np.where(p["greedy"], LISTS, np.resize(MIXED_FORMS, B)))


def test_workspace_of_large_contexts():
    """Records are for 256 rows and 262144 ids at most: past them a row and an
    id cost what the other regions take."""
    from tensormark_amd import Sampler

    def size(B, V):
        s = Sampler(max_batch=B, max_vocab=V)
        try:
            return s.lib.tms_workspace_bytes(s.handle)
        finally:
            s.close()

    row = (size(512, 32000) - size(256, 32000)) / 256      # lists, statistics, history lists
    assert row < 128 * 1024, row
    ids = (size(64, 524288) - size(64, 262144)) / 64 / 262144
    assert ids < 17.0, ids                                   # the whole-row region's 16 bytes an id


def test_history_rows(ctx, orc):
    """The history pre-pass's values as a row's penalised entries: the n-gram
    ban and DRY on rows without a top-k."""
    import torch

    from tensormark_amd import make_history
    from tests.test_gpu_history import _repeating

    B, V = 8, 60011
    rng = np.random.default_rng(12)
    x, wide = _rows(rng, B, V, "f32", 1.5)
    recent = _repeating(rng, B, 700, 60).astype(np.int32)
    for b in range(B):
        x[b, np.unique(recent[b])] += 4.0
    p = _mixed(B, 4)
    p["repeat_penalty"], p["repeat_last_n"], p["presence_penalty"] = 1.1, 500, 0.2
    h = make_history(B, no_repeat_ngram=3, dry_multiplier=0.8, dry_penalty_last_n=600)
    out = ctx.sample(torch.from_numpy(x).to("cuda:0"), p, recent=torch.from_numpy(recent).to("cuda:0"), history=h,
                     topk_cap=20)
    torch.cuda.synchronize()
    assert forms(ctx, B) == MIXED_FORMS
    want = orc.sample_batch(x, p, recent=recent, history=h, topk_cap=20)
    check({k: v.cpu().numpy() for k, v in out.items()}, want, topk_cap=20)


@pytest.mark.parametrize("window,form", [(32767, BUCKETS), (32768, ROW)])
def test_window_counts(ctx, orc, window, form):
    """Windows up to the 15-bit counts of a record, and one id past them; one id
    in every position of a row's."""
    B, V = 3, 30000
    rng = np.random.default_rng(window)
    x, wide = _rows(rng, B, V, "f32", 1.0)
    recent = rng.integers(0, 900, (B, 33000))
    recent[0] = 5
    x[0, 5] = 1.0
    p = params_array(B, top_k=0, temperature=1.0, top_p=0.9, repeat_penalty=1.0001, repeat_last_n=window,
                     seed=np.arange(B))
    check(run_gpu(ctx, x, p, recent=recent), orc.sample_batch(x, p, recent=recent))
    assert forms(ctx, B) == [form] * B


def _peaked(rng, B, V, n):
    x = np.full((B, V), -100.0, np.float32)
    for b in range(B):
        x[b, rng.choice(V, n, replace=False)] = rng.normal(0.0, 1.0, n)
    return x


def test_whole_rows_beside_dense_ones(ctx, orc):
    """Rows that the general kernel leaves for an id list longer than its own
    lists, which go to the full-row form at once, between rows whose records and
    ranges the other workgroups help with."""
    B, V = 8, 70000
    rng = np.random.default_rng(31)
    x, _ = _rows(rng, B, V, "f32", 2.0)
    x[1::2] = _peaked(rng, 4, V, 600)
    p = params_array(B, temperature=1.0, top_k=0, seed=np.arange(B))
    p["top_p"] = np.resize([1.0, 0.9, 0.95, 1.0], B)
    check(run_gpu(ctx, x, p, topk_cap=1100), orc.sample_batch(x, p, topk_cap=1100), topk_cap=1100)
    assert forms(ctx, B) == [SUMS, ROW, BUCKETS, ROW] * 2


def test_replays_with_and_without_rows_left(ctx):
    """A captured call whose logits change: replays that leave rows to the
    second launch, none, and other rows."""
    import torch

    B, V = 6, 50000
    rng = np.random.default_rng(8)
    dense = _rows(rng, B, V, "f32", 2.0)[0]
    peaked = _peaked(rng, B, V, 300)
    half = np.where(np.arange(B)[:, None] % 2, dense, peaked)
    p = ctx.params_tensor(_mixed(B, 6))
    sets = []
    for x in (dense, peaked, half):
        x = torch.from_numpy(x).to("cuda:0")
        sets.append((x, {k: v.clone() for k, v in ctx.sample(x, p).items()}, forms(ctx, B)))
    assert sets[1][2] == [LISTS] * B and LISTS not in sets[0][2]
    x = sets[0][0].clone()
    out = {k: torch.zeros_like(v) for k, v in sets[0][1].items()}
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ctx.sample(x, p, out=out)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            ctx.sample(x, p, out=out)
    torch.cuda.synchronize()
    for i in (0, 1, 2, 1, 1, 2, 0, 1, 0):
        x.copy_(sets[i][0])
        for v in out.values():
            v.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(out[k], sets[i][1][k]) for k in out), i
        assert forms(ctx, B) == sets[i][2], i
        ctx.sample(sets[(i + 1) % 3][0], p)   # the program's own work between replays
