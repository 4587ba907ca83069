"""The HIP membership kernel against the oracle: ``ok`` and ``above`` exactly equal to the
batched reference semantics (oracle.member.check_members_ref) and to the per-row FP64
reference; ``mass_above`` within member_eps32 of the FP64 reference.  Covers the reference's
tests/test_member.py batched cases, the LDS fast path and both fallbacks (candidate overflow,
k above 1024), and the BASELINE workload (256 x 151,936 logits, top-k 50, top-p 0.9) with 1% of
tokens replaced by out-of-set tokens that must all be flagged, with no false alarm."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle.member import check_member, check_members_ref
from pck.cuda._lib import PckMemberArgs, lib
from pck.member import check_members, member_eps32

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]


def run(logits, tokens, top_k=None, top_p=None, greedy=None, top_k_host=None, tol=1e-4):  # type: ignore[no-untyped-def]
    t = lambda a, dt=None: None if a is None else torch.as_tensor(a, dtype=dt).cuda()  # noqa: E731
    out = check_members(
        t(logits, torch.float32), t(tokens), t(top_k), t(top_p), t(greedy), tol, top_k_host
    )
    return {k: v.cpu().numpy() for k, v in out.items()}


def assert_matches_oracle(logits, tokens, top_k=None, top_p=None, greedy=None, top_k_host=None) -> None:  # type: ignore[no-untyped-def]
    got = run(logits, tokens, top_k, top_p, greedy, top_k_host)
    want = check_members_ref(logits, tokens, top_k, top_p, greedy, top_k_host=top_k_host)
    np.testing.assert_array_equal(got["ok"], want["ok"])
    np.testing.assert_array_equal(got["above"], want["above"])
    vocab = logits.shape[1]
    if top_p is not None:
        finite = np.isfinite(want["mass_above"])
        assert np.all(np.abs(got["mass_above"][finite] - want["mass_above"][finite]) <= 2 * member_eps32(vocab))


def test_the_batched_check_matches_the_reference() -> None:
    rng = np.random.default_rng(0)
    logits = (rng.standard_normal((64, 500)) * 3).astype(np.float32)
    logits[:, :5] = 7.0
    tokens = rng.integers(0, 500, 64)
    tokens[:32] = np.argsort(-logits[:32], axis=1)[np.arange(32), rng.integers(0, 20, 32)]
    top_k = rng.choice([1, 5, 20, 500], 64)
    top_p = rng.choice([0.3, 0.9, 1.0], 64)
    greedy = rng.random(64) < 0.1
    out = run(logits, tokens, top_k, top_p, greedy)
    for i in range(64):
        k = None if top_k[i] == 500 else int(top_k[i])
        p = None if top_p[i] == 1.0 else float(top_p[i])
        ref = check_member(logits[i], int(tokens[i]), k, p, greedy=bool(greedy[i]))
        assert bool(out["ok"][i]) == ref.ok, i
        assert int(out["above"][i]) == ref.above
        if ref.ok and p is not None and not greedy[i]:
            assert abs(float(out["mass_above"][i]) - ref.mass_above) <= member_eps32(500)
    assert_matches_oracle(logits, tokens, top_k, top_p, greedy)


@pytest.mark.parametrize("host", [False, True])
def test_the_top_k_path_counts_ties_beyond_the_largest_k(host: bool) -> None:
    rng = np.random.default_rng(1)
    rows, vocab = 48, 400
    logits = (rng.standard_normal((rows, vocab)) * 4).astype(np.float32)
    top_k = rng.choice([1, 3, 10, 40], rows)
    for i in range(0, rows, 2):
        order = np.argsort(-logits[i])
        logits[i, order[top_k[i] - 1 : top_k[i] + 29]] = logits[i, order[top_k[i] - 1]]
    tokens = np.array([np.argsort(-row)[rng.integers(0, k)] for row, k in zip(logits, top_k)])
    tokens[::5] = rng.integers(0, vocab, len(tokens[::5]))
    top_p = rng.choice([0.2, 0.6, 0.95], rows)
    out = run(logits, tokens, top_k.astype(np.int32), top_p, top_k_host=top_k if host else None)
    for i in range(rows):
        ref = check_member(logits[i], int(tokens[i]), int(top_k[i]), float(top_p[i]))
        assert bool(out["ok"][i]) == ref.ok, i
        if ref.ok:
            assert abs(float(out["mass_above"][i]) - ref.mass_above) <= member_eps32(vocab)


def test_fp32_terms_stay_within_the_bound_on_wide_logits() -> None:
    rng = np.random.default_rng(2)
    rows, vocab = 16, 5000
    logits = rng.uniform(-300, 40, (rows, vocab)).astype(np.float32)
    logits[:, :50] = rng.uniform(30, 40, (rows, 50)).astype(np.float32)
    tokens = np.argsort(-logits, axis=1)[:, 7]
    out = run(logits, tokens, top_p=np.full(rows, 0.99))
    for i in range(rows):
        ref = check_member(logits[i], int(tokens[i]), top_p=0.99)
        assert abs(float(out["mass_above"][i]) - ref.mass_above) <= member_eps32(vocab)


def test_bad_token_ids_and_a_stale_host_top_k_reject_instead_of_crashing() -> None:
    rng = np.random.default_rng(3)
    logits = rng.standard_normal((4, 50)).astype(np.float32)
    tokens = np.array([-1, 50, 10_000, int(logits[3].argmax())])
    out = run(logits, tokens, np.array([5, 5, 5, 20], dtype=np.int32), np.full(4, 0.9),
              top_k_host=np.array([5, 5, 5, 5]))  # fmt: skip
    assert out["ok"].tolist() == [False, False, False, True]


def test_nan_rows_reject() -> None:
    logits = np.random.default_rng(4).standard_normal((3, 300)).astype(np.float32)
    logits[1, 17] = np.nan
    out = run(logits, np.array([0, 0, 0]), top_p=np.full(3, 0.999999))
    assert not out["ok"][1] and out["ok"][0] == check_member(logits[0], 0, top_p=0.999999).ok


CASES = ["all_equal", "many_ties", "k_above_1024", "keep_all_rows", "mixed", "k_700",
         "k_700_offset", "one_wave_overflows", "wide_window"]  # fmt: skip


@pytest.mark.parametrize("case", CASES)
def test_fallback_paths_match_the_oracle(case: str) -> None:
    """Rows whose candidate set overflows LDS, k_eff above 1024, rows without top-k.  k_700 and
    k_700_offset leave ~1400 candidates (several per lane of each wave's segment, none
    overflowing), spread over four binades or packed into one.  one_wave_overflows puts 512
    equal maxima in the stream slots of one wave only (that wave's segment overflows while the
    row's total fits).  wide_window plants three huge logits per row among ordinary candidates
    (rows with top-k 50 hold at most one candidate per lane, rows with 700 several)."""
    rng = np.random.default_rng(5)
    rows, vocab = 8, 20000
    if case == "one_wave_overflows":
        rows, vocab = 2, 151_936
    logits = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
    top_k = np.full(rows, 50)
    if case in ("k_700", "k_700_offset"):
        top_k[:] = 700
        if case == "k_700_offset":
            logits += 100.0
    elif case == "wide_window":
        for r in range(rows):
            logits[r, rng.choice(vocab, 3, replace=False)] = [1e20, 3e10, 7e5]
        top_k[rows // 2 :] = 700
    elif case == "one_wave_overflows":
        # the stream starts at logit 16384; lane t of the workgroup reads quad 4096 + t +
        # 1024 j, so wave 3 (lanes 192..255) reads logits 16384 + 4096 j + 768 .. + 1023
        for j in range(2):
            start = 16384 + 4096 * j + 768
            logits[:, start : start + 256] = 50.0
    elif case == "all_equal":
        logits[:] = 1.25
    elif case == "many_ties":
        logits[:, : vocab // 2] = 3.0  # 10000 values tied at the top
    elif case == "k_above_1024":
        top_k[:] = 3000
    elif case == "keep_all_rows":
        top_k[::2] = vocab
    else:
        top_k = rng.choice([1, 50, 2000, vocab], rows)
        logits[0] = 0.5
    tokens = np.argsort(-logits, axis=1, kind="stable")[np.arange(rows), rng.integers(0, 40, rows)]
    tokens[1] = int(np.argmin(logits[1]))
    top_p = np.full(rows, 0.9)
    assert_matches_oracle(logits, tokens, top_k, top_p)
    assert_matches_oracle(logits, tokens, top_k, top_p, top_k_host=top_k)


@pytest.mark.parametrize("vocab", [20001, 20003, 151937])
def test_odd_vocab_rows_take_every_alignment(vocab: int) -> None:
    """With an odd vocab the rows start at every 4-byte offset: aligned rows end in an
    element tail, the others stream element by element with lanes dropping out at the end of
    each range (the per-wave candidate counts must survive both), and short prefixes are
    re-read from memory.  Top-k + top-p rows (the candidate path) and rows without a top-k."""
    rng = np.random.default_rng(vocab)
    rows = 8
    logits = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    hot = rng.integers(0, vocab, (rows, 6))
    logits[np.arange(rows)[:, None], hot] += 12.0
    top_k = np.array([50, 50, 50, 50, 200, 700, vocab, 50])
    order = np.argsort(-logits, axis=1, kind="stable")
    tokens = order[np.arange(rows), rng.integers(0, 60, rows)]
    top_p = np.full(rows, 0.9)
    assert_matches_oracle(logits, tokens, top_k, top_p)
    assert_matches_oracle(logits, tokens, top_k, top_p, top_k_host=top_k)


def vllm_kept_row(row: np.ndarray, k: int, p: float) -> np.ndarray:
    """Token ids vLLM's own top-k then top-p masking keeps (apply_top_k_top_p_pytorch)."""
    order = np.argsort(row.astype(np.float64), kind="stable")
    srt = row.astype(np.float64)[order]
    srt[srt < srt[srt.size - k]] = -np.inf
    e = np.exp(srt - srt.max())
    cum = np.cumsum(e / e.sum())
    drop = cum <= 1 - p
    drop[-1] = False
    return order[np.isfinite(srt) & ~drop]


def test_baseline_workload_flags_every_planted_token() -> None:
    """256 x 151,936 FP32 logits ~ N(0, 3) with 8 hot tokens per row at +10..+20, top-k 50,
    top-p 0.9, T = 1: honest tokens drawn from vLLM's kept set all pass; 1% of rows get an
    out-of-set token (the row's argmin, as the plugin's fault injection does, or a token with at
    least 50 larger logits) and every one is flagged."""
    rows, vocab = 256, 151_936
    rng = np.random.default_rng(0)
    logits = (rng.standard_normal((rows, vocab)) * 3).astype(np.float32)
    for i in range(rows):
        hot = rng.choice(vocab, 8, replace=False)
        logits[i, hot] += rng.uniform(10, 20, 8).astype(np.float32)
    tokens = np.array([rng.choice(vllm_kept_row(logits[i], 50, 0.9)) for i in range(rows)])
    bad = rng.choice(rows, rows // 100, replace=False)
    for j, i in enumerate(bad):
        order = np.argsort(-logits[i])
        tokens[i] = int(np.argmin(logits[i])) if j % 2 == 0 else int(order[rng.integers(60, 5000)])
    top_k = np.full(rows, 50)
    top_p = np.full(rows, 0.9)
    out = run(logits, tokens, top_k, top_p, top_k_host=top_k)
    planted = np.zeros(rows, dtype=bool)
    planted[bad] = True
    assert not out["ok"][planted].any()  # every planted token caught
    assert out["ok"][~planted].all()  # no false alarm
    want = check_members_ref(logits[:32], tokens[:32], top_k[:32], top_p[:32], top_k_host=top_k[:32])
    np.testing.assert_array_equal(out["ok"][:32], want["ok"])
    np.testing.assert_array_equal(out["above"][:32], want["above"])
    for i in range(8):
        ref = check_member(logits[i], int(tokens[i]), 50, 0.9)
        if ref.ok:
            assert abs(float(out["mass_above"][i]) - ref.mass_above) <= member_eps32(vocab)


def test_top_k_outside_one_to_vocab_is_clamped_like_the_reference() -> None:
    """Requested top-k values below 1 or above V act as 1 and V (reference
    src/pck/member.py:153); the kernel clamps them, so no host-side clamp launch is needed."""
    rng = np.random.default_rng(3)
    logits = (rng.standard_normal((6, 300)) * 3).astype(np.float32)
    order = np.argsort(-logits, axis=1)
    tokens = order[np.arange(6), [0, 1, 0, 5, 2, 299]]
    top_k = np.array([0, -3, 1, 10**9, 301, 300])
    clamped = np.clip(top_k, 1, 300)
    got = run(logits, tokens, top_k, np.full(6, 0.9), top_k_host=clamped)
    want = run(logits, tokens, clamped, np.full(6, 0.9), top_k_host=clamped)
    for key in ("ok", "above"):
        np.testing.assert_array_equal(got[key], want[key])
    # candidates meet in LDS in arrival order, so the FP64 sums may differ in their last bits
    assert np.all(np.abs(got["mass_above"] - want["mass_above"]) <= 2 * member_eps32(300))
    assert_matches_oracle(logits, tokens, clamped, np.full(6, 0.9), top_k_host=clamped)


def test_request_index_outside_the_temperature_array_rejects_the_row() -> None:
    """The sampler-hook entry reads greedy through a per-row request index: an index outside
    [0, len(temperature)) rejects that row (counted as rejected in the device totals) without
    reading past the array, and the other rows keep their verdicts."""
    from pck.member import launch_check, new_totals

    rng = np.random.default_rng(11)
    rows, vocab = 8, 3000
    logits = torch.from_numpy(rng.standard_normal((rows, vocab)).astype(np.float32)).cuda()
    tokens = logits.argmax(dim=1)  # allowed under any top-k / top-p: every row passes
    temperature = torch.tensor([0.0, 1.0, 0.7], device="cuda")
    good = torch.tensor([0, 1, 2, 1, 0, 2, 1, 0], device="cuda")
    ref = launch_check(logits, tokens, temperature=temperature, temperature_index=good)
    assert bool(ref["ok"].all())
    bad = good.clone()
    bad[2], bad[5] = 3, -1  # past the end, negative
    totals = new_totals(logits.device)
    out = launch_check(logits, tokens, temperature=temperature, temperature_index=bad, totals=totals)
    assert out["ok"].tolist() == [True, True, False, True, True, False, True, True]
    assert int(totals[0]) == rows and int(totals[1]) == 2


SPLIT_CASES = ["plain", "ties", "masked", "all_masked", "nan", "sorted", "overflow", "overflow16", "mixed"]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("vocab", [24576, 24577, 32003, 151_937])
@pytest.mark.parametrize("case", SPLIT_CASES)
def test_rows_split_over_workgroups_match_the_oracle(case: str, vocab: int, dtype: torch.dtype) -> None:
    """Whole and partial last segments, rows at any 2- or 4-byte address, 16-bit logits read as
    they are; ties at the k-th logit, masked (-inf) rows, NaN, a row sorted within its segments,
    and segments with more logits above their bound than slots (one wave's logits all low), which
    takes the whole-row select.  Top-k 1, 50, 128 and none, with top-p; then top-k alone."""
    rng = np.random.default_rng(vocab + len(case))
    rows = 6
    logits = rng.standard_normal((rows, vocab)) * 3
    logits[np.arange(rows)[:, None], rng.integers(0, vocab, (rows, 6))] += 9.0
    if case == "ties":
        logits[:, 100:400] = np.sort(logits, axis=1)[:, -20:-19]
    elif case in ("masked", "all_masked"):
        keep = rng.random((rows, vocab)) < (0.001 if case == "masked" else 0.0)
        keep[:, rng.integers(0, vocab, 3)] |= case == "masked"
        logits[~keep] = -np.inf
        if case == "all_masked":
            logits[:, 7] = 1.0
    elif case == "nan":
        logits[::2, vocab - 1] = np.nan
    elif case == "sorted":
        logits[:] = 5.0 - (np.arange(vocab) % 8192) * 2.0**-9 + np.arange(rows)[:, None]
    elif case == "overflow":  # the fourth wave's FP32 logits
        logits[:, np.arange(vocab) % 1024 >= 768] = -50.0
    elif case == "overflow16":  # its 16-bit ones
        logits[:, np.arange(vocab) % 2048 >= 1536] = -50.0
    t = torch.from_numpy(logits).to(dtype)
    host = t.float().numpy()
    order = np.argsort(-np.nan_to_num(host, nan=-1e30), axis=1, kind="stable")
    top_k = np.array([1, 50, 128, 50, 7, vocab] if case == "mixed" else [1, 50, 128, 50, 7, 20])
    tokens = order[np.arange(rows), [0, 3, 90, 60, 2, 5]]
    top_p = np.array([0.9, 0.5, 0.999, 0.9, 1.0, 0.9])
    dev = lambda a: None if a is None else torch.as_tensor(a).cuda()  # noqa: E731
    for k, p in ((top_k, top_p), (None, top_p), (top_k, None)):
        out = check_members(t.cuda(), dev(tokens), dev(k), dev(p), top_k_host=k)
        got = {name: v.cpu().numpy() for name, v in out.items()}
        want = check_members_ref(host, tokens, k, p, None, top_k_host=k)
        np.testing.assert_array_equal(got["ok"], want["ok"])
        np.testing.assert_array_equal(got["above"], want["above"])
        if p is not None:
            finite = np.isfinite(want["mass_above"]) & ~np.isnan(host).any(axis=1)
            err = np.abs(got["mass_above"] - want["mass_above"])[finite]
            assert np.all(err <= 2 * member_eps32(vocab))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("tail", [1, 255, 257, 1105, 1600, 8191])
@pytest.mark.parametrize("case", ["plain", "sorted", "run"])
def test_candidates_of_ordinary_rows_fit_their_slots(case: str, tail: int, dtype: torch.dtype) -> None:
    """Rows whose last segment holds ``tail`` logits; logits sorted by token id; finite logits only
    in runs of 1,105.  No segment may have more logits above its bound than slots (the row would be
    selected again from memory, ten times slower), read from the headers of a workspace that the
    test holds: 48 bytes a segment, the count at byte 16, then the FP32 slots."""
    rows, vocab, k = 3, 12 * 8192 + tail, 50
    g = torch.Generator(device="cuda")
    g.manual_seed(tail)
    logits = torch.randn((rows, vocab), generator=g, device="cuda") * 3
    if case == "sorted":
        logits = logits.sort(dim=1, descending=True).values
    elif case == "run":
        logits[:, torch.arange(vocab, device="cuda") % 8192 >= 1105] = -torch.inf
    logits = logits.to(dtype).contiguous()
    tokens = logits.float().argmax(1)
    top_k = torch.full((rows,), k, device="cuda")
    top_p = torch.full((rows,), 0.9, dtype=torch.float64, device="cuda")
    ok = torch.empty(rows, dtype=torch.bool, device="cuda")
    args = PckMemberArgs(logits=logits.data_ptr(), rows=rows, vocab=vocab, tokens=tokens.data_ptr(),
                         top_k=top_k.data_ptr(), k_lim=k, all_k=1, top_p=top_p.data_ptr(),
                         slack=1e-4, ok=ok.data_ptr())  # fmt: skip
    kind = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}[dtype]
    need = ctypes.c_int64(0)
    assert lib().pck_check_members_workspace(args, kind, ctypes.byref(need)) == 0 and need.value > 0
    work = torch.zeros(need.value, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    assert lib().pck_check_members_split(args, kind, work.data_ptr(), need.value, stream) == 0
    torch.cuda.synchronize()
    assert bool(ok.all())
    segments = rows * 13
    slots = (need.value - 48 * segments) // (4 * segments)
    counts = work[: 48 * segments].view(torch.int32).view(segments, 12)[:, 4]
    assert int(counts.max()) <= slots, (slots, counts.tolist())


# (vocab, first hot id, top-k): the finish launch reads the first slots of 20 segments of 8,192 logits
# ahead and walks the others, and holds the headers of 256 in registers; ties at the k-th logit.
MANY_SEGMENTS = [(163_841, 163_840, [1, 50, 100, 7]), (262_144, 20 * 8192, [1, 50, 80, 7]),
                 (2_100_000, 256 * 8192, [1, 9, 5, 9])]  # fmt: skip


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize(("vocab", "hot", "ks"), MANY_SEGMENTS, ids=str)
def test_rows_of_many_segments_match_the_oracle(vocab: int, hot: int, ks: list[int], dtype: torch.dtype) -> None:
    """The largest logits, the k-th among them with its ties, lie in segments past those held ahead
    (row 3: before them); top-p with top-k, and top-p alone."""
    rng = np.random.default_rng(vocab)
    logits = np.clip(rng.standard_normal((4, vocab)) * 2, -9, 7)
    for r, k in enumerate(ks):
        start, end = (0, hot) if r == 3 else (hot, vocab)
        at = rng.permutation(end - start)[: 2 * k] + start
        logits[r, at] = 8 + np.arange(at.size)[::-1] / 16  # descending: at[k - 1] is the k-th
        if at.size > k > 1:
            logits[r, at[k:]] = logits[r, at[k - 1]]
    t = torch.from_numpy(logits).to(dtype)
    host = t.float().numpy()
    order = np.argsort(-host, axis=1, kind="stable")
    top_k = np.array(ks)
    tokens = order[np.arange(4), [0, 1, top_k[2] - 1, 3]]
    top_p = np.array([0.9, 0.9, 1 - 1e-9, 0.5])
    for k in (top_k, None):
        dev = None if k is None else torch.from_numpy(k).cuda()
        out = check_members(t.cuda(), torch.from_numpy(tokens).cuda(), dev, torch.from_numpy(top_p).cuda(), top_k_host=k)
        want = check_members_ref(host, tokens, k, top_p, None, top_k_host=k)
        np.testing.assert_array_equal(out["ok"].cpu().numpy(), want["ok"])
        np.testing.assert_array_equal(out["above"].cpu().numpy(), want["above"])
        err = np.abs(out["mass_above"].cpu().numpy() - want["mass_above"])
        assert np.all(err <= 2 * member_eps32(vocab))


@pytest.mark.parametrize("vocab", [12_548, 14_532, 16_320, 31_004, 47_408, 64_900])
@pytest.mark.parametrize("k", [5, 60, 200])
def test_candidates_at_the_end_of_the_unrolled_loads_are_all_kept(vocab: int, k: int) -> None:
    """FP32 rows whose last unrolled step of four 16-byte loads ends inside a wave: the lanes past that
    point take their last loads one at a time.  The kept logits lie in that wave's last loads, on both
    sides of the point, so one lost or written over changes the k-th logit, the masses or the verdict."""
    base = 0 if vocab < 16_384 else 4096  # quads before the streamed part
    n = vocab // 4 - base
    edge = n % 4096 - 3072  # the first lane whose last unrolled step is not whole
    assert 0 < edge < 1024 and edge % 64 != 0
    t = np.arange(edge // 64 * 64, edge // 64 * 64 + 64)
    quads = (base + n // 4096 * 4096 + t[:, None] + 1024 * np.arange(4)).reshape(-1)
    places = (4 * quads[quads < vocab // 4][:, None] + np.arange(4)).reshape(-1)
    rng = np.random.default_rng(vocab + k)
    rows = 170  # one workgroup per row at every vocabulary here
    logits = np.clip(rng.standard_normal((rows, vocab)) * 2, -9, 7).astype(np.float32)
    for r in range(rows):
        at = rng.permutation(places)[: k + 20]
        logits[r, at] = 8 + np.arange(at.size, dtype=np.float32)[::-1] / 64
    order = np.argsort(-logits, axis=1, kind="stable")
    tokens = order[np.arange(rows), rng.integers(0, k, rows)]
    top_k, top_p = np.full(rows, k), np.full(rows, 0.7)
    assert_matches_oracle(logits, tokens, top_k, top_p, top_k_host=top_k)
