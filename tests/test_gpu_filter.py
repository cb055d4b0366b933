"""GPU parity of top-k / top-p filtering (specdec/sampler.py:19-56) against the oracle.

* ``spv_filter_logits``: over rows of V = 151,936 logits ~ N(0, 2^2) at T = 1
  and 0.7, with top_k in {50, 1000}, top_p in {0.9, 0.5} and their
  combinations, the kept values are identical to the oracle's
  ``apply_top_p(apply_top_k(z / T))`` (-inf everywhere else) and so is the
  kept set, except where the nucleus rule is decided within rounding. The
  kernel sums masses in fp64 against the exact total; torch's fp32 softmax of
  a 151,936-entry row sums to 1 +- eps (its normalisation rounds), which
  shifts every preceding mass it compares with top_p by up to eps. A value
  whose exact (float64) preceding mass lies within 2 eps + 2e-6 of top_p may
  therefore fall either way. The kernel reports, per row, how many values lie
  within its fixed window (5e-5 W, W the kept mass) of the edge: the test
  checks that the window covers 2 eps + 2e-6 on every row, that every
  differing value lies in it, and that the kernel's count equals the count of
  the oracle's float64 masses (up to the values within 1e-6 W of the window's
  own edges, where the kernel's fp32-rounded masses may place them otherwise).
  Ties at the k-th value all stay.
* the reference's own filter tests (tests/test_sampler.py:34-49, 76-78).
* the fused verify sampler at the Qwen2.5 vocabulary (B = 64, gamma = 5,
  V = 151,936, T = 1) with top_k = 50, top_k = 1000 and top_p = 0.9: token ids,
  accept lengths bit-exact against the oracle; batched draft sampling with a
  filter likewise.
"""

from __future__ import annotations

import pytest
import torch

from engine import _hip
from engine import spec_scheduler as es
from oracle import sampler as S
from oracle import spec_step as ref_step
from specdec import sampler as gs
from specdec.config import SamplingConfig

pytestmark = pytest.mark.gpu

V = 151936


def _softmax_sum_error(x, top_k):
    """|sum of torch's fp32 softmax over the sorted kept values - 1| (the
    reference's normalisation error on this row)."""
    r = S.apply_top_k(x.float(), top_k)
    s, _ = torch.sort(r, descending=True)
    return abs(float(torch.softmax(s, -1).double().sum()) - 1.0)


def _mass_before(x, top_k):
    """float64 mass before each value of a row in descending order, over what
    top-k kept (inf where top-k dropped the value)."""
    r = S.apply_top_k(x.float(), top_k).double()
    keep = torch.isfinite(r)
    w = torch.where(keep, torch.exp(r - r[keep].max()), torch.zeros_like(r))
    order = torch.argsort(r, descending=True, stable=True)
    before = torch.empty_like(w)
    before[order] = torch.cumsum(w[order], 0) - w[order]
    before = before / w.sum()
    return torch.where(keep, before, torch.full_like(before, float("inf")))


WINDOW = 5e-5  # the kernel's window around the nucleus edge, relative to the kept mass


def _compare_kept(got, want, scaled, top_k, top_p, counts=None):
    """Kept values equal where both keep; a differing kept flag only where the
    rule is decided within rounding; the kernel's window counts equal the
    oracle's. Returns (values in the window, differing)."""
    gk, wk = torch.isfinite(got), torch.isfinite(want)
    both = gk & wk
    assert torch.equal(got[both], want[both])
    amb = diff = 0
    for r in range(got.shape[0]):
        d = (gk[r] != wk[r]).nonzero().flatten()
        if not 0.0 < top_p < 1.0:
            assert d.numel() == 0, r
            if counts is not None:
                assert int(counts[r]) == 0
            continue
        rounding = 2 * _softmax_sum_error(scaled[r], top_k) + 2e-6
        assert rounding <= WINDOW, (r, rounding)
        dist = (_mass_before(scaled[r], top_k) - top_p).abs()
        near = dist < WINDOW
        amb += int(near.sum())
        diff += int(d.numel())
        assert bool(near[d].all()), (r, d.tolist()[:8])
        if counts is not None:
            edge = int(((dist - WINDOW).abs() < 1e-6).sum())
            assert abs(int(counts[r]) - int(near.sum())) <= edge, (r, int(counts[r]), int(near.sum()), edge)
    return amb, diff


@pytest.mark.parametrize("T", [1.0, 0.7])
@pytest.mark.parametrize("top_k,top_p", [(50, 1.0), (1000, 1.0), (0, 0.9), (0, 0.5), (1000, 0.9), (50, 0.5)])
def test_filter_rows_match_the_oracle(cuda, T, top_k, top_p):
    g = torch.Generator().manual_seed(top_k * 7 + int(top_p * 10) + int(T * 100))
    z = torch.randn(6, V, generator=g) * 2
    want = S.filter_logits(z, T, top_k, top_p)
    got, counts = _hip.filter_rows(z.to(cuda), T, top_k, top_p, ambiguous=True)
    got_plain = _hip.filter_rows(z.to(cuda), T, top_k, top_p)
    assert torch.equal(got, got_plain)  # the window searches change nothing kept
    amb, diff = _compare_kept(got.cpu(), want, z / T, top_k, top_p, counts.cpu())
    print("top_k {} top_p {} T {}: {} values within the window (kernel {}), {} differ".format(
        top_k, top_p, T, amb, int(counts.sum()), diff))


def test_window_count_at_a_crafted_edge(cuda):
    """Rows built so that many distinct values sit at the nucleus edge: 4,000
    logits spaced 1e-6 apart carry nearly all the mass, so each holds ~1/4000
    of W and the window (5e-5 W on each side of 0.6 W) holds at most the one
    value whose preceding mass is nearest the edge; and a row whose edge falls
    far from any value's preceding mass (count 0)."""
    z = torch.full((2, V), -30.0)
    z[0, :4000] = torch.arange(4000, dtype=torch.float32) * 1e-6
    z[1, 10] = 5.0
    z[1, 20] = 4.0
    want = S.filter_logits(z, 1.0, 0, 0.6)
    got, counts = _hip.filter_rows(z.to(cuda), 1.0, 0, 0.6, ambiguous=True)
    _compare_kept(got.cpu(), want, z, 0, 0.6, counts.cpu())
    assert int(counts[0]) <= 1
    assert int(counts[1]) == 0


def test_ties_at_the_kth_value_all_stay(cuda):
    z = torch.zeros(2, 1000)
    z[0, :10] = torch.tensor([9.0, 8.0, 7.0, 7.0, 7.0, 5.0, 4.0, 3.0, 2.0, 1.0])
    z[1, 500:505] = 6.0  # five equal maxima, top_k = 2
    want = S.filter_logits(z, 1.0, 3, 1.0)
    got = _hip.filter_rows(z.to(cuda), 1.0, 3, 1.0).cpu()
    assert torch.equal(got, want)
    assert int(torch.isfinite(got[0]).sum()) == 5 and int(torch.isfinite(got[1]).sum()) == 5


def test_reference_filter_tests_on_the_gpu(cuda):
    f = gs.apply_top_k(torch.tensor([[5.0, 4.0, 3.0, 2.0, 1.0]], device=cuda), 2).cpu()
    assert torch.isfinite(f).sum().item() == 2 and float(f[0, 0]) == 5.0
    f = gs.apply_top_p(torch.log(torch.tensor([[0.5, 0.3, 0.15, 0.05]], device=cuda)), 0.8)
    probs = torch.softmax(f, dim=-1).cpu()
    assert float(probs[0, 3]) == 0.0 and float(probs.sum()) >= 0.8 - 1e-6
    logits = torch.randn(1, 8)
    assert torch.allclose(gs.apply_top_p(logits.to(cuda), 1.0).cpu(), logits)


def test_logits_to_probs_with_filters(cuda):
    g = torch.Generator().manual_seed(3)
    z = torch.randn(4, 5000, generator=g) * 2
    cfg = SamplingConfig(temperature=0.8, top_k=100, top_p=0.9)
    got = gs.logits_to_probs(z.to(cuda), cfg).cpu()
    want = S.logits_to_probs(z, 0.8, 100, 0.9)
    assert torch.equal(got == 0, want == 0)
    assert torch.allclose(got, want, rtol=2e-6, atol=1e-9)


def _workload(seed, B=64, gamma=5):
    g = torch.Generator().manual_seed(seed)
    target = torch.randn(B, gamma + 1, V, generator=g) * 2.0
    draft = target[:, :gamma] + torch.randn(B, gamma, V, generator=g)
    u = torch.rand(B, gamma, generator=g)
    noise = torch.empty(B, V).exponential_(1, generator=g)
    return g, target, draft, u, noise


@pytest.mark.parametrize("top_k,top_p", [(50, 1.0), (1000, 1.0), (0, 0.9)])
def test_fused_sampler_with_filters(cuda, top_k, top_p):
    g, target, draft, u, noise = _workload(70 + top_k)
    q = S.logits_to_probs(draft, 1.0, top_k, top_p)
    x = torch.multinomial(q.reshape(-1, V), 1, generator=g).reshape(64, 5)
    want = S.verify_from_logits(target, draft, x, u, noise, 1.0, top_k, top_p)
    res = es.verify_sample(target.to(cuda), draft.to(cuda), x.to(cuda), u.to(cuda), noise.to(cuda), 1.0,
                           top_k=top_k, top_p=top_p)
    flags = res.flags.tolist()
    for b, (g_, w, f) in enumerate(zip(res.accepted_lists(), want, flags)):
        assert g_ == w or f, (b, g_, w)
    if top_p == 1.0:
        assert flags.count(0) >= len(flags) - 2  # top-k alone is exact; decisions rarely flagged
    print("{} of {} sequences flagged ({} with a row at the nucleus edge)".format(
        sum(1 for f in flags if f), len(flags), sum(1 for f in flags if f & _hip.FLAG_TOP_P_BAND)))


def test_draft_sample_with_filters(cuda):
    g = torch.Generator().manual_seed(5)
    z = torch.randn(16, V, generator=g) * 2
    e = torch.empty(16, V).exponential_(1, generator=g)
    for top_k, top_p in ((50, 1.0), (0, 0.9), (200, 0.5)):
        want = [S.race_argmax(S.logits_to_probs(z[b], 1.0, top_k, top_p), e[b]) for b in range(16)]
        got = es.draft_sample(z.to(cuda), 1.0, e.to(cuda), top_k=top_k, top_p=top_p)
        assert got.tolist() == want, (top_k, top_p)


def _general(t, d, x, u, noise, T, top_k, top_p):
    """Filtered rows, then the unfiltered sampler on them at T = 1."""
    ft, nt = _hip.filter_rows(t, T, top_k, top_p, ambiguous=True)
    fd, nd = _hip.filter_rows(d, T, top_k, top_p, ambiguous=True)
    res = es.verify_sample(ft, fd, x, u, noise, 1.0)
    res.flags.bitwise_or_(((nt.sum(1) + nd.sum(1)) > 0).int() * _hip.FLAG_TOP_P_BAND)
    return res


@pytest.mark.parametrize("B,gamma,vocab,T,top_k,top_p", [
    (3, 2, 8, 1.0, 3, 0.7),              # a row shorter than a wave
    (2, 1, 1023, 0.7, 400, 0.9),         # rows that are not whole float4, few values per thread
    (3, 4, 50257, 1.3, 50, 0.95),        # the same over several small pieces
    (1, 32, 10236, 1.0, 20, 1.0),        # one full small piece; the longest draft
    (1, 3, 10240, 0.5, 512, 0.8),        # one value more than a piece; the largest top_k
    (40, 5, 40957, 1.0, 100, 0.9),       # two large pieces, unaligned rows
    (60, 5, 16380, 1.0, 30, 0.9),        # one full middle piece
    (60, 5, 16381, 0.9, 30, 0.8),        # one value more, unaligned
    (20, 5, 151936, 1.0, 129, 0.9),      # the largest top_k of the middle pieces, and one more
    (20, 5, 151936, 1.0, 130, 0.9),
    (64, 5, 151936, 0.8, 50, 0.9),       # the fused workload
    (20, 2, 151936, 1.0, 513, 0.9),      # top_k above the short form's
])
def test_filtered_sampler_short_form_equals_the_general_path(cuda, B, gamma, vocab, T, top_k, top_p):
    g = torch.Generator(device=cuda).manual_seed(B * 1000 + vocab)
    t = torch.randn(B, gamma + 1, vocab, generator=g, device=cuda) * 2
    d = t[:, :gamma] + 0.5 * torch.randn(B, gamma, vocab, generator=g, device=cuda)
    # bf16-valued rows (ties at the edges), rows with most entries masked, values of both signs of zero
    t[0] = t[0].bfloat16().float()
    if B > 1:
        t[1, 0, 5:] = float("-inf")
        d[1, 0, 5:] = float("-inf")
        t[1, 1] = torch.where(t[1, 1] > 0, 0.0, -0.0)
    d = d.contiguous()
    q = torch.softmax(_hip.filter_rows(d, T, top_k, top_p), -1)
    x = torch.multinomial(q.reshape(-1, vocab), 1, generator=g).reshape(B, gamma).int()
    u = torch.rand(B, gamma, generator=g, device=cuda)
    noise = torch.empty(B, vocab, device=cuda).exponential_(1, generator=g)
    want = _general(t, d, x, u, noise, T, top_k, top_p)
    for _ in range(2):  # the arrival counters are left at zero
        got = es.verify_sample(t, d, x, u, noise, T, top_k=top_k, top_p=top_p)
        certain = (want.flags | got.flags) == 0
        assert torch.equal(got.accept_len[certain], want.accept_len[certain])
        assert torch.equal(got.out_tokens[certain], want.out_tokens[certain])
        assert torch.equal(got.n_commit, got.accept_len + 1)
        differ = int(((got.out_tokens != want.out_tokens).any(1)).sum())
        assert differ <= B // 16, differ  # flagged sequences mostly agree as well
        # the nucleus window's count moves only where a value lies at the window's own rim
        assert int((got.flags != want.flags).sum()) <= B // 16 + (1 if top_p < 1 else 0)


@pytest.mark.parametrize("odd", ["nan", "inf", "ties", "masked", "zero_noise", "tiny_T"])
def test_filtered_sampler_rows_the_short_form_leaves(cuda, odd):
    """Sequence 1's rows or noise are outside the short form; the others' are not."""
    B, gamma, vocab, T = 4, 3, 30000, 1.0
    g = torch.Generator(device=cuda).manual_seed(3)
    t = torch.randn(B, gamma + 1, vocab, generator=g, device=cuda) * 2
    d = t[:, :gamma] + torch.randn(B, gamma, vocab, generator=g, device=cuda)
    noise = torch.empty(B, vocab, device=cuda).exponential_(1, generator=g)
    if odd == "nan":
        t[1, 0, 77] = float("nan")
    elif odd == "inf":
        d[1, 1, 4000] = float("inf")
    elif odd == "ties":
        t[1, 0] = 1.0  # every value is the k-th largest
    elif odd == "masked":
        t[1, 2] = float("-inf")
    elif odd == "zero_noise":
        noise[1, 12345] = 0.0
    else:
        T = 1e-4  # the whole call
    d = d.contiguous()
    x = d.nan_to_num(0.0, 0.0).argmax(-1).int()
    u = torch.rand(B, gamma, generator=g, device=cuda)
    want = _general(t, d, x, u, noise, T, 40, 0.9)
    got = es.verify_sample(t, d, x, u, noise, T, top_k=40, top_p=0.9)
    assert torch.equal(got.accept_len, want.accept_len)
    assert torch.equal(got.out_tokens, want.out_tokens)
    assert torch.equal(got.flags, want.flags)


@pytest.mark.parametrize("T", [1.0, 0.7])
@pytest.mark.parametrize("top_k,above", [(40, 30), (600, 590)])  # the short form, the general path
def test_both_zeros_tie_at_the_kth_value(cuda, T, top_k, above):
    """The k-th value is +0.0: the float comparison drops neither zero, so a token
    at -0.0 stays and can be drawn."""
    vocab, B, gamma = 3000, 3, 2
    g = torch.Generator().manual_seed(top_k)
    z = -torch.rand(B, gamma + 1, vocab, generator=g) - 0.5
    perm = torch.randperm(vocab, generator=g)
    up, plus, minus = perm[:above], perm[above:above + 20], perm[above + 20:above + 45]
    z[..., up] = torch.rand(B, gamma + 1, above, generator=g) * 0.5
    z[..., plus], z[..., minus] = 0.0, -0.0
    want = S.filter_logits(z, T, top_k, 1.0)
    assert bool(torch.isfinite(want[..., minus]).all()) and int(torch.isfinite(want[0, 0]).sum()) == above + 45
    assert torch.equal(_hip.filter_rows(z.to(cuda), T, top_k, 1.0).cpu(), want)
    draft = z[:, :gamma].contiguous()
    x = up[torch.arange(B * gamma).reshape(B, gamma)].int()
    u = torch.zeros(B, gamma)
    noise = torch.empty(B, vocab).exponential_(1, generator=g).clamp_min_(0.1)
    noise[:, minus[3]] = 1e-6  # the bonus draw goes to a token at -0.0
    got = es.verify_sample(z.to(cuda), draft.to(cuda), x.to(cuda), u.to(cuda), noise.to(cuda), T, top_k=top_k)
    assert got.accepted_lists() == S.verify_from_logits(z, draft, x, u, noise, T, top_k, 1.0)
    assert all(t[-1] == int(minus[3]) for t in got.accepted_lists())


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("top_p", [1.0, 0.9])
@pytest.mark.parametrize("eos,budget", [(None, True), (3, True), (3, False), (None, False)])
def test_commit_of_filtered_sampling_matches_oracle(cuda, eos, budget, top_p, mixed):
    """Start positions, budgets (zero and negative ones too) and an eos among the
    accepted tokens or drawn, in the one-launch form; ``mixed``: every third sequence
    has 2,992 ties at the k-th value, which the general kernels commit."""
    B, gamma, vocab, top_k = 36, 4, 3000, 8
    g = torch.Generator().manual_seed(22 + int(10 * top_p))
    target = torch.randn(B, gamma + 1, vocab, generator=g) - 8.0
    target[..., :8] += 8.0  # eight likely tokens, the eos among them
    draft = target[:, :gamma] + 0.3 * torch.randn(B, gamma, vocab, generator=g)
    if mixed:
        target[1::3, 0, 8:] = -12.0
        target[1::3, 0, 5:8] = -13.0
    q = S.logits_to_probs(draft, 1.0, top_k, top_p)
    x = torch.multinomial(q.reshape(-1, vocab), 1, generator=g).reshape(B, gamma)
    u = torch.rand(B, gamma, generator=g)
    noise = torch.empty(B, vocab).exponential_(1, generator=g)
    start = torch.randint(10, 100, (B,), generator=g)
    remaining = torch.randint(1, 7, (B,), generator=g)
    remaining[:8] = torch.tensor([0, 0, -1, -1, -2, -2, 1, 1])  # both kinds of sequence
    want = S.verify_from_logits(target, draft, x, u, noise, 1.0, top_k, top_p)
    res = es.verify_sample(target.to(cuda), draft.to(cuda), x.to(cuda), u.to(cuda), noise.to(cuda), 1.0,
                           start_pos=start.to(cuda), remaining=remaining.to(cuda) if budget else None, eos_id=eos,
                           top_k=top_k, top_p=top_p)
    n_commit, fin, new_len = res.n_commit.tolist(), res.finished.tolist(), res.new_len.tolist()
    flags, hits = res.flags.tolist(), [0, 0]
    assert flags.count(0) >= B - 6
    for b, got in enumerate(res.accepted_lists()):
        assert got == want[b] or flags[b], b
        rem = int(remaining[b]) if budget else len(got)
        kept, eos_hit = ref_step.cut_accepted(got, rem, eos)
        k = len(kept)
        assert n_commit[b] == k, b
        assert fin[b] == int(eos_hit or k == 0 or (budget and k >= rem)), b
        assert new_len[b] == (int(start[b]) + k if k > 0 else -1), b
        if eos_hit:
            hits[k == len(got) - 1] += 1
    assert eos is None or min(hits) > 0  # an eos among the accepted tokens, and drawn


@pytest.mark.parametrize("top_k", [0, 5])
@pytest.mark.parametrize("top", [-2.5e38, -3.4e38, torch.finfo(torch.float32).min])
def test_rows_masked_with_the_lowest_value(cuda, top, top_k):
    """A row whose largest value times log2 e is beyond fp32: three values share the
    mass, the others (the type's lowest, or nothing at all) have none."""
    vocab, low = 900, torch.finfo(torch.float32).min
    z = torch.full((2, 2, vocab), low if top > low else float("-inf"))
    z[..., [7, 300, 899]] = top
    want = S.filter_logits(z, 1.0, top_k, 0.9)
    assert int(torch.isfinite(want).sum()) == 3 * 4
    got, near = _hip.filter_rows(z.to(cuda), 1.0, top_k, 0.9, ambiguous=True)
    assert torch.equal(got.cpu(), want) and not bool(near.any())
    if top_k:  # the one-launch form
        x = torch.tensor([[7], [300]], dtype=torch.int32)
        u, noise = torch.tensor([[0.5], [0.5]]), torch.ones(2, vocab)
        noise[0, 899] = noise[1, 7] = 0.25
        draft = z[:, :1].contiguous()
        res = es.verify_sample(z.to(cuda), draft.to(cuda), x.to(cuda), u.to(cuda), noise.to(cuda), 1.0,
                               top_k=top_k, top_p=0.9)
        assert res.accepted_lists() == S.verify_from_logits(z, draft, x, u, noise, 1.0, top_k, 0.9) == [[7, 899], [300, 7]]
        assert res.flags.tolist() == [0, 0]


@pytest.mark.parametrize("top_k,top_p", [(0, 0.9), (0, 1e-6), (3, 0.5), (1, 1.0), (2, 0.99)])
@pytest.mark.parametrize("odd", ["nan", "two nans", "inf", "inf and nan", "-inf row"])
def test_rows_without_a_mass(cuda, odd, top_k, top_p):
    """The masses of a row with a NaN or +inf have no value: nothing is masked by
    them, as in the reference; a NaN at the k-th place drops nothing."""
    for vocab in (5, 300, 5000):
        z = torch.randn(4, vocab, generator=torch.Generator().manual_seed(vocab)).round()  # ties
        if "nan" in odd:
            z[1, 3] = float("nan")
        if odd == "two nans":
            z[1, vocab - 1] = float("nan")
        if "inf" in odd:
            z[2, 1] = float("inf")
        if odd == "-inf row":
            z[2] = float("-inf")
        want = S.filter_logits(z, 1.0, top_k, top_p)
        for _ in range(3):
            got, near = _hip.filter_rows(z.to(cuda), 1.0, top_k, top_p, ambiguous=True)
            for b, whole in ((1, "nan" in odd), (2, "inf" in odd)):
                if whole:
                    assert torch.equal(got[b].cpu().nan_to_num(7.5), want[b].nan_to_num(7.5)), (vocab, b)
                    assert int(near[b]) == 0 or odd == "-inf row"
            assert torch.equal(got[0].isfinite().sum().cpu(), want[0].isfinite().sum())
