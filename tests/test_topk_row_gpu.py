"""logprob_topk where its one-read kernel begins and ends: vocabularies at the edges of the
registers' vectors, rows off 16-byte alignment, ties past the candidate buffers, rows
without a bound and rule lists at the limit -- against a stable 64-bit sort."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
# vocabulary, forced and banned tokens where the kernel hands over
ROWS, LAST, BANS = 56 * 1024 - 16, 33, 21


def expect(logits, k, log_softmax, bans=(), forced=None):
    x = logits.double().cpu()
    scores = torch.log_softmax(x, -1) if log_softmax else x.clone()
    if forced is not None:
        scores.fill_(-math.inf)
        scores[:, [t for t in forced if t < x.shape[1]]] = 0.0
    scores[:, list(bans)] = -math.inf
    best, ids = torch.sort(scores, dim=-1, descending=True, stable=True)
    return best[:, :k], ids[:, :k]


def check(logits, k, log_softmax, want, **kw):
    from vflorence_amd import decoder_ops

    got_v, got_i = decoder_ops.logprob_topk(logits, k, log_softmax=log_softmax, **kw)
    # scores are 32-bit sums of up to 57 thousand terms, summed in parallel
    torch.testing.assert_close(got_v.double().cpu(), want[0], rtol=2e-6, atol=2e-6)
    assert torch.equal(got_i.cpu(), want[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("vocab", [1, 9, 63, 1025, 8 * 1024 + 5, 50265, ROWS - 1, ROWS, ROWS + 1])
@pytest.mark.parametrize("offset", [0, 3])
def test_sizes_and_alignment(dtype, vocab, offset):
    g = torch.Generator(device="cuda").manual_seed(vocab)
    pool = (torch.randn(5, vocab + 7, device="cuda", generator=g) * 3).to(dtype)
    logits = pool[:, offset:offset + vocab]
    for k, log_softmax in ((min(16, vocab), True), (1, False), (min(5, vocab), True)):
        check(logits, k, log_softmax, expect(logits, k, log_softmax))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows, vocab", [
    (3, 448), (3, 449), (3, 896), (3, 897),              # as many groups as k = 8 takes
    (257, 704), (257, 705), (257, 1408), (257, 1409),    # half as many again
    (512, 9001), (513, 9001), (513, 11999), (513, 12000), (513, 19999), (513, 20000),
])
def test_sizes_around_the_rule(dtype, rows, vocab):
    g = torch.Generator(device="cuda").manual_seed(rows + vocab)
    logits = (torch.randn(rows, vocab, device="cuda", generator=g) * 3).to(dtype)
    check(logits, 8, True, expect(logits, 8, True))


@pytest.mark.parametrize("tied", [3, 40, 200, 511, 513, 3000])
def test_ties_at_the_threshold(tied):
    """``tied`` tokens share the second largest value: the lowest of them are listed."""
    g = torch.Generator(device="cuda").manual_seed(tied)
    logits = torch.randn(4, 50265, device="cuda", generator=g).bfloat16().clamp(max=8)
    for row in logits:
        where = torch.randperm(50265, device="cuda", generator=g)
        row[where[:tied]] = 9.0
        row[where[-1]] = 10.0
    for k in (8, 16):
        check(logits, k, True, expect(logits, k, True))


@pytest.mark.parametrize("finite", [0, 5, 300])
def test_rows_of_few_finite_values(finite):
    logits = torch.full((3, 50265), -math.inf, device="cuda")
    logits[:, 100:100 + finite] = torch.arange(finite, device="cuda").float() / 8
    check(logits, 8, False, expect(logits, 8, False))
    if finite:
        check(logits, 8, True, expect(logits, 8, True))


@pytest.mark.parametrize("count", [1, 17, BANS - 1, BANS, LAST - 1, LAST, 200])
@pytest.mark.parametrize("k", [1, 16])
def test_rule_lists(count, k):
    """Banned tokens that would be the best ones; forced tokens, some repeated, banned or
    past the vocabulary, at the lowest and other token ids."""
    from vflorence_amd import decoder_ops

    g = torch.Generator(device="cuda").manual_seed(count)
    logits = torch.randn(6, 50265, device="cuda", generator=g)
    bans = torch.randperm(50265, device="cuda", generator=g)[:count]
    logits[:, bans] += 20
    bans = bans.tolist()
    forced = ([3, 50300, 3, 0, bans[0]] + torch.randperm(50265, generator=torch.Generator(
        ).manual_seed(count)).tolist())[:count]
    rules = decoder_ops.TopkRules(eos=[2], suppress=[], begin_suppress=bans, forced_bos=[],
                                  forced_eos=forced, min_length=0, max_length=9, begin_index=8,
                                  device="cuda")
    for length, kw in ((8, dict(bans=bans, forced=forced)), (7, {})):
        lengths = torch.full((6,), length, dtype=torch.int64, device="cuda")
        check(logits, k, True, expect(logits, k, True, **kw), lengths=lengths, rules=rules)
    rules = decoder_ops.TopkRules(eos=[], suppress=bans, begin_suppress=[], forced_bos=[],
                                  forced_eos=[], min_length=0, max_length=99, begin_index=-1,
                                  device="cuda")
    lengths = torch.full((6,), 7, dtype=torch.int64, device="cuda")
    check(logits, k, True, expect(logits, k, True, bans=bans), lengths=lengths, rules=rules)
    # forced tokens with one ban: the limits of the two lists are apart
    rules = decoder_ops.TopkRules(eos=[2], suppress=[], begin_suppress=[forced[-1]], forced_bos=[],
                                  forced_eos=forced, min_length=0, max_length=9, begin_index=8,
                                  device="cuda")
    lengths = torch.full((6,), 8, dtype=torch.int64, device="cuda")
    check(logits, k, True, expect(logits, k, True, bans=forced[-1:], forced=forced),
          lengths=lengths, rules=rules)
