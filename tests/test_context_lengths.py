"""The lengths that a timed decode step's sequences have (``CausalLM.tune``)."""
import pytest

from pytorch_transformers_amd import tuning


@pytest.mark.parametrize("longest,mean,n", [(4090, 2224, 16), (1100, 1100, 8), (2049, 2049, 64), (700, 300, 3), (5000, 200, 16), (100, 1, 16), (10, 9, 4),
                                            (4090, 3900, 16), (3, 1, 2), (1, 1, 5), (8192, 4096, 64), (900, 450, 1), (500, 700, 4)])
def test_longest_and_mean_come_out(longest, mean, n):
    lens = tuning.context_lengths(longest, mean, n)
    assert len(lens) == n and max(lens) == longest and min(lens) >= 1
    want = max(min(mean, longest) * n, longest + n - 1) if n > 1 else longest  # n sequences of one key at the least, beside the longest
    assert sum(lens) == want
    if mean >= longest:
        assert set(lens) == {longest}


def test_spread_and_in_no_order():
    lens = tuning.context_lengths(4096, 2048, 16)
    assert len(set(lens)) == 16 and min(lens) < 300
    steps = [b - a for a, b in zip(sorted(lens), sorted(lens)[1:])]
    assert max(steps) <= 2 * 4096 / 15 and lens != sorted(lens) and lens != sorted(lens, reverse=True)
    ups = sum(b > a for a, b in zip(lens, lens[1:]))
    assert 5 <= ups <= 10
