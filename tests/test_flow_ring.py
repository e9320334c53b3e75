"""The exchange ring of value-only scan launches, checked as a protocol on
the CPU.

Every commit stores its word with the number of its snapshot in slot
s % RING of a ring; a read of a word of snapshot s waits until the slot
holds that number (jq_scan.hip, flow_gather).  Before every RING / 2-th
cycle c a block waits until every block has completed at least
c - (RING / 2 - 1) cycles (flow_room), so that no commit overwrites a word
that somebody has still to read.

Random schedules that starve some of the blocks follow only these two
rules: no read may find its slot already overwritten, and some block must
always be able to run.  A room rule that is one cycle too generous, or
none, must lose a word in some schedule."""
import numpy as np
import pytest

from test_flow_protocol import _chains, _script

RING = 8


def _lost(chains, nb, M, cycles, rng, slack=RING // 2 - 1, room=True):
    """Runs one random schedule; true when a read found its slot overwritten."""
    lo = min(min(w) for parts in chains.values() for _, w in parts if w)
    ring = [dict() for _ in range(RING)]
    step = [0] * nb
    slow = set(rng.choice(nb, max(1, nb // 4), replace=False).tolist())
    while min(step) < cycles * M:
        ready = []
        for b in range(nb):
            c, m = divmod(step[b], M)
            if c == cycles:
                continue
            if room and m == 0 and c and c % (RING // 2) == 0 and \
                    any(q // M + slack < c for q in step):
                continue
            held = [(c + o, w) for reads, _ in chains[(m, b)] for w, o in reads
                    if w >= lo and c + o > 0]
            at = [ring[k % RING].get(w, 0) for k, w in held]
            if any(a > k for a, (k, _) in zip(at, held)):
                return True
            if all(a == k for a, (k, _) in zip(at, held)):
                ready.append(b)
        assert ready, "no block can run: the rules deadlock"
        fast = [b for b in ready if b not in slow]
        b = int(rng.choice(fast if fast and rng.random() < 0.995 else ready))
        c, m = divmod(step[b], M)
        for _, writes in chains[(m, b)]:
            for w in writes:
                ring[(c + 1) % RING][w] = c + 1
        step[b] += 1
    return False


def _pipeline():
    """Four blocks, two major stages: each block's stage-1 word is made from
    its stage-0 word and read by the next block a cycle later.  Nobody waits
    for a reader, so the front can run away from the back: what the room
    rule is for.  {(m, b): [(reads, writes)]} as _chains gives it."""
    chains = {}
    for b in range(4):
        chains[(0, b)] = [([(10 + 2 * b - 1, False)] if b else [(0, False)], [10 + 2 * b])]
        chains[(1, b)] = [([(10 + 2 * b, True)], [11 + 2 * b])]
    return chains, 4, 2


def _random():
    s = _script(4000, 12, 4, 150, 6)
    return _chains(s), s.num_blocks, s.num_major_stages


@pytest.mark.parametrize("design", [_random, _pipeline])
def test_no_read_is_overwritten_and_none_waits_for_ever(design):
    d = design()
    rng = np.random.default_rng(3)
    assert not any(_lost(*d, 40, rng) for _ in range(8))


@pytest.mark.parametrize("mistake", [dict(slack=RING // 2), dict(room=False)])
def test_a_room_rule_that_is_too_generous_loses_words(mistake):
    d = _pipeline()
    rng = np.random.default_rng(4)
    assert any(_lost(*d, 40, rng, **mistake) for _ in range(40))
