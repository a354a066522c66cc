"""CPU model of how a traversal notes exact ties while its drained wave shares
work, and settles them afterwards (trace_persistent in csrc/rt_trace_dev.hpp),
checked against a plain search.

A ray meets its leaves in some order; lanes hold pieces of it, and an idle
lane takes a busy one's last piece.  The rules are the kernel's:

* a lane takes a leaf strictly closer than its best, which clears its tie, and
  notes a tie at an equal t once it has a best;
* a helper starts from its donor's best hit and tie;
* at hand-over the owner takes a closer hit with its tie; at an equal t it has
  a tie if the hits are different triangles or either side noted one;
* a ray that ends with a tie gets the first leaf at its closest t in the order
  of the caller's tree, one without keeps its best.

Leaves beyond a lane's or its owner's best may be left out at will: culling
drops boxes, and never one that holds a hit at the closest t."""
import math
import random

import pytest


class Lane:
    def __init__(self, segs, best_t=math.inf, best=None, tied=False):
        self.segs = [list(s) for s in segs if s]
        self.best_t, self.best, self.tied = best_t, best, tied
        self.helpers = 0

    def step(self, leaves, bound, rng):
        leaf = self.segs[0].pop(0)
        if not self.segs[0]:
            self.segs.pop(0)
        t = leaves[leaf]
        if t > min(self.best_t, bound) and rng.random() < 0.7:
            return                                  # culled
        if t < self.best_t:
            self.best_t, self.best, self.tied = t, leaf, False
        elif t == self.best_t and self.best is not None:
            self.tied = True


def hand_over(owner, helper, compare_hits=True):
    if helper.best is not None and helper.best_t < owner.best_t:
        owner.best_t, owner.best, owner.tied = helper.best_t, helper.best, helper.tied
    elif helper.best is not None and helper.best_t == owner.best_t:
        owner.tied = owner.tied or helper.tied or (compare_hits and helper.best != owner.best)


def trace(leaves, order, callers, rng, compare_hits=True):
    """Triangle reported for the ray, with random pieces and a random schedule."""
    cuts = sorted(rng.sample(range(1, len(order)), min(len(order) - 1, rng.randrange(6)))) if len(order) > 1 else []
    segs = [order[a:b] for a, b in zip([0] + cuts, cuts + [len(order)])]
    owner = Lane(segs)
    helpers = []
    while owner.segs or helpers:
        busy = [x for x in [owner] + helpers if x.segs]
        donors = [x for x in busy if len(x.segs) > 1]
        if donors and rng.random() < 0.3:
            d = rng.choice(donors)
            helpers.append(Lane([d.segs.pop()], d.best_t, d.best, d.tied))
            continue
        ended = [h for h in helpers if not h.segs]
        if ended and (not busy or rng.random() < 0.5):
            h = rng.choice(ended)
            helpers.remove(h)
            hand_over(owner, h, compare_hits)
            continue
        rng.choice(busy).step(leaves, owner.best_t, rng)
    if owner.tied:
        return next(k for k in callers if leaves[k] == owner.best_t)
    return owner.best


def runs(seed, count, **kw):
    rng = random.Random(seed)
    wrong = 0
    for _ in range(count):
        n = rng.randrange(1, 14)
        leaves = [float(rng.randrange(1, 4)) for _ in range(n)]
        order, callers = rng.sample(range(n), n), rng.sample(range(n), n)
        want = next(k for k in callers if leaves[k] == min(leaves))
        wrong += trace(leaves, order, callers, rng, **kw) != want
    return wrong


@pytest.mark.parametrize("seed", range(4))
def test_ties_are_noted_whatever_the_schedule(seed):
    assert runs(seed, 3000) == 0


def test_the_model_finds_a_missing_comparison():
    """Hand-overs that do not compare the two hits miss ties between lanes."""
    assert runs(0, 3000, compare_hits=False) > 0
