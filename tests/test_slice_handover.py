"""The hand-over of the shared finishing (splitk_exchange_sliced), step by step in every order: a workgroup arrives, waits or
gives up at any moment, marks its K tile, looks at the arrivals again, departs.  For every interleaving of up to four
workgroups each K tile's share is finished by exactly one of them, after all have arrived, and the tile's counter and mask are
left at zero.  (A model of the protocol: every step below is one atomic operation of the kernel.)"""
import pytest


def runs_of(tiles):
    """Explores all interleavings; returns the number of distinct end states reached and checks each of them."""
    # a workgroup: (step, verdict of its own share, shares taken over, departures it saw)
    start = (0, 0, 0, tuple(("arrive", False, 0, 0) for _ in range(tiles)), (0,) * tiles)
    seen, stack, ends = {start}, [start], set()
    while stack:
        arrived, departed, mask, groups, done = stack.pop()
        if all(g[0] == "left" for g in groups):
            assert done == (1,) * tiles, done
            assert (arrived, departed, mask) == (0, 0, 0)
            ends.add((arrived, departed, mask, done))
            continue
        for k, (step, mine, over, before) in enumerate(groups):
            everyone = all(g[0] != "arrive" for g in groups)
            for state in steps(tiles, k, step, mine, over, before, arrived, departed, mask, done, everyone):
                a, d, m, group, finished = state
                nxt = (a, d, m, groups[:k] + (group,) + groups[k + 1:], finished)
                if nxt not in seen:
                    seen.add(nxt)
                    stack.append(nxt)
    return len(ends), len(seen)


def steps(tiles, k, step, mine, over, before, arrived, departed, mask, done, everyone):
    bit = 1 << k
    if step == "arrive":  # fetch_add on the counter: the last one looks at the mask, the others wait
        last = arrived == tiles - 1
        yield arrived + 1, departed, mask, ("look" if last else "wait", last, 0, 0), done
    elif step == "look":  # load of the mask; an exchange follows if it was not empty
        yield arrived, departed, mask, ("take" if mask else "depart", True, 0, 0), done
    elif step == "take":  # exchange with zero: whoever marked and was not yet seen to is taken over
        yield arrived, departed, 0, ("depart", True, mask, 0), done
    elif step == "wait":  # load of the counter: everyone is there, or time is up
        if arrived == tiles:
            yield arrived, departed, mask, ("depart", True, 0, 0), done
        else:
            yield arrived, departed, mask, ("mark", False, 0, 0), done
    elif step == "mark":  # fetch_or of the own bit
        yield arrived, departed, mask | bit, ("again", False, 0, 0), done
    elif step == "again":  # load of the counter behind the mark
        yield arrived, departed, mask, ("unmark" if arrived == tiles else "depart", False, 0, 0), done
    elif step == "unmark":  # fetch_and: the returned bit says whether the share is still the workgroup's own
        yield arrived, departed, mask & ~bit, ("depart", bool(mask & bit), 0, 0), done
    elif step == "depart":  # fetch_add on the counter's upper half, ahead of the read-back
        yield arrived, departed + 1, mask, ("finish", mine, over, departed), done
    elif step == "finish":
        shares = (bit if mine else 0) | over
        assert everyone or not shares  # nobody reads partial sums that are not there (the counter may be cleared already)
        assert not shares & sum(1 << i for i, n in enumerate(done) if n), "a share is finished twice"
        finished = tuple(n + (shares >> i & 1) for i, n in enumerate(done))
        yield arrived, departed, mask, ("clear" if before == tiles - 1 else "left", mine, over, before), finished
    elif step == "clear":  # the last to depart leaves the counter at zero
        yield 0, 0, mask, ("left", mine, over, before), done


@pytest.mark.parametrize("tiles", [2, 3, 4])
def test_every_share_is_finished_once(tiles):
    ends, states = runs_of(tiles)
    assert ends == 1 and states > 10 * tiles
