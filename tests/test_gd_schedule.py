"""A model of how gate_up_down's single kernel (k_gd) orders its units, on the CPU: two launches share an XCD's slots, each
XCD starts each launch's workgroups in order, and every interleaving of their steps is walked.

The kernel's rules, as the model states them. Units are numbered gate_up first (row-major), then down (row-major), and
dealt to the XCDs in turn: unit g to XCD g mod X (one list), or row i's all to XCD i mod X (a list an XCD). A gate_up unit
waits for nothing: it adds one to its row's word; the unit whose addition is the row's last forms h and adds one more,
and runs the blocks that the word it read names as left. A down unit polls its row's word for that last count. In one list
it may give its slot back instead while the row's gate_up units are not all counted (once they are, the unit that forms h
runs and waits for nothing): it sets its block's bit in the word and leaves, unless the value it read shows h ready.
Each block's unit then counts; the row's last one clears the word.

What holds in every order: every launch ends (no state without a next step but the end), each block is run once, and
the words are zero. One list without the leaving -- a wait that only ends when other units have run -- does not hold it:
two launches whose down units fill each other's XCDs wait for ever.
"""
import pytest

GU, H, LEFT, DN, RUN = range(5)          # a running unit's next step


class Model:
    def __init__(self, xcds, slots, launches, rows, ugu, nblk, one_list, leaves):
        self.X, self.slots, self.L, self.R, self.ugu, self.nblk = xcds, slots, launches, rows, ugu, nblk
        self.leaves = leaves
        gate = [("g", i, u) for i in range(rows) for u in range(ugu)]
        down = [("d", i, b) for i in range(rows) for b in range(nblk)]
        self.lists = []                  # per XCD: its units of one launch, in start order
        for x in range(xcds):
            if one_list:
                self.lists.append([u for n, u in enumerate(gate + down) if n % xcds == x])
            else:
                self.lists.append([u for u in gate if u[1] % xcds == x] + [u for u in down if u[1] % xcds == x])

    def start(self):
        # (next unit of each (launch, XCD), the running units, per (launch, row): (count, left bits, done), blocks run)
        return (((0,) * (self.L * self.X)), (), ((0, 0, 0),) * (self.L * self.R),
                (0,) * (self.L * self.R * self.nblk))

    def final(self, s):
        return not s[1] and all(n == len(self.lists[k % self.X]) for k, n in enumerate(s[0]))

    def steps(self, s):
        nxt, run, words, ran = s
        used = [0] * self.X
        for r in run:
            used[r[1]] += 1
        for k, n in enumerate(nxt):
            la, x = divmod(k, self.X)
            if used[x] < self.slots and n < len(self.lists[x]):
                kind, i, u = self.lists[x][n]
                unit = (la, x, i, GU if kind == "g" else DN, u, 0)
                yield self._set(s, nxt=nxt[:k] + (n + 1,) + nxt[k + 1:], run=self._add(run, unit))
        for j in sorted(set(run)):
            yield from self._advance(s, j)

    @staticmethod
    def _add(run, unit):
        return tuple(sorted(run + (unit,)))

    @staticmethod
    def _drop(run, unit):
        k = run.index(unit)
        return run[:k] + run[k + 1:]

    @staticmethod
    def _set(s, nxt=None, run=None, words=None, ran=None):
        return (s[0] if nxt is None else nxt, s[1] if run is None else run, s[2] if words is None else words,
                s[3] if ran is None else ran)

    def _word(self, words, la, i, w):
        k = la * self.R + i
        return words[:k] + (w,) + words[k + 1:]

    def _run_block(self, s, la, i, b):
        """Block b of row i run and counted; the row's last count clears the word."""
        cnt, left, done = s[2][la * self.R + i]
        k = (la * self.R + i) * self.nblk + b
        ran = s[3][:k] + (s[3][k] + 1,) + s[3][k + 1:]
        w = (0, 0, 0) if done + 1 == self.nblk else (cnt, left, done + 1)
        return self._set(s, words=self._word(s[2], la, i, w), ran=ran)

    def _advance(self, s, unit):
        la, x, i, pc, u, mask = unit
        run = self._drop(s[1], unit)
        cnt, left, done = s[2][la * self.R + i]
        want = self.ugu + 1
        if pc == GU:
            t = self._set(s, words=self._word(s[2], la, i, (cnt + 1, left, done)))
            yield self._set(t, run=self._add(run, (la, x, i, H, u, 0)) if cnt == self.ugu - 1 else run)
        elif pc == H:                    # h is stored; its count returns the bits set before it
            t = self._set(s, words=self._word(s[2], la, i, (cnt + 1, left, done)))
            yield self._set(t, run=self._add(run, (la, x, i, LEFT, u, left)) if left else run)
        elif pc == LEFT:
            b = (mask & -mask).bit_length() - 1
            t = self._run_block(s, la, i, b)
            mask &= mask - 1
            yield self._set(t, run=self._add(run, (la, x, i, LEFT, u, mask)) if mask else run)
        elif pc == DN:
            if cnt >= want:
                yield self._set(s, run=self._add(run, (la, x, i, RUN, u, 0)))
            # the polls are spent: the unit leaves while gate_up units of the row are missing in the value it read last --
            # which may be an older one than the word now ("late"), or not ("early")
            if self.leaves == "late" or (self.leaves == "early" and cnt < self.ugu):
                t = self._set(s, words=self._word(s[2], la, i, (cnt, left | 1 << u, done)))
                yield self._set(t, run=self._add(run, (la, x, i, RUN, u, 0)) if cnt >= want else run)
        else:
            yield self._set(self._run_block(s, la, i, u), run=run)


def walk(m, limit=2_000_000):
    """Every reachable state once: (the states with no next step that are not the end, the ends)."""
    first = m.start()
    seen, todo, stuck, ends = {first}, [first], [], []
    while todo:
        s = todo.pop()
        n = 0
        for t in m.steps(s):
            n += 1
            if t not in seen:
                seen.add(t)
                todo.append(t)
        if n == 0:
            (ends if m.final(s) else stuck).append(s)
        assert len(seen) < limit
    return stuck, ends


def _holds(m):
    stuck, ends = walk(m)
    assert not stuck, f"{len(stuck)} states end with units waiting, such as {stuck[0]}"
    assert ends
    for s in ends:
        assert all(w == (0, 0, 0) for w in s[2]) and all(n == 1 for n in s[3])


@pytest.mark.parametrize("one_list,leaves", [(True, "late"), (True, "early"), (False, "")])
@pytest.mark.parametrize("launches,rows,ugu,nblk,slots", [(2, 2, 1, 2, 1), (2, 2, 2, 2, 1), (2, 3, 1, 1, 2), (1, 2, 2, 3, 3)])
def test_every_order_of_starts_ends_with_each_block_run_once(one_list, leaves, launches, rows, ugu, nblk, slots):
    _holds(Model(2, slots, launches, rows, ugu, nblk, one_list, leaves))


def test_a_wait_that_holds_its_slot_across_the_xcds_does_not_end():
    """The rule that the model is there to refuse: one list, and a down unit that only waits."""
    stuck, _ = walk(Model(2, 1, 2, 2, 1, 2, one_list=True, leaves=""))
    assert stuck
    _holds(Model(2, 1, 1, 2, 1, 2, one_list=True, leaves=""))    # a launch alone ends
