"""The windows of a tile that share the finishing of it (wq_gemm_stream.hip): the steps of one workgroup at the tile's counter, run in every
order that several of them can take them in, with and without fellows that come late."""
import pytest

ARRIVED, ACCOUNTED = 1, 1 << 16


def resigned(w):
    return 0x100 << w


class Tile:
    """What is shared: the counter, which (window, part) partials have been written, which parts are finished and by whom."""

    def __init__(self, windows):
        self.windows, self.counter, self.written, self.finished, self.returned = windows, 0, set(), {}, 0

    def add(self, value):
        assert not self.returned, "the counter is touched after it was returned to zero"
        before, self.counter = self.counter, self.counter + value
        return before

    def all_in(self, v):
        return v & 0xFF == self.windows


def workgroup(tile, w, looks):
    """The steps of window w's workgroup; what lies between two yields is one access to memory.  `looks` at the counter, then it resigns."""
    everyone = range(tile.windows)
    tile.written |= {(w, part) for part in everyone if part != w}
    yield
    v = tile.add(ARRIVED) + ARRIVED
    left = v >> 8 & 0xFF if tile.all_in(v) else 0
    for _ in range(looks):
        if tile.all_in(v):
            break
        yield
        v = tile.add(0)
    parts = {w} | {p for p in everyone if left >> p & 1} if tile.all_in(v) else set()
    if not parts:
        yield
        tile.written.add((w, w))
        yield
        if tile.all_in(tile.add(resigned(w))):
            parts = {w}
        else:
            return
    yield
    if (tile.add(ACCOUNTED * len(parts)) + ACCOUNTED * len(parts)) >> 16 == tile.windows:
        yield
        tile.counter, tile.returned = 0, tile.returned + 1
    yield
    for part in parts:
        assert part not in tile.finished, "two workgroups finish a part"
        assert all((o, part) in tile.written for o in everyone if o != w), "a partial is read before it was written"
        tile.finished[part] = w


def run(order, windows, looks):
    """The workgroups' steps in `order` (indices into those that still have one); the number that had one at each step."""
    tile, choices = Tile(windows), []
    groups = [workgroup(tile, w, looks) for w in range(windows)]
    while groups:
        i = order[len(choices)] if len(choices) < len(order) else 0
        choices.append(len(groups))
        try:
            next(groups[i])
        except StopIteration:
            groups.pop(i)
    return tile, choices


@pytest.mark.parametrize("windows,looks", [(2, 0), (2, 1), (2, 2)])
def test_every_part_is_finished_once_in_every_order(windows, looks):
    order, runs = [], 0
    while order is not None:
        tile, choices = run(order, windows, looks)
        assert sorted(tile.finished) == list(range(windows)) and tile.counter == 0 and tile.returned == 1, order
        runs += 1
        order = (order + [0] * len(choices))[:len(choices)]
        while order and order[-1] + 1 >= choices[len(order) - 1]:
            order.pop()
        order = order[:-1] + [order[-1] + 1] if order else None
    assert runs > 20


@pytest.mark.parametrize("windows", [3, 5, 8])
def test_every_part_is_finished_once_in_random_orders(windows):
    import random

    rng, seen = random.Random(windows), set()
    for _ in range(4000):
        late = rng.random()
        order = [0 if rng.random() < late else rng.randrange(windows) for _ in range(40 * windows)]
        tile = Tile(windows)
        groups = [workgroup(tile, w, rng.choice((0, 2, 8))) for w in range(windows)]
        for i in order + [0] * 1000:
            if not groups:
                break
            try:
                next(groups[i % len(groups)])
            except StopIteration:
                groups.pop(i % len(groups))
        assert sorted(tile.finished) == list(range(windows)) and tile.counter == 0 and tile.returned == 1
        seen.add(len(set(tile.finished.values())))
    assert len(seen) > 1, "parts are finished by their own workgroups and by the last to arrive"
