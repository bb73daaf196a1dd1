"""The work split of the ragged launch (paged_prefill.hip), in Python: the units, tiles and shares
that its workers and its merge compute must cover every 64-key chunk of every tile exactly once and
agree on the partials, whatever the batch."""

import random

import numpy as np
import pytest

ROWS, CHUNK, MIN_CHUNKS, SNAP = 128, 64, 2, 2


class DivG:
    def __init__(self, G):
        self.G, self.inv = G, np.float32(1) / np.float32(G)

    def div(self, x):
        q = int(np.float32(x) * self.inv)
        r = x - q * self.G
        return q - 1 if r < 0 else q + 1 if r >= self.G else q

    def floors(self, x):
        q = self.div(x)
        return self.G * (q * (q - 1) // 2) + q * (x - q * self.G)

    def every_other(self, a, n):
        all_ = self.floors(a + 2 * n) - self.floors(a)
        r = a + 1 - self.div(a + 1) * self.G
        miss = 0 if r == 0 else self.G - r
        hits = 0
        if self.G & 1:
            t0 = (miss + self.G) // 2 if miss & 1 else miss // 2
            hits = self.div(n - 1 - t0) + 1 if t0 < n else 0
        elif not miss & 1:
            t0 = miss // 2
            hits = self.div(2 * (n - 1 - t0)) + 1 if t0 < n else 0
        return (all_ - hits) // 2


class Seq:
    """ragged_seq: one sequence's tiles and their chunks."""

    def __init__(self, qlen, ctx, g, max_q, max_ctx):
        bad = qlen > 0 and (ctx < qlen or ctx > max_ctx)
        none = qlen <= 0 or bad
        self.g, self.rows = g, 0 if none else min(qlen, max_q) * g.G
        self.tiles = -(-self.rows // ROWS)
        c0 = 0 if none else ctx - qlen
        self.a = (g.G * (c0 + CHUNK) + ROWS - 1) // CHUNK
        self.last = 0 if none else (c0 + min(qlen, max_q) - 1 + CHUNK) // CHUNK
        self.units = 0 if none else self.before(self.tiles - 1) + self.last
        self.c0 = c0

    def before(self, t):
        return self.g.every_other(self.a, t) if t > 0 else 0

    def chunks(self, t):
        return self.g.div(self.a + 2 * t) if t + 1 < self.tiles else self.last

    def plain(self, t):
        """chunks(t) from the rows: the last row of tile t sees c0 + its query + 1 keys."""
        last = min(ROWS * (t + 1), self.rows) - 1
        return -(-(self.c0 + last // self.g.G + 1) // CHUNK)

    def find(self, u):
        """The tile of unit u: 64 candidates a step, as a wave looks for it."""
        tile, step = 0, (self.tiles + 63) // 64
        while True:
            at = [t for t in range(tile, tile + 64 * step, step)
                  if t < self.tiles and self.before(t) <= u]
            tile += (len(at) - 1) * step
            if step == 1:
                return tile
            step = 1


def split(lens, G, KVH, max_q, max_ctx, grid):
    """Every worker's pieces, as (worker, sequence, KV head, tile, first chunk, end), and the merges
    {(sequence, KV head, tile): (worker that begins it, pieces)}."""
    g = DivG(G)
    seqs = [Seq(q, c, g, max_q, max_ctx) for q, c in lens]
    C = KVH * sum(s.units for s in seqs)
    W = min((C + MIN_CHUNKS - 1) // MIN_CHUNKS, grid)
    pieces, merges = [], {}
    for w in range(W):
        share, extra = C // W, C % W
        U = w * share + w * extra // W
        left = (w + 1) * share + (w + 1) * extra // W - U
        b, base = 0, 0
        while base + KVH * seqs[b].units <= U:
            base += KVH * seqs[b].units
            b += 1
        kvh, u = divmod(U - base, seqs[b].units)
        at = [b, kvh, seqs[b].find(u)]
        c0 = u - seqs[b].before(at[2])

        def step():
            nonlocal base
            at[2] += 1
            if at[2] < seqs[at[0]].tiles:
                return True
            at[2] = 0
            at[1] += 1
            if at[1] < KVH:
                return True
            at[1] = 0
            base += KVH * seqs[at[0]].units
            at[0] += 1
            while at[0] < len(seqs) and not seqs[at[0]].units:
                at[0] += 1
            return at[0] < len(seqs)

        work = True
        if c0 <= SNAP:
            left, c0 = left + c0, 0
        elif seqs[b].chunks(at[2]) - c0 <= SNAP:
            left -= seqs[b].chunks(at[2]) - c0
            work, c0 = left > 0 and step(), 0
        while work:
            s = seqs[at[0]]
            n = s.chunks(at[2])
            c1 = min(n, c0 + left)
            if c1 < n:
                if c1 <= SNAP:
                    break
                if n - c1 <= SNAP:
                    c1 = n
            pieces.append((w, *at, c0, c1))
            if c0 == 0 and c1 < n:
                end = base + at[1] * s.units + s.before(at[2]) + n
                assert tuple(at) not in merges
                merges[tuple(at)] = (w, ((end - SNAP) * W - 1) // C - w + 1)
            left -= c1 - c0
            work, c0 = left > 0 and step(), 0
    return seqs, pieces, merges


def check(lens, G, KVH, max_q, max_ctx, grid):
    seqs, pieces, merges = split(lens, G, KVH, max_q, max_ctx, grid)
    tiles, slots = {}, set()
    for w, b, kvh, t, c0, c1 in pieces:
        tiles.setdefault((b, kvh, t), []).append((c0, c1, w))
        if not (c0 == 0 and c1 == seqs[b].chunks(t)):
            slot = 2 * w + (c0 == 0)      # a worker continues one tile and begins one at most
            assert slot not in slots
            slots.add(slot)
    assert len(tiles) == KVH * sum(s.tiles for s in seqs)
    for (b, kvh, t), got in tiles.items():
        n = seqs[b].chunks(t)
        assert n == seqs[b].plain(t) and t < seqs[b].tiles
        got.sort()
        assert [c for c, _, _ in got] + [n] == [0] + [e for _, e, _ in got], "a chunk lost or twice"
        if len(got) > 1:
            w, count = merges.pop((b, kvh, t))
            assert [x for _, _, x in got] == list(range(w, w + count))
    assert not merges


@pytest.mark.parametrize("seed", range(20))
def test_every_chunk_once(seed):
    r = random.Random(seed)
    for _ in range(12):
        G, KVH, n = r.randint(1, 20), r.randint(1, 8), r.randint(1, 80)
        lens = []
        for _ in range(n):
            q = r.choice([0, 1, 1, 1, r.randint(1, 20), r.randint(1, 700)])
            lens.append((q, q + r.choice([0, r.randint(0, 100), r.randint(0, 4000)])))
        if r.random() < 0.3:
            lens[r.randrange(n)] = (5, 3)                       # bad: no work
        lens[0] = (1, 1 + r.randint(0, 500))
        check(lens, G, KVH, max(q for q, _ in lens), max(c for _, c in lens),
              r.choice([1, 2, 7, 64, 256, 768, 1024]))


@pytest.mark.parametrize("q,G", [(1300, 7), (8000, 7), (4096, 128), (5000, 3), (8191, 1)])
@pytest.mark.parametrize("grid", [1, 256, 512, 768])
def test_sequences_of_more_than_64_tiles(q, G, grid):
    """The tile search's coarse step."""
    check([(1, 100)] * 3 + [(q, q + 77), (1, 3000)], G, 2, q, max(q + 77, 3000), grid)


def test_division_is_exact_below_2_24():
    r = random.Random(5)
    for G in list(range(1, 70)) + [100, 127, 128, 1000]:
        d = DivG(G)
        xs = [r.randrange(1 << 24) for _ in range(200)] + [0, G - 1, G, (1 << 24) - 1]
        xs += [k * G + e for k in (r.randrange((1 << 24) // G) for _ in range(50)) for e in (-1, 0)
               if k * G + e >= 0]
        assert all(d.div(x) == x // G for x in xs)
        for _ in range(20):
            a, n = r.randrange(1, 5000), r.randrange(1, 300)
            assert d.every_other(a, n) == sum((a + 2 * t) // G for t in range(n))
