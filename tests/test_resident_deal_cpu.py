"""The deals of the kernel with resident tables (run() in turbodeberta_amd/csrc/attn_resident.hip), restated step by step: whatever the
lengths, the grid and the heads, every unit of query rows has to go to exactly one workgroup."""
import math

import numpy as np
import pytest

WAVES, HALF, BN = 8, 4, 64
COST = {1: (6, 4), 2: (9, 6)}                   # a step of a whole tile and of half of one, by query groups per unit


def groups_of(wgs, heads):
    n = math.gcd(wgs, heads)
    return wgs // n, heads // n                 # workgroups and heads of a group


class Ragged:
    """Sequences of different lengths, up to 64 of them."""

    def __init__(self, lens, heads, per_group, QG):
        self.lens = sorted(lens, reverse=True)  # (ties by index: the order of equals does not matter here)
        self.n = self.lens + [0] * (64 - len(lens))
        self.heads, self.per_group, self.QG, self.UQ = heads, per_group, QG, 16 * QG
        units = [-(-n // self.UQ) for n in self.n]
        self.units = units
        self.upto = np.cumsum([(u // WAVES + (u % WAVES > HALF)) * heads for u in units]), np.cumsum([(0 < u % WAVES <= HALF) * heads for u in units])
        self.wholes = int(self.upto[0][63])
        self.all = self.wholes + int(self.upto[1][63])
        self.rest = self.all % per_group
        self.full = self.all - self.rest
        self.rounds = self.full // per_group
        longest, shortest = self.lens[0], self.lens[-1]
        far_apart = longest > 8 * BN and 2 * shortest < longest and 8 * self.rest < 7 * per_group
        self.reckon = longest > 5 * BN and self.rest > 0 and per_group <= 64 and 0 < self.rounds <= (5 if far_apart else 2)
        self.halved = max(self.wholes - self.full, 0)
        if self.rest + self.halved > per_group:
            self.halved = per_group - self.rest
            if self.reckon:
                first, second = (self.n[self.before(self.full + i)] for i in (0, self.halved))
                if 10 * second > 9 * first:
                    self.halved = 0
            elif self.rounds > 0:
                self.halved = 0

    def before(self, k):
        whole = k < self.wholes
        at, among = 0, k if whole else k - self.wholes
        for step in (32, 16, 8, 4, 2, 1):
            if self.upto[0 if whole else 1][at + step - 1] <= among:
                at += step
        return at

    def last_tile(self, i):
        return self.full + (i >> 1 if i < 2 * self.halved else i - self.halved)

    def cost(self, n, half):
        return (-(-n // BN) + 1) * COST[self.QG][half]

    def tile(self, j, workgroup):
        return j * self.per_group + (self.per_group - 1 - workgroup if j & 1 else workgroup)

    def last_piece(self, mine):
        """Which piece of the last round a workgroup takes."""
        if not self.reckon:
            return self.per_group - 1 - mine if self.rounds & 1 else mine
        load = [sum(self.cost(self.n[self.before(self.tile(j, g))], self.tile(j, g) >= self.wholes) for j in range(self.rounds)) for g in range(self.per_group)]
        last = sum(a < load[mine] or (a == load[mine] and g < mine) for g, a in enumerate(load))
        if self.halved > 0:
            tiles = [self.last_tile(i) for i in range(64)]
            key = [self.cost(self.n[self.before(k)], i < 2 * self.halved or k >= self.wholes) * 64 + 63 - i if k < self.all else -1 for i, k in enumerate(tiles)]
            rank = [(0 if k < self.all else 64) + sum(other > key[i] for other in key) for i, k in enumerate(tiles)]
            last = rank.index(last) if last in rank else self.per_group
        return last

    def units_of(self, mine):
        """(head, sequence, unit) of a workgroup, tile by tile."""
        last = self.last_piece(mine)
        for j in range(self.rounds + 1):
            k = self.tile(j, mine) if j < self.rounds else self.last_tile(last)
            if k >= self.all:
                return
            at = self.before(k)
            units = self.units[at]
            end, per_head = units % WAVES, units // WAVES + (units % WAVES > HALF)
            if k < self.wholes:
                head, tile = divmod(k - (int(self.upto[0][at]) - per_head * self.heads), max(per_head, 1))
                first = WAVES * tile
            else:
                head, first = k - self.wholes - (int(self.upto[1][at]) - self.heads), units - end
            stop = first + WAVES
            if j == self.rounds and last < 2 * self.halved:
                first, stop = (first + HALF, stop) if last & 1 else (first, stop - HALF)
            assert 0 <= head < self.heads and first >= 0
            yield [(head, at, u) for u in range(first, min(stop, units))]


def equal_units_of(L, seqs, per_group, UQ, mine):
    """(sequence and head, unit) of a workgroup where all sequences have one length."""
    per_head = -(-L // (UQ * HALF))
    pairs, every = (per_head + 1) // 2, seqs * per_head
    begin, end = every * mine // per_group, every * (mine + 1) // per_group
    if every > per_group and seqs * pairs <= per_group:
        begin = mine // pairs * per_head + 2 * (mine % pairs)
        end = min(begin + 2, (mine // pairs + 1) * per_head) if mine < seqs * pairs else begin
    following = (begin // per_head + 1) * per_head
    pairs0 = (min(following, end) - begin + 1) >> 1
    j = 0
    while True:
        more = max(j - pairs0, 0) // pairs
        k = begin + 2 * j if j < pairs0 else following + more * per_head + 2 * (j - pairs0 - more * pairs)
        if k >= end:
            return
        seq, first = k // per_head, HALF * (k % per_head)
        yield [(seq, u) for u in range(first, min(first + HALF * min(2, end - k), -(-L // UQ)))]
        j += 1


RS = np.random.RandomState(0)
BATCHES = {
    "benchmark": RS.randint(16, 513, 64), "padded": RS.randint(384, 513, 32), "equal": [512] * 48, "long": RS.randint(1024, 4097, 8), "far_apart": np.linspace(450, 1800, 19).astype(int),
    "one": [700], "empty_ones": [0, 300, 0, 1, 900], "nothing": [0, 0], "wholes_by_halves": [1100] * 7, "longest_by_halves": [2000, 1732, 1464, 1196, 928, 660],
    "ends": [289] * 50, "one_token": [1] * 64, "few": [330, 340], "three": [1600, 900, 400],
} | {f"drawn{i}": RS.randint(0, RS.choice([200, 520, 2100, 4097]), RS.randint(1, 65)) for i in range(20)}


@pytest.mark.parametrize("wgs,heads", [(256, 12), (256, 16), (256, 1), (256, 24), (256, 8), (256, 5), (256, 64), (8, 12), (40, 12), (248, 16), (304, 12)])
@pytest.mark.parametrize("QG", [1, 2])
def test_every_unit_goes_to_one_workgroup(wgs, heads, QG):
    per_group, of_group = groups_of(wgs, heads)
    for name, lens in BATCHES.items():
        deal = Ragged([int(n) for n in lens], of_group, per_group, QG)
        got = sorted(u for g in range(per_group) for tile in deal.units_of(g) for u in tile)
        want = sorted((h, s, u) for h in range(of_group) for s in range(64) for u in range(deal.units[s]))
        assert got == want, name


@pytest.mark.parametrize("wgs,heads", [(256, 12), (256, 16), (256, 1), (256, 24), (256, 64), (8, 12), (40, 12)])
@pytest.mark.parametrize("UQ", [16, 32])
def test_every_unit_of_equal_sequences_goes_to_one_workgroup(wgs, heads, UQ):
    per_group, of_group = groups_of(wgs, heads)
    for B, L in [(1, 161), (1, 512), (8, 513), (16, 257), (33, 289), (70, 500), (3, 1537), (4, 4096), (2, 385), (1, 1), (64, 64)] + [(int(RS.randint(1, 40)), int(RS.randint(1, 1200))) for _ in range(12)]:
        seqs = of_group * B
        got = sorted(u for g in range(per_group) for tile in equal_units_of(L, seqs, per_group, UQ, g) for u in tile)
        assert got == [(s, u) for s in range(seqs) for u in range(-(-L // UQ))], (B, L)
