"""CPU transcription of the index arithmetic of the multi-position row products on the matrix cores
(lastro-rust_amd/csrc/prefill.hip: XGeo, xg_load, xg_steps, xg_run; dev_rows.h: member_tile) and of the attention's
lane-to-position maps (attn_mm.hip). For every weight type and row length the kernels are built for: each chunk of a row
is taken once, by the chain of its decode lane and in that chain's order; the LDS nodes are in bounds, each written once
(the zeros of runs without a chunk included) before it is read; the sums form the decode kernels' pairwise tree. For the
members of the experts: every member is in one tile, and the launched tiles are enough for every routing."""
import os
import re

import numpy as np
import pytest

CHUNK = {"f32": 4, "q8_0": 16, "q4_0": 32}  # elements per 16-byte payload chunk (Fmt<DT>::kElems)
SOURCE = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lastro-rust_amd", "csrc",
                           "prefill.hip")).read()


class XGeo:
    """Geo<DT, K> and XGeo<DT, K>."""

    def __init__(self, dt, K):
        self.CE = CHUNK[dt]
        self.NCH = K // self.CE
        self.LPR = next((n for n in (1, 2, 4, 8, 16, 32) if self.NCH <= n), 64)
        self.NJ = -(-self.NCH // self.LPR)
        self.SE = min(self.CE, 16)
        self.HPC = self.CE // self.SE
        self.NG = self.LPR // 4
        self.KW = min(self.NG, 4)
        self.SUB = 2 if self.NG >= 2 * self.KW and self.even(2) else 1
        assert self.even(self.SUB)
        self.ROUNDS = self.NG // (self.KW * self.SUB)
        self.NN = self.NG // self.SUB
        assert self.ROUNDS * self.KW * self.SUB == self.NG  # no group is left out

    def even(self, sub):
        for r in range(self.NG // (self.KW * sub)):
            for jj in range(self.NJ):
                lo, hi = (4 * (r + i) * self.KW * sub + self.LPR * jj for i in (0, 1))
                if lo < self.NCH < hi:
                    return False
        return True

    def valid(self, r, jj):
        return 4 * r * self.KW * self.SUB + self.LPR * jj < self.NCH

    def steps(self):
        return [(r, u, jj, h) for r in range(self.ROUNDS) for u in range(self.SUB) for jj in range(self.NJ)
                for h in range(self.HPC) if self.valid(r, jj)]


GEOMETRIES = [(dt, K) for dt in CHUNK for K in (128, 256, 512, 1024, 1536)]


@pytest.mark.parametrize("dt,K", GEOMETRIES)
def test_every_chunk_is_taken_once_in_its_chain(dt, K):
    x = XGeo(dt, K)
    elements = {}  # (chain) -> its elements in the order of the MFMAs
    for w in range(x.KW):
        for r, u, jj, h in x.steps():
            for gq in range(4):
                chain = 4 * ((r * x.KW + w) * x.SUB + u) + gq
                j = chain + x.LPR * jj
                assert j < x.NCH  # the loads of the row and of the activations stay inside it
                elements.setdefault(chain, []).extend(range(j * x.CE + h * x.SE, j * x.CE + (h + 1) * x.SE))
    want = {c: [e for j in range(c, x.NCH, x.LPR) for e in range(j * x.CE, (j + 1) * x.CE)] for c in range(x.LPR)}
    assert elements == {c: e for c, e in want.items() if e}  # decode lane c: its chunks, element by element
    # the accumulator of a group starts with its first step and its node is formed with its last
    s = x.steps()
    for i, (r, u, jj, h) in enumerate(s):
        first = jj == 0 and h == 0
        last = i + 1 == len(s) or (s[i + 1][0], s[i + 1][1]) != (r, u)
        assert first == (i == 0 or (s[i - 1][0], s[i - 1][1]) != (r, u))
        assert last == (i + 1 == len(s) or (s[i + 1][2] == 0 and s[i + 1][3] == 0))


@pytest.mark.parametrize("MT,NT", [(2, 1), (2, 2)])
@pytest.mark.parametrize("dt,K", GEOMETRIES)
def test_nodes_form_the_pairwise_tree(dt, K, MT, NT):
    x = XGeo(dt, K)
    lds = x.NN * MT * NT * 256  # xg_lds
    assert lds * 4 <= 160 * 1024
    nodes = [None] * lds
    chains_used = min(x.NCH, x.LPR)

    def put(i, v):
        assert nodes[i] is None
        nodes[i] = v

    lane = 5  # the node of a lane holds its own column: one lane stands for all, the offsets are lane-free
    for w in range(x.KW):
        s = x.steps()
        pend = {}
        for i, (r, u, jj, h) in enumerate(s):
            if i + 1 == len(s) or (s[i + 1][0], s[i + 1][1]) != (r, u):
                c0 = 4 * ((r * x.KW + w) * x.SUB + u)
                f = ((c0, c0 + 1), (c0 + 2, c0 + 3))
                pend[r] = f if u == 0 else (pend[r], f)
                if u == x.SUB - 1:
                    for t in range(MT):
                        for n in range(NT):
                            for q in range(4):
                                put((((r * x.KW + w) * MT + t) * NT + n) * 256 + 64 * q + lane, (pend[r], t, n, q))
        if not x.valid(x.ROUNDS - 1, 0):
            for r in range(x.ROUNDS):
                if not x.valid(r, 0):
                    for t in range(MT * NT * 4):
                        put((r * x.KW + w) * MT * NT * 256 + 64 * t + lane, "zero")

    def tree(i, n, stride):
        return nodes[i] if n == 1 else (tree(i, n // 2, stride), tree(i + n // 2 * stride, n // 2, stride))

    def chains(v):
        """The chains under a tree of nodes, with the outputs they belong to; zeros have none."""
        if v == "zero":
            return None, None
        if len(v) == 4:
            return v[0], {v[1:]}
        (a, oa), (b, ob) = chains(v[0]), chains(v[1])
        if b is None:
            return a, oa  # a + 0
        return (a, b), oa | ob

    def balanced(lo, n):
        if lo >= chains_used:
            return None  # lanes without a chunk: zeros
        if n == 1:
            return lo
        a, b = balanced(lo, n // 2), balanced(lo + n // 2, n // 2)
        return a if b is None else (a, b)

    seen = set()
    assert NT * 4 % x.KW == 0
    for w in range(x.KW):
        for e in range(NT * 4 // x.KW):
            it = w * (NT * 4 // x.KW) + e
            for t in range(MT):
                got, outs = chains(tree(t * NT * 256 + it * 64 + lane, x.NN, MT * NT * 256))
                assert outs == {(t, it >> 2, it & 3)}  # tile row t, position tile, quad of rows
                seen |= outs
                assert got == balanced(0, 1 << (chains_used - 1).bit_length())
    assert len(seen) == MT * NT * 4


@pytest.mark.parametrize("heads,kvh,hidden", [(4, 2, 256), (16, 8, 1024), (24, 8, 1536)])
def test_rows_and_positions_of_the_grids(heads, kvh, hidden):
    """k_qkv_x: rows (j, j + 32) of a head; k_oproj_x: 32 rows; positions 16 NT to a workgroup, the last one clamped."""
    rows = (heads + 2 * kvh) * 64
    q = np.zeros(rows, int)
    for bx in range(rows // 32):
        for i in range(16):
            r = (bx >> 1) * 64 + 16 * (bx & 1) + i
            q[[r, r + 32]] += 1
    assert (q == 1).all()
    o = np.zeros(hidden, int)
    for bx in range(hidden // 32):
        for lane_g in range(4):
            for r in range(4):
                o[[32 * bx + 4 * lane_g + r, 32 * bx + 4 * lane_g + r + 16]] += 1
    assert (o == 1).all()
    for nv in (1, 15, 16, 17, 33, 500, 512):
        for NT in (1, 2):
            p = np.zeros(nv, int)
            for by in range(-(-nv // (16 * NT))):
                for n in range(NT):
                    for i in range(16):
                        pos = by * 16 * NT + 16 * n + i
                        assert min(pos, nv - 1) >= 0
                        if pos < nv:
                            p[pos] += 1
            assert (p == 1).all()


def member_tile(cnt, NP, tile):
    """member_tile<NP> of dev_rows.h: (expert, first member, members) or None."""
    t = (cnt + NP - 1) // NP
    end = np.cumsum(t)
    hit = np.flatnonzero((tile >= end - t) & (tile < end))
    if not len(hit):
        return None
    e = int(hit[0])
    return e, (tile - (end[e] - t[e])) * NP, int(cnt[e])


def routings(nv, k, E, rng):
    yield np.stack([rng.choice(E, k, replace=False) for _ in range(nv)])            # spread
    yield np.tile(np.arange(k), (nv, 1))                                             # all to the same experts
    p = 1.0 / np.arange(1, E + 1) ** 1.1
    yield np.stack([rng.choice(E, k, replace=False, p=p / p.sum()) for _ in range(nv)])
    yield (np.arange(nv)[:, None] * k + np.arange(k)) % E                            # as even as can be


@pytest.mark.parametrize("E,k", [(4, 2), (8, 2), (32, 8), (40, 8), (64, 8), (64, 1)])
def test_every_member_is_in_one_launched_tile(E, k):
    rng = np.random.default_rng(E + k)
    for nv in (1, 2, 15, 16, 17, 33, 70, 300, 512):
        slots = nv * k
        for ids in routings(nv, k, E, rng):
            cnt = np.bincount(ids.ravel(), minlength=64)
            assert cnt.max() <= nv  # list[e * cap + c], c < cap: an expert has a position once
            for NP in (16, 32):
                tiles = slots // NP + min(slots, E)  # launch_layer_b, launch_grp_experts
                seen = np.zeros((64, nv), int)
                for tile in range(tiles):
                    m = member_tile(cnt, NP, tile)
                    if m is None:
                        continue
                    e, first, members = m
                    assert first < members
                    for c in range(NP):
                        assert min(first + c, members - 1) < members
                        if first + c < members:
                            seen[e, first + c] += 1
                assert all((seen[e, :cnt[e]] == 1).all() and (seen[e, cnt[e]:] == 0).all() for e in range(64))


def test_entries_of_the_grouped_lists():
    """k_grp_plan's list entries: slot << 16 | position for passes of up to 512 positions, 256 slots to a step."""
    for sb, pl, off in ((0, 0, 0), (15, 31, 255), (3, 7, 200)):
        slot, pos = sb * 32 * 8 + off, sb * 32 + pl
        entry = slot << 16 | pos
        assert entry < 1 << 31 and entry >> 16 == slot and entry & 0xffff == pos


def test_attention_lanes_and_positions():
    """k_attn_mm: lane (group gq, index i) loads the K row of position 16 gq + 4 (i & 3) + (i >> 2) of the tile as row i
    of block gq. Element 4 b + r of a lane of group G (row 4 G + r of block b) is then position 16 b + 4 r + G, the
    operand k = G of the p.v product over positions 4 (4 b + r) .. +3; the V rows e of a lane are positions 4 e + gq."""
    row = {(gq, i): 16 * gq + 4 * (i & 3) + (i >> 2) for gq in range(4) for i in range(16)}
    assert sorted(row.values()) == list(range(64))
    for G in range(4):
        for b in range(4):
            for r in range(4):
                pos = row[(b, 4 * G + r)]
                assert pos == 16 * b + 4 * r + G
                assert pos // 4 == 4 * b + r and pos % 4 == G
                v = 4 * b + r  # element v = 4 b + r, valid rows of it: 4 v < nv - G
                for nv in range(65):
                    assert (4 * v < nv - G) == (pos < nv)
        assert sorted(4 * e + G for e in range(16)) == [p for p in range(64) if p % 4 == G]


def test_the_transcribed_names_are_the_kernels():
    for text in ("SE = G::CE < 16 ? G::CE : 16", "KW = NG < 4 ? NG : 4", "SUB = NG >= 2 * KW && even(2) ? 2 : 1",
                 "const int slots = nv * d.top_k, tiles = slots / (two ? 32 : 16) + std::min(slots, d.experts);",
                 "const int j = 4 * ((st.r * X::KW + w) * X::SUB + st.u) + gq + G::LPR * st.jj;"):
        assert text in SOURCE, text
    assert not re.search(r"xslot|stage_group", SOURCE)  # those are few.hip's


def test_one_or_two_position_tiles():
    """two_tiles: by the workgroups on the fullest of the device's compute units (not a fixed number of them). At the
    measured points of 256 units (us, one / two tiles) it is never more than 3% from the faster one."""
    body = re.search(r"static bool two_tiles\(int row_groups, int nv, int cus\) \{(.*?)\n\}", SOURCE, re.S)[1]
    assert "256" not in body and body.count(", cus)") == 2 and "return 17 * c2 < 10 * c1;" in body

    def two(groups, nv, cus=256):
        c1, c2 = (-(-groups * -(-nv // n) // cus) for n in (16, 32))
        return 17 * c2 < 10 * c1

    times = {(80, 48): (10.5, 14.2), (80, 64): (15.8, 14.2), (80, 128): (21.5, 23.2), (80, 192): (27.4, 23.9),
             (80, 256): (33.2, 32.6), (80, 512): (60.6, 52.1), (48, 64): (9.8, 13.0), (48, 128): (15.3, 12.9),
             (48, 256): (21.2, 22.1), (48, 512): (38.4, 32.6), (64, 64): (7.8, 10.9), (64, 128): (11.1, 10.6),
             (64, 192): (15.5, 17.4), (64, 256): (19.6, 18.0), (64, 384): (27.4, 25.9), (64, 512): (35.0, 31.7),
             (32, 128): (7.4, 9.7), (32, 192): (11.0, 9.9), (32, 256): (11.1, 10.0), (32, 384): (15.2, 17.0),
             (32, 512): (19.2, 17.1)}
    for (groups, nv), (one, both) in times.items():
        assert (both if two(groups, nv) else one) <= 1.03 * min(one, both), (groups, nv)
    assert two(48, 64, 32) and not two(48, 64, 256)  # an eighth of the device: its own count decides
