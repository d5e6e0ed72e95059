"""Transposing wave reductions against the plain DPP tree, symbolically.

coffin_amd/csrc/common.hpp sums the 64 lane chains of a unit with a fixed tree
(wave_sum_to_lane63: lanes l^1, l^2, quads, half rows, rows, halves); a batched row must have the
bits of the single-row call (reference contract: models/qwen35/batch.py:19-22), so a
transposing reduction -- several values per lane together, each lane keeping half
of its values per level -- has to build exactly that tree for every value: over whole wavefronts
(wave_sum_pair), and over the 16 blocks of four lanes that the batch kernels' MFMA
steps work on (quarter_sum of gemv_w8a16_batch.hip).  Here both are run on
symbols, with fp32 addition modelled as an unordered pair (it commutes bit for bit and does not
associate), the cross-lane moves modelled after the ISA (DPP quad_perm / row_half_mirror /
row_mirror / row_bcast, v_permlane16_swap, v_permlane32_swap).  The GPU parity tests check the
kernel itself; this pins the lane -> value map and the choice of halves it relies on.
"""
import pytest


def add(a, b):
    """fp32 addition on symbols: commutative, not associative."""
    return frozenset([a, b]) if a != b else ("dup", a)


def dpp(vals, ctrl):
    """What each lane reads through a DPP control: quad_perm [1,0,3,2] / [2,3,0,1],
    row_half_mirror, row_mirror."""
    out = [None] * 64
    for lane in range(64):
        row, j = lane // 16, lane % 16
        if ctrl == 0xB1:
            src = row * 16 + (j ^ 1)
        elif ctrl == 0x4E:
            src = row * 16 + (j ^ 2)
        elif ctrl == 0x141:
            src = row * 16 + (j & 8) + (7 - (j & 7))
        else:
            assert ctrl == 0x140
            src = row * 16 + (15 - j)
        out[lane] = vals[src]
    return out


def original(vals):
    """wave_sum_to_lane63 of one value: the total as lane 63 holds it."""
    v = list(vals)
    for ctrl in (0xB1, 0x4E, 0x141, 0x140):
        d = dpp(v, ctrl)
        v = [add(v[lane], d[lane]) for lane in range(64)]
    w = list(v)
    for lane in range(64):      # row_bcast15 into rows 1 and 3
        row = lane // 16
        if row in (1, 3):
            w[lane] = add(v[lane], v[(row - 1) * 16 + 15])
    v, w = w, list(w)
    for lane in range(32, 64):  # row_bcast31 into rows 2 and 3
        w[lane] = add(v[lane], v[31])
    return w[63]


def swap16(a, b):
    """v_permlane16_swap: odd rows of the first operand <-> even rows of the second."""
    na, nb = list(a), list(b)
    for lane in range(64):
        row, j = lane // 16, lane % 16
        if row % 2 == 1:
            na[lane] = b[(row - 1) * 16 + j]
            nb[(row - 1) * 16 + j] = a[lane]
    return na, nb


def swap32(a, b):
    """v_permlane32_swap: upper half of the first operand <-> lower half of the second."""
    na, nb = list(a), list(b)
    for lane in range(32, 64):
        na[lane] = b[lane - 32]
        nb[lane - 32] = a[lane]
    return na, nb


def level(vals, ctrl, half, upper):
    """One transposing level: pair sums of values i and i + half, a lane keeps one of the two."""
    out = []
    for i in range(half):
        dl, dh = dpp(vals[i], ctrl), dpp(vals[i + half], ctrl)
        lo = [add(vals[i][lane], dl[lane]) for lane in range(64)]
        hi = [add(vals[i + half][lane], dh[lane]) for lane in range(64)]
        out.append([hi[lane] if upper(lane) else lo[lane] for lane in range(64)])
    return out


def pair(vals, upper=lambda l: (l ^ (l >> 2)) & 1):
    """wave_sum_pair of two values: what every lane ends with."""
    t = level(vals, 0xB1, 1, upper)[0]
    for ctrl in (0x4E, 0x141, 0x140):
        d = dpp(t, ctrl)
        t = [add(t[lane], d[lane]) for lane in range(64)]
    for swap in (swap16, swap32):
        x, y = swap(t, t)
        t = [add(x[lane], y[lane]) for lane in range(64)]
    return t


def test_two_rows_of_one_tree_are_the_plain_trees():
    vals = [[(i, lane) for lane in range(64)] for i in range(2)]
    got = pair(vals)
    for lane in range(64):
        assert got[lane] == original(vals[(lane ^ (lane >> 2)) & 1]), lane
    assert got[0] == original(vals[0]) and got[1] == original(vals[1])    # the lanes that store
    # chosen by the plain bit, a lane and its partner of the half row hold different values
    assert original(vals[0]) not in pair(vals, lambda l: l & 1)


def batch(mg, vals, first=lambda l: ((l >> 2) ^ (l >> 3)) & 1):
    """quarter_sum<mg> of gemv_w8a16_batch.hip: 4 mg values a lane over the 16 blocks of four lanes."""
    nv = 4 * mg
    a = level(vals, 0x141, nv // 2, first)
    b = level(a, 0x140, nv // 4, lambda l: (l >> 3) & 1)

    def swapped(swap, x, y):
        p, q = swap(x, y)
        return [add(p[lane], q[lane]) for lane in range(64)]

    if mg == 4:
        return swapped(swap32, swapped(swap16, b[0], b[2]), swapped(swap16, b[1], b[3]))
    c = swapped(swap16, b[0], b[1] if mg == 2 else b[0])
    return swapped(swap32, c, c)


def reversed_in_odd_blocks(lane):
    """lane_row: the activation row that a lane of a block holds."""
    return 3 - (lane & 3) if lane & 4 else lane & 3


def wrong_lanes(mg, got, act):
    """Lanes whose value is not the plain tree over the blocks, b ^ 1, b ^ 2, b ^ 4, b ^ 8 in this order, of value quarter_index and
    the lane's activation row; and the outputs of the lanes that store."""
    def tree(i, j):
        cur = [[(i, lane) for lane in range(4 * b, 4 * b + 4) if act(lane) == j][0] for b in range(16)]
        while len(cur) > 1:
            cur = [add(cur[2 * b], cur[2 * b + 1]) for b in range(len(cur) // 2)]
        return cur[0]

    wrong, held = [], set()
    for lane in range(64):
        s1, s2, b4, b5 = ((lane >> 2) ^ (lane >> 3)) & 1, (lane >> 3) & 1, (lane >> 4) & 1, (lane >> 5) & 1
        i = {4: s1 * 8 + s2 * 4 + b4 * 2 + b5, 2: s1 * 4 + s2 * 2 + b4, 1: s1 * 2 + s2}[mg]
        if got[lane] != tree(i, act(lane)):
            wrong.append(lane)
        if mg == 4 or not lane & (32 if mg == 2 else 48):
            held.add((i, act(lane)))
    return wrong, held


@pytest.mark.parametrize("mg", [1, 2, 4])
def test_batch_reduction_continues_the_single_row_tree(mg):
    """The levels of wave_sum_to_lane63 between chunks that differ in one bit; the lanes that store cover every output exactly once."""
    vals = [[(i, lane) for lane in range(64)] for i in range(4 * mg)]
    wrong, held = wrong_lanes(mg, batch(mg, vals), reversed_in_odd_blocks)
    assert not wrong and held == {(i, j) for i in range(4 * mg) for j in range(4)}


@pytest.mark.parametrize("mg", [1, 2, 4])
def test_batch_reduction_with_other_halves_or_rows_is_caught(mg):
    """Halves kept by the plain lane bit, and activation rows that are not reversed in odd blocks: sums of what does not belong together."""
    vals = [[(i, lane) for lane in range(64)] for i in range(4 * mg)]
    assert wrong_lanes(mg, batch(mg, vals, lambda l: (l >> 2) & 1), reversed_in_odd_blocks)[0]
    assert wrong_lanes(mg, batch(mg, vals), lambda l: l & 3)[0]


def test_single_row_tree_pairs_chunks_by_one_bit():
    """wave_sum_to_lane63 on symbols equals the tree over lane numbers, lowest bit first."""
    cur = [(0, lane) for lane in range(64)]
    want = list(cur)
    while len(want) > 1:
        want = [add(want[2 * b], want[2 * b + 1]) for b in range(len(want) // 2)]
    assert original(cur) == want[0]
