"""The field scenarios' convection plan (csrc/field_env_kernel.hip,
fe_conv_plan_kernel) restated in Python and checked against the reference
core's sequential algorithm (complete_port/csim/sb_convect.c:39-73 with
sb_rng.c's masked-rejection interval draw), on the CPU:

  - the producer's records (`hops`) and the walk over them (`room_pairs`), as
    the kernel has them: windows of 104 words entered at any word, whole swaps
    of the commonest candidate count from the records, other counts from the
    first two bytes, longer draws past the window's end, cells without or with
    one candidate. The pairs and the stream position after the room equal the
    sequential draws, over random rooms and one of 46,900 cells, for every
    kind of commonest count (none, up to 64) and counts up to 255; and a
    record alone, at every word of a window;
  - the shuffle's draws as the fixed point over 64 words, and the shuffle
    composed into the room's inverse permutation q from the top (q <- q o (a b)
    as each pair becomes final) and applied as moves T_new[q[i]] = T_old[i],
    equal to the reference's Fisher-Yates shuffle then swaps in order.
"""
from __future__ import annotations

import numpy as np

W = 64


def smear(x: int) -> int:
    for s in (1, 2, 4, 8, 16):
        x |= x >> s
    return x


def interval(words: list, pos: int, mx: int) -> tuple[int, int]:
    """sb_rng_interval (sb_rng.c:45-54) on the stream from pos: (value, next pos)."""
    if mx == 0:
        return 0, pos
    mask = smear(mx)
    while True:
        v = words[pos] & mask
        pos += 1
        if v <= mx:
            return v, pos


def sequential_pairs(words: list, pos: int, ncand, thr: int):
    """sb_conv_apply's cell loop: u <= p (as the 53-bit draw <= thr) and candidates."""
    pairs = []
    for j in range(len(ncand)):
        a, b = words[pos], words[pos + 1]
        pos += 2
        if (((a >> 5) << 26) | (b >> 6)) > thr or ncand[j] == 0:
            continue
        pick, pos = interval(words, pos, int(ncand[j]) - 1)
        pairs.append((j, pick))
    return pairs, pos


def test_composed_moves_equal_shuffled_swaps():
    rng = np.random.default_rng(7)
    for trial in range(200):
        n = int(rng.integers(2, 300))
        m = int(rng.integers(0, n + 1))
        left = rng.integers(0, n, size=m).tolist()
        right = rng.integers(0, n, size=m).tolist()
        words = [int(x) for x in rng.integers(0, 2 ** 32, size=8 * m + 64, dtype=np.uint64)]
        T = rng.normal(size=n)
        # the reference: Fisher-Yates over the pairs from the top, then swaps in order
        L, R, pos = list(left), list(right), 0
        for t in range(m - 1, 0, -1):
            j2, pos = interval(words, pos, t)
            L[t], L[j2] = L[j2], L[t]
            R[t], R[j2] = R[j2], R[t]
        ref = T.copy()
        for a, b in zip(L, R):
            ref[a], ref[b] = ref[b], ref[a]
        # the plan kernel: pair t final once the shuffle passes it, composed into q
        pr = [a | (b << 16) for a, b in zip(left, right)]
        q = list(range(n))
        pos = 0

        def compose(y):
            a, b = y & 0xFFFF, y >> 16
            q[a], q[b] = q[b], q[a]

        for t in range(m - 1, 0, -1):
            j2, pos = interval(words, pos, t)
            x, y = pr[t], pr[j2]
            pr[j2] = x
            compose(y)
        if m > 0:
            compose(pr[0])
        got = T.copy()
        moves = [(q[i], i) for i in range(n) if q[i] != i]
        vals = [T[src] for _, src in moves]
        for (dst, _), v in zip(moves, vals):
            got[dst] = v
        assert np.array_equal(got, ref), trial


def test_draws_by_fixed_point_equal_sequential_draws():
    """The shuffle's draws 64 words at a time: the accepted words of a window
    as the fixed point of "v <= t - (accepted lanes below)", a window ending
    where the draws' mask changes, against one masked rejection after another."""
    rng = np.random.default_rng(31)
    for m in list(range(0, 70)) + [127, 128, 129, 255, 256, 257, 600, 1025, 5000]:
        words = [int(x) for x in rng.integers(0, 2 ** 32, size=8 * m + 256, dtype=np.uint64)]
        start = int(rng.integers(0, 50))
        want, pos = {}, start
        for t in range(m - 1, 0, -1):
            want[t], pos = interval(words, pos, t)
        got, gpos, tt = {}, start, m - 1
        while tt > 0:
            mask = smear(tt)
            low = (mask >> 1) + 1
            v = [words[gpos + i] & mask for i in range(W)]
            acc = [v[i] <= tt for i in range(W)]
            for passes in range(W + 1):
                mine = [tt - sum(acc[:i]) for i in range(W)]
                a2 = [mine[i] >= low and v[i] <= mine[i] for i in range(W)]
                if a2 == acc:
                    break
                acc = a2
            assert a2 == acc
            for i in range(W):
                if acc[i]:
                    assert mine[i] not in got
                    got[mine[i]] = v[i]
            cnt = sum(acc)
            gpos += max(i for i in range(W) if acc[i]) + 1 if cnt == tt - low + 1 else W
            tt -= cnt
        assert got == want and gpos == pos, m


CHUNK = 104          # words of a window (kWin)
NO_HOP = 0xFE        # kNoHop


def hops(w: list, thr: int, usual: int) -> list:
    """produce(): the records of the window whose first word is w[0], and the words past it."""
    swap = [(((w[i] >> 5) << 26) | (w[i + 1] >> 6)) <= thr for i in range(CHUNK)]
    umax, umask = usual - 1, smear(max(usual - 1, 0))
    out = []
    for x in range(CHUNK):
        d = next((q - x for q in range(x, CHUNK, 2) if swap[q]), None)
        if d is None:
            out.append(NO_HOP)
            continue
        v = [w[x + d + 2 + i] & 0xFF & umask for i in range(3)]
        k = 1 if v[0] <= umax else 2 if v[1] <= umax else 3
        ok = v[k - 1] <= umax and x + d + 2 + k < CHUNK
        out.append((d + 2) << 1 | (1 | k << 8 | v[k - 1] << 10 if ok else 0))
    return out


def room_pairs(words: list, pos: int, ncand, thr: int, usual: int):
    """room_pairs(): the walk of one room from stream word pos; the pairs and the position after it."""
    n, pairs, j = len(ncand), [], 0
    if n == 0:
        return pairs, pos
    x0 = pos // CHUNK * CHUNK
    x = drift = pos - x0
    while True:
        rec = hops(words[x0:x0 + CHUNK + 8], thr, usual)
        rule, is_usual = [], []
        for i in range(W):
            nc = int(ncand[min(j + i, n - 1)])
            mx = -2 if j + i >= n or nc == 0 else nc - 1 if nc > 1 else -1
            rule.append((smear(nc - 1) if mx >= 0 else 0, mx))
            is_usual.append(j + i < n and nc == usual)
        got, ahead = [], drift + 2
        while x < CHUNK:
            while True:
                h = rec[x]
                xs = x + ((h >> 1) & 0x7F)
                c = (xs - ahead) >> 1
                if not (is_usual[c & 63] and h & 1):
                    break
                got.append((c, (h >> 10) & 0x3F))
                k = (h >> 8) & 3
                ahead += k
                x = xs + k      # (a whole swap ends before its window does)
                assert x < CHUNK
            if h & NO_HOP == NO_HOP:
                break
            mask, mx = rule[c & 63]
            x = xs
            if mx == -2:
                continue
            v = 0
            if mx >= 0:
                v = words[x0 + x] & 0xFF & mask
                x += 1
                if v > mx:
                    v = words[x0 + x] & 0xFF & mask
                    x += 1
            while mx >= 0 and v > mx:
                v = words[x0 + x] & 0xFF & mask
                x += 1
            got.append((c, v))
            ahead = x - 2 * c
        assert len(got) <= W and all(c < W for c, _ in got)
        drift = ahead - 2
        pairs += [(j + c, v) for c, v in got]
        xe = max(x, CHUNK + (x & 1))
        ce = (xe - drift) >> 1
        if ce >= n - j:
            return pairs, x0 + 2 * (n - j) + drift
        j += ce
        x = xe
        while True:
            x -= CHUNK
            x0 += CHUNK
            if x < CHUNK:
                break
        drift = x


def test_walk_over_records_equals_sequential_draws():
    rng = np.random.default_rng(77)
    for trial in range(400):
        usual = int(rng.choice([0, 2, 3, 8, 24, 33, 48, 63, 64]))
        n = int(rng.integers(0, 500)) if trial else 46900
        p = float(rng.choice([0.0, 0.05, 0.1, 0.3, 0.6, 0.95, 1.0])) if trial else 0.6
        thr = (1 << 53) if p >= 1 else int(np.floor(p * 2.0 ** 53))
        others = np.concatenate([[0, 1], rng.integers(2, 65, 4), rng.integers(65, 256, 4)])
        if trial % 4 == 1:   # a draw that rejects often: 129 of 256 values
            others = np.array([129])
        ncand = rng.choice(others, size=n)
        if usual:
            ncand[rng.random(n) < float(rng.choice([0.1, 0.87, 1.0]))] = usual
        elif n:
            ncand[(ncand >= 2) & (ncand <= 64)] = 0   # the host sets 0 only where no count is in 2..64
        words = [int(x) for x in rng.integers(0, 2 ** 32, size=8 * n + 1000, dtype=np.uint64)]
        start = int(rng.integers(0, 700))
        assert room_pairs(words, start, ncand, thr, usual) == sequential_pairs(words, start, ncand, thr), (trial, n, p)


def test_walk_where_draws_run_past_whole_windows():
    """A candidate draw whose words are all rejected over two windows and more."""
    rng = np.random.default_rng(78)
    for trial in range(40):
        n, usual = int(rng.integers(1, 200)), int(rng.choice([0, 24, 64]))
        ncand = rng.choice([1, 0, 129, 129], size=n) if usual == 0 else rng.choice([usual, 129], size=n)
        words = [int(x) for x in rng.integers(0, 2 ** 32, size=8 * n + 3000, dtype=np.uint64)]
        start = int(rng.integers(0, 300))
        a = start + int(rng.integers(0, 4 * n))
        for q in range(a, a + int(rng.integers(100, 400))):
            words[q] |= 0xFF
        for thr in (1 << 53, 1 << 52):
            assert room_pairs(words, start, ncand, thr, usual) == sequential_pairs(words, start, ncand, thr), trial


def test_hop_records_equal_sequential_draws():
    """A record's whole swap (csrc/field_env_kernel.hip, produce): for a cell of
    `usual` candidates the distance to the next swap of the word's parity, the
    draw's words (at most three, inside the window) and its candidate are those
    of the sequential draws, at every word of a window; whole numbers, so equal."""
    rng = np.random.default_rng(41)
    for trial in range(60):
        usual = int(rng.choice([2, 3, 8, 19, 24, 33, 64]))
        thr = int(np.floor(float(rng.choice([0.0, 0.1, 0.6, 1.0])) * 2.0 ** 53))
        w = [int(x) for x in rng.integers(0, 2 ** 32, size=CHUNK + 700, dtype=np.uint64)]
        for x in range(CHUNK):
            at = [q for q in range(x, CHUNK, 2) if (((w[q] >> 5) << 26) | (w[q + 1] >> 6)) <= thr]
            vs = [(w[at[0] + 2 + i] & 0xFF) & smear(usual - 1) for i in range(3)] if at else []
            k = next((i + 1 for i, v in enumerate(vs) if v <= usual - 1), 0)
            whole = k > 0 and at[0] + 2 + k < CHUNK
            pairs, end = sequential_pairs(w, x, [usual] * ((at[0] - x) // 2 + 1 if at else (CHUNK + 1 - x) // 2), thr)
            assert len(pairs) == (1 if at else 0)
            if whole:
                assert pairs[0] == ((at[0] - x) // 2, vs[k - 1]) and end == at[0] + 2 + k, (trial, x)
