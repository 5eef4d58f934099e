"""CPU checks of kernels' load schedules (restated here from their sources).

k_sgemm (csrc/k3moe_sgemm.hpp), its loader stream, in the bf16 forms (test_sgemm_*)
and the FP4 form (test_fgemm_stream_schedule): units stream back to back; a
loader issues the step ring - 1 ahead at every barrier, waits before it until only
the loads of later steps may be outstanding, and puts weight-scale chunk c of a
unit into buffer (unit's first chunk number + c) & 1. Checked: the wait counts equal
the loads issued after the awaited step, no slot or chunk buffer is overwritten
while a step still reads its older content, and a unit's rows are there when used.

k_latent_sk (csrc/k3moe_latent.hpp): the (row tile, step) items are cut into G
equal runs; a tile must be whole in one run or cut once, every cut tile's two
segments must carry the parts they store, and the second to count in must sum
both into every step of the tile, each part exactly once.
"""
import pytest


def sgemm_scale_reads(KB, sc_steps):
    """(row of 16, first byte, bytes) of every weight-scale load of a row tile whose rows are KB bytes."""
    if KB % 16:   # 4 bytes per step
        for ks in range(KB // 4):
            for row in range(16):
                yield row, 4*ks, 4
        return
    words = sc_steps // 4   # 16-byte words of a row per chunk, each row's in a rotated order
    for c in range(-(-KB // (16*words))):
        for row in range(16):
            for pos in range(words):
                at = 16*words*c + 16*(pos ^ (row >> (2 if words == 4 else 3)))
                if at < KB:
                    yield row, at, 16


@pytest.mark.parametrize('KB', [4, 8, 12, 16, 20, 24, 48, 56, 64, 72, 112, 224])
@pytest.mark.parametrize('sc_steps', [8, 16])
def test_sgemm_scale_loads_stay_in_their_rows(KB, sc_steps):
    """Every scale byte of the tile is loaded once and no load leaves its row (the last row ends the tensor)."""
    seen = [[0]*KB for _ in range(16)]
    for row, b, n in sgemm_scale_reads(KB, sc_steps):
        assert b + n <= KB, (KB, row, b, n)
        for j in range(b, b + n):
            seen[row][j] += 1
    assert all(v == 1 for row in seen for v in row)


def sgemm_stream(ring, sc_steps, KS, unit_rows, row_loads=1, step_loads=0, gather_loads=1):
    """One loader's run over units with unit_rows blocks of activation rows each (row_loads loads a block; step_loads
    more in every step): its waits, slots, scale chunks and gathered rows."""
    wide, gather, ahead = KS % 4 == 0, KS >= ring - 1, ring - 1
    nsc = -(-KS // sc_steps)
    total = KS*len(unit_rows)
    issued, landed_rows = [], {}

    def issue(g):
        u, ks = divmod(g, KS)
        n = 4 + row_loads*unit_rows[u] + step_loads + (0 if wide else 1)
        if gather and ks == 0:
            if u > 0:   # the unit's rows came with step 0 of the unit before, which has been waited for
                assert landed_rows[u] <= waited, (g, waited)
            if u + 1 < len(unit_rows):
                landed_rows[u + 1] = g
                n += gather_loads
        chunk = None
        if wide and (ks == 0 or (ks >= ahead and (ks - ahead) % sc_steps == 0 and (ks - ahead)//sc_steps + 1 < nsc)):
            c = 0 if ks == 0 else (ks - ahead)//sc_steps + 1
            chunk = u*nsc + c
            n += 4 if sc_steps == 16 else 2   # (two tiles' chunks a load)
        issued.append((g, n, chunk))

    def chunk_of(g):
        return g//KS*nsc + g % KS//sc_steps

    waited = -1
    counts = []
    for g in range(min(ahead, total)):
        issue(g)
        counts.append(issued[-1][1])
    later = sum(counts[1:])
    counts = counts[1:] + [0]*(ahead - len(counts))
    for g in range(total):
        assert later == sum(n for gs, n, _ in issued if gs > g)
        waited = g
        done = g - 1   # at this barrier the MFMA waves have read every step up to this one
        if wide:       # the step's chunk has been loaded, into the buffer it is read from
            assert any(c == chunk_of(g) for gs, _, c in issued if gs <= g)
        later -= counts[0]
        counts = counts[1:] + [0]
        if g + ahead < total:
            issue(g + ahead)
            assert g + ahead - ring <= done   # the slot's last step
            chunk = issued[-1][2]
            if chunk is not None:   # the buffer held chunk - 2: no unread step uses it
                assert all(chunk_of(s) != chunk - 2 for s in range(done + 1, total))
            counts[-1] = issued[-1][1]
            later += counts[-1]


@pytest.mark.parametrize('ring,sc_steps', [(5, 16), (4, 8), (3, 16)])
@pytest.mark.parametrize('KS', [1, 2, 3, 4, 5, 6, 8, 12, 16, 20, 24, 28, 48, 56, 64])
@pytest.mark.parametrize('unit_rows', [[2], [1, 3, 2], [3, 1, 1, 2, 3, 1, 2]])
def test_sgemm_stream_schedule(ring, sc_steps, KS, unit_rows):
    """The bf16 forms (units of 32 and 64 pairs; ring 3 as the FP4 form's): steps issued ring - 1 ahead across units
    whose activation loads differ."""
    sgemm_stream(ring, sc_steps, KS, unit_rows)


@pytest.mark.parametrize('KS', [2, 4, 6, 8, 12, 16, 20, 24, 28, 32, 48, 56, 64])
@pytest.mark.parametrize('nunits', [1, 2, 3, 5])
@pytest.mark.parametrize('scale_dwords', [0, 1])
def test_fgemm_stream_schedule(KS, nunits, scale_dwords):
    """The FP4 form (96 pairs, two steps ahead): each block of rows is loaded in both terms, three of the four loaders
    also take the rows' scale dwords, and a unit's rows are gathered in two loads."""
    sgemm_stream(3, 16, KS, [1 + u % 3 for u in range(nunits)], row_loads=2, step_loads=scale_dwords, gather_loads=2)


def sk_order(lo, hi, KS):
    """k_latent_sk's processing order of a run's (tile, step) items: the last
    tile's head when that tile is cut, the first tile's tail when that one is,
    then the whole tiles between; (rt, ks, k0, k1) per item, k0 / k1 the
    tile's first step and end in the run."""
    rt_lo, ks_lo = lo // KS, lo % KS
    rt_hi, ks_end = (hi - 1) // KS, (hi - 1) % KS + 1
    cut_first, cut_last = ks_lo > 0, rt_hi != rt_lo and ks_end < KS
    entries = []
    if cut_last:
        entries.append((rt_hi, rt_hi, 0, ks_end))
    if cut_first:
        entries.append((rt_lo, rt_lo, ks_lo, KS))
    if rt_lo + cut_first <= rt_hi - cut_last:
        entries.append((rt_lo + cut_first, rt_hi - cut_last, 0, KS))
    items = []
    for r0, r1, k0, k1 in entries:
        for rt in range(r0, r1 + 1):
            a = k0 if rt == r0 else 0
            b = k1 if rt == r1 else KS
            items += [(rt, ks, a, b) for ks in range(a, b)]
    return items


def latent_sk_runs(RT, KS, KS0, G, out, second_first=False):
    NI = RT * KS
    has0 = lambda ka: (not out) or ka < KS0
    has1 = lambda kb: out and kb > KS0
    parts, result, count = {}, {}, {}
    counts = []
    for b in range(G):
        lo, hi = NI * b // G, NI * (b + 1) // G
        assert hi - lo >= KS
        items = sk_order(lo, hi, KS)
        assert sorted((rt * KS + ks) for rt, ks, _, _ in items) == list(range(lo, hi))
        acc0, acc1, cuts = set(), set(), []
        for rt, ks, ka, kb in items:
            (acc1 if out and ks >= KS0 else acc0).add((rt, ks))
            if ks + 1 == kb:
                if ka == 0 and kb == KS:
                    result[rt] = (frozenset(acc0), frozenset(acc1))
                else:
                    seg = 0 if ka == 0 else 1
                    if has0(ka):
                        parts[(rt, seg, 0)] = frozenset(acc0)
                    if has1(kb):
                        parts[(rt, seg, 1)] = frozenset(acc1)
                    cuts.append((rt, kb if ka == 0 else ka))
                acc0, acc1 = set(), set()
        assert len(cuts) <= 2  # the kernel keeps two
        counts += cuts
    # the counts arrive in any order; the second of a tile's two sums both
    # segments (after every partial is stored)
    for rt, kc in (reversed(counts) if second_first else counts):
        count[rt] = count.get(rt, 0) + 1
        if count[rt] == 1:
            continue
        s0 = parts[(rt, 0, 0)] | (parts[(rt, 1, 0)] if has0(kc) else frozenset())
        s1 = (parts[(rt, 0, 1)] if has1(kc) else frozenset()) | (parts[(rt, 1, 1)] if has1(KS) else frozenset())
        result[rt] = (s0, s1)
    assert all(c == 2 for c in count.values())
    for rt in range(RT):
        want0 = frozenset((rt, k) for k in range(KS) if (not out) or k < KS0)
        want1 = frozenset((rt, k) for k in range(KS0, KS)) if out else frozenset()
        assert result[rt] == (want0, want1), rt


@pytest.mark.parametrize('RT,KS,KS0,G,out', [
    (448, 34, 28, 256, True),    # latent_out of a Kimi K3 TP8 rank
    (320, 23, 20, 256, True),    # the test geometry with cut tiles
    (320, 56, 56, 256, False),
    (64, 12, 4, 64, True),
    (300, 7, 5, 256, True),
])
def test_latent_sk_segments(RT, KS, KS0, G, out):
    latent_sk_runs(RT, KS, KS0, G, out)
    latent_sk_runs(RT, KS, KS0, G, out, second_first=True)


def test_latent_sk_order_puts_cut_segments_first():
    # run [5, 5 + 20) of 8-step tiles: tile 0 steps 5-7, tile 1, tile 2, tile 3 steps 0-0
    items = sk_order(5, 25, 8)
    assert items[0] == (3, 0, 0, 1)
    assert [it[:2] for it in items[1:4]] == [(0, 5), (0, 6), (0, 7)]
    assert [it[:2] for it in items[4:]] == [(1, k) for k in range(8)] + [(2, k) for k in range(8)]
    assert sk_order(16, 24, 8) == [(2, k, 0, 8) for k in range(8)]
