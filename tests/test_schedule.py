"""CPU replay of the assembly kernels' scatter schedules (k_thermal, k_ns) and
of the kernels that own their rows (k_q2box, k_q2res, k_gather_rows: at the end).

The three scattering schedules of `assembly.colouring` are restated here from
the kernel's index arithmetic (lattice.hpp `element_of`, `element_of_seg`,
`axis_key`; assemble.hip `launch_colors`, the first-touch flags and the x-segment
LDS image) and replayed on small lattices:

* every element is assembled exactly once;
* race freedom: two work units that may run at the same time never write the
  same CRS entry or residual row (element / segment colouring: one launch;
  block colouring: one launch, different workgroups, or one workgroup and one
  sub-phase);
* first touch: every entry of the CRS pattern has exactly one writer whose
  first-touch flag is set, and it runs strictly before every other writer of
  that entry, so overwrite mode needs no zero fill;
* the segment image: the LDS slot an element's (row, column) contribution is
  summed into decodes, in the write-out loop, to the same global entry, and
  the workgroup's strided loops visit every slot exactly once.

The reference adds every contribution with atomics and a column search
(assemblyManager_scatter.hpp:164-278); these are the invariants that let the
coloured, atomic-free form produce the same matrix.
"""
from __future__ import annotations

import itertools

import pytest

# ---------------------------------------------------------------------------
# kernel configuration (assemble.hip Cfg / SegCfg)
# ---------------------------------------------------------------------------


def pow2ceil(x):
    r = 1
    while r < x:
        r *= 2
    return r


def cfg(dim, p, block=256):
    nb = (p + 1) ** dim
    g = max(4, pow2ceil(nb + 1))
    return dict(NB=nb, G=g, GPB=block // g, BLOCK=block)


def seg_cfg(dim, p, s):
    p1 = p + 1
    rp = p1 ** (dim - 1)
    cp = rp
    wv, wi = 2 * p + 1, p + 1
    sv, si = rp * cp * wv, rp * cp * wi
    gs = sv + (p - 1) * si
    return dict(P1=p1, RP=rp, CP=cp, WV=wv, WI=wi, SV=sv, SI=si, GS=gs, NPL=p * s + 1, kSize=s * gs + sv,
                kRows=(p * s + 1) * rp)


def plane_off(sc, p, x):
    return (x // p) * sc["GS"] + (0 if x % p == 0 else sc["SV"] + (x % p - 1) * sc["SI"])


def block_shape(dim, gpb):
    s = [1, 1, 1]
    prod = 1
    while prod < gpb:
        d = 0
        for k in range(1, dim):
            if s[k] < s[d]:
                d = k
        s[d] *= 2
        prod *= 2
    return s


# ---------------------------------------------------------------------------
# launches: (launch index, workgroup, sub-phase, unit) per element, as the
# kernel enumerates them
# ---------------------------------------------------------------------------
ELEM, BLOCKED, SEG = 0, 1, 2


def schedule(mode, dim, nel, gpb):
    """Yield dicts: launch, wg, sub, elems (list of ec tuples), seg (sx, s_act) or None,
    plus the AsmArgs fields the key functions read."""
    nel = list(nel) + [1] * (3 - len(nel))
    s = block_shape(dim, gpb)
    bw = [2 * x for x in s]
    nseg = (nel[0] + gpb - 1) // gpb
    ncol = 1 << dim
    for col in range(ncol):
        cn = [0, 0, 0]
        cnt = 1
        for d in range(3):
            cd = (col >> d) & 1
            units = nel[d] if d < dim else 1
            if d < dim and mode == BLOCKED:
                units = (nel[d] + bw[d] - 1) // bw[d]
            if d == 0 and mode == SEG:
                units = nseg
            n = (units - cd + 1) // 2 if d < dim else 1
            if d >= dim and cd:
                n = 0
            cn[d] = n
            cnt *= n
        if cnt == 0:
            continue
        blocks = (cnt + gpb - 1) // gpb if mode == ELEM else cnt
        for b in range(blocks):
            if mode == ELEM:
                for g in range(gpb):
                    idx = b * gpb + g
                    if idx >= cnt:
                        continue
                    t = idx
                    e0 = 2 * (t % cn[0]) + (col & 1)
                    t //= cn[0]
                    e1 = 2 * (t % cn[1]) + ((col >> 1) & 1)
                    t //= cn[1]
                    e2 = 2 * t + ((col >> 2) & 1) if dim == 3 else 0
                    yield dict(launch=col, wg=b, sub=0, elems=[(e0, e1, e2)], seg=None, bw=bw, nseg=nseg)
            elif mode == BLOCKED:
                for sub in range(ncol):
                    for g in range(gpb):
                        gc = [g % s[0], (g // s[0]) % s[1], g // (s[0] * s[1])]
                        t = b
                        ec = [0, 0, 0]
                        ok = True
                        for d in range(dim):
                            bi = 2 * (t % cn[d]) + ((col >> d) & 1)
                            t //= cn[d]
                            ec[d] = bi * bw[d] + 2 * gc[d] + ((sub >> d) & 1)
                            ok = ok and ec[d] < nel[d]
                        if ok:
                            yield dict(launch=col, wg=b, sub=sub, elems=[tuple(ec)], seg=None, bw=bw, nseg=nseg)
            else:
                t = b
                sx = 2 * (t % cn[0]) + (col & 1)
                t //= cn[0]
                e1 = 2 * (t % cn[1]) + ((col >> 1) & 1)
                t //= cn[1]
                e2 = 2 * t + ((col >> 2) & 1) if dim == 3 else 0
                rest = nel[0] - sx * gpb
                s_act = min(rest, gpb)
                elems = [(sx * gpb + g, e1, e2) for g in range(gpb) if g < s_act]
                yield dict(launch=col, wg=b, sub=0, elems=elems, seg=(sx, s_act), bw=bw, nseg=nseg)


def axis_key(mode, bw, d, e):
    return (((e // bw[d]) & 1) * 2 if mode == BLOCKED else 0) + (e & 1)


def first_flags(mode, dim, nel, unit, ec):
    lo, hi = [True] * 3, [True] * 3
    for d in range(dim):
        if mode == SEG and d == 0:
            sx = unit["seg"][0]
            lo[0] = sx == 0 or (sx & 1) < ((sx - 1) & 1)
            hi[0] = sx == unit["nseg"] - 1 or (sx & 1) < ((sx + 1) & 1)
            continue
        k = axis_key(mode, unit["bw"], d, ec[d])
        lo[d] = ec[d] == 0 or k < axis_key(mode, unit["bw"], d, ec[d] - 1)
        hi[d] = ec[d] == nel[d] - 1 or k < axis_key(mode, unit["bw"], d, ec[d] + 1)
    return lo, hi


def local(i, p, dim):
    p1 = p + 1
    return (i % p1, (i // p1) % p1, i // (p1 * p1) if dim == 3 else 0)


def gnode(ec, loc, p):
    return tuple(p * ec[d] + loc[d] for d in range(3))


# ---------------------------------------------------------------------------
# writes of one work unit: {(row node, col node): first?}
# ---------------------------------------------------------------------------


def unit_writes_element(mode, dim, p, nel, unit):
    (ec,) = unit["elems"]
    lo, hi = first_flags(mode, dim, nel, unit, ec)
    nb = (p + 1) ** dim
    out = {}
    for i in range(nb):
        il = local(i, p, dim)
        for j in range(nb):
            jl = local(j, p, dim)
            f = True
            for d in range(dim):
                if il[d] == jl[d] and il[d] in (0, p):
                    f = f and (lo[d] if il[d] == 0 else hi[d])
            out[(gnode(ec, il, p), gnode(ec, jl, p))] = f
    return out


def unit_writes_segment(dim, p, nel, unit, nn):
    """The write-out loop of the x-segment scatter: decode every LDS slot
    back to (row, column) and apply the kernel's skip and first-touch rules."""
    sx, s_act = unit["seg"]
    gpb = unit["gpb"]
    sc = seg_cfg(dim, p, gpb)
    ec0 = unit["elems"][0]
    lo, hi = first_flags(SEG, dim, nel, unit, ec0)
    x0g = p * sx * gpb
    xend = p * s_act
    yb, zb = p * ec0[1], p * ec0[2]
    p1 = p + 1
    out = {}
    for eix in range(sc["kSize"]):
        grp, rem = divmod(eix, sc["GS"])
        if rem < sc["SV"]:
            X = p * grp
            r = rem // (sc["CP"] * sc["WV"])
            cb = (rem // sc["WV"]) % sc["CP"]
            xo = rem % sc["WV"]
        else:
            r2 = rem - sc["SV"]
            X = p * grp + 1 + r2 // sc["SI"]
            rr = r2 % sc["SI"]
            r = rr // (sc["CP"] * sc["WI"])
            cb = (rr // sc["WI"]) % sc["CP"]
            xo = rr % sc["WI"]
        xg = x0g + X
        if X > xend or xg >= nn[0]:
            continue
        xcol = xg - p + xo if X % p == 0 else xg - X % p + xo
        if xcol < 0 or xcol >= nn[0]:
            continue
        if (X == 0 and xcol < xg) or (X == xend and xcol > xg):
            continue
        iy, iz = r % p1, (r // p1 if dim == 3 else 0)
        jy, jz = cb % p1, (cb // p1 if dim == 3 else 0)
        sh = True
        if X == 0 and xcol == xg:
            sh = sh and lo[0]
        if X == xend and xcol == xg:
            sh = sh and hi[0]
        if iy == jy == 0:
            sh = sh and lo[1]
        if iy == jy == p:
            sh = sh and hi[1]
        if dim == 3 and iz == jz == 0:
            sh = sh and lo[2]
        if dim == 3 and iz == jz == p:
            sh = sh and hi[2]
        out[((xg, yb + iy, zb + iz), (xcol, yb + jy, zb + jz))] = (sh, eix)
    return out


def element_entries(ec, p, dim):
    nb = (p + 1) ** dim
    return {(gnode(ec, local(i, p, dim), p), gnode(ec, local(j, p, dim), p)) for i in range(nb) for j in range(nb)}


def pattern_entries(dim, p, nel):
    """The CRS pattern: union of element couplings (linearAlgebraInterface_construct.hpp:243-258)."""
    nel3 = list(nel) + [1] * (3 - len(nel))
    ents = set()
    for ec in itertools.product(*(range(n) for n in nel3)):
        ents |= element_entries(ec, p, dim)
    return ents


# ---------------------------------------------------------------------------
# checks
# ---------------------------------------------------------------------------
CASES = [
    # dim, p, nel
    (2, 1, (9, 7)),
    (2, 2, (11, 6)),
    (2, 3, (7, 5)),
    (3, 1, (9, 5, 4)),
    (3, 2, (9, 4, 3)),
    (3, 2, (17, 3, 3)),
]


def replay(mode, dim, p, nel, gpb):
    nel3 = list(nel) + [1] * (3 - len(nel))
    nn = [p * n + 1 for n in nel3]
    writes = {}  # entry -> list of (time, concurrency key, first)
    seen = {}
    for unit in schedule(mode, dim, nel, gpb):
        unit["gpb"] = gpb
        for ec in unit["elems"]:
            seen[ec] = seen.get(ec, 0) + 1
        if mode == SEG:
            w = {k: v[0] for k, v in unit_writes_segment(dim, p, nel3, unit, nn).items()}
            # every contribution of the segment's elements is in its image
            covered = set()
            for ec in unit["elems"]:
                covered |= element_entries(ec, p, dim)
            assert covered == set(w), "segment image misses or adds entries"
        else:
            w = unit_writes_element(mode, dim, p, nel3, unit)
        # time: launch, then sub-phase inside one workgroup (block colouring)
        for ent, f in w.items():
            writes.setdefault(ent, []).append(((unit["launch"], unit["sub"]), unit["wg"], f))
    return nel3, seen, writes


@pytest.mark.parametrize("mode", [ELEM, BLOCKED, SEG], ids=["element", "block", "segment"])
@pytest.mark.parametrize("gpb", [4, 8])
@pytest.mark.parametrize("dim,p,nel", CASES)
def test_schedule_race_free_and_first_touch(mode, gpb, dim, p, nel):
    nel3, seen, writes = replay(mode, dim, p, nel, gpb)
    # every element exactly once
    all_el = set(itertools.product(*(range(n) for n in nel3)))
    assert set(seen) == all_el and all(v == 1 for v in seen.values())
    # the union of writes is the CRS pattern
    assert set(writes) == pattern_entries(dim, p, nel)
    for ent, ws in writes.items():
        # race freedom: writers with the same launch run concurrently unless
        # they are sub-phases of one workgroup (barrier between sub-phases)
        for (t1, wg1, _), (t2, wg2, _) in itertools.combinations(ws, 2):
            if t1[0] == t2[0]:
                assert mode == BLOCKED and wg1 == wg2 and t1[1] != t2[1], f"race on {ent}: {ws}"
        firsts = [w for w in ws if w[2]]
        assert len(firsts) == 1, f"entry {ent}: {len(firsts)} first touchers in {ws}"
        t0 = firsts[0][0]
        assert all(w[0] > t0 for w in ws if not w[2]), f"entry {ent}: a later touch runs before the first"


def test_residual_rows_race_free():
    """Residual rows follow the diagonal entries' schedule: the same replay
    restricted to (row, row)."""
    for mode in (ELEM, BLOCKED, SEG):
        nel3, _, writes = replay(mode, 3, 2, (9, 4, 3), 8)
        diag = {e: w for e, w in writes.items() if e[0] == e[1]}
        nn = [2 * n + 1 for n in nel3]
        assert len(diag) == nn[0] * nn[1] * nn[2]
        for ws in diag.values():
            assert sum(1 for w in ws if w[2]) == 1


# ---------------------------------------------------------------------------
# the x-segment LDS image
# ---------------------------------------------------------------------------
BUILT = [(2, p) for p in range(1, 7)] + [(3, 1), (3, 2)]


@pytest.mark.parametrize("dim,p", BUILT)
def test_segment_image_slot_decodes_to_its_entry(dim, p):
    """The slot an element's contribution is summed into (scatter phase) and
    the (row, column) the write-out loop decodes from that slot agree, and
    no two contributions of different entries share a slot."""
    c = cfg(dim, p)
    gpb = c["GPB"]
    sc = seg_cfg(dim, p, gpb)
    p1 = p + 1
    nel = (gpb, 1, 1) if dim == 2 else (gpb, 1, 1)
    nn = [p * n + 1 for n in nel]
    unit = dict(launch=0, wg=0, sub=0, elems=[(g, 0, 0) for g in range(gpb)], seg=(0, gpb), bw=[2, 2, 2], nseg=1,
                gpb=gpb)
    decoded = {v[1]: k for k, v in unit_writes_segment(dim, p, list(nel), unit, nn).items()}
    slot_of = {}
    for g in range(gpb):
        for i in range(c["NB"]):
            ix, iy, iz = local(i, p, dim)
            for j in range(c["NB"]):
                jx, jy, jz = local(j, p, dim)
                vtx = ix == 0 or ix == p
                w = sc["WV"] if vtx else sc["WI"]
                xo = jx - ix + p if vtx else jx
                idx = plane_off(sc, p, p * g + ix) + ((iy + p1 * iz) * sc["CP"] + (jz * p1 + jy)) * w + xo
                assert 0 <= idx < sc["kSize"]
                ent = ((p * g + ix, iy, iz), (p * g + jx, jy, jz))
                assert slot_of.setdefault(ent, idx) == idx
                assert decoded[idx] == ent
    assert len(set(slot_of.values())) == len(slot_of)
    # residual rows: (plane, row-in-plane) slots inside kRows
    assert max((p * (gpb - 1) + p) * sc["RP"] + (p1 ** (dim - 1) - 1), 0) < sc["kRows"]


def strided_visits(n, block, stride, chunk=1):
    """How often each slot is visited by `for (b = tid; b < n; b += stride * chunk)
    for c < chunk: k = b + c * stride` over tid < block."""
    cnt = [0] * n
    for tid in range(block):
        b = tid
        while b < n:
            for c in range(chunk):
                k = b + c * stride
                if k < n:
                    cnt[k] += 1
            b += stride * chunk
    return cnt


@pytest.mark.parametrize("dim,p", BUILT)
@pytest.mark.parametrize("block", [128, 256])
def test_segment_loops_visit_every_slot_once(dim, p, block):
    """The zeroing, residual and write-out loops stride by the workgroup size.
    With the stride equal to the block every slot is visited once; a fixed
    256-lane stride in a 128-lane build leaves half the image unzeroed and
    unwritten (the disagreement a 128-lane build once showed)."""
    c = cfg(dim, p, block)
    if c["GPB"] < 2:
        pytest.skip("fewer than two elements per workgroup")
    sc = seg_cfg(dim, p, c["GPB"])
    for n, chunk in ((sc["kSize"], 1), (sc["kRows"], 1), (sc["kSize"], 8)):
        assert strided_visits(n, block, block, chunk) == [1] * n
    if block == 128:
        bad = strided_visits(sc["kSize"], 128, 256)
        assert 0 in bad


# ---------------------------------------------------------------------------
# row-owned kernels (one writer per row, one launch): assemble_q2box.hip
# (assembly.colouring = 3, Q2 hexahedra on boxes), assemble_q2res.hip (its
# residual alone) and the row gather of assemble_elem.hip.  Restated from the
# kernels' lane arithmetic: every write is (CRS position or row, contributing
# elements in the order of the sums).  The replay checks that every entry of the
# CRS pattern is written once, at its position, with the contribution of every
# element that holds both of its nodes exactly once.
# ---------------------------------------------------------------------------
def node_elems(node, nel, p=2):
    """Elements holding a lattice node."""
    rng = []
    for c, n in zip(node, nel):
        cand = [c // p - 1, c // p] if c % p == 0 else [c // p]
        rng.append([e for e in cand if 0 <= e < n])
    return sorted(itertools.product(*rng))


def axis_row(c, n, p=2):
    """First column and number of columns of lattice coordinate c."""
    if c % p:
        return c - c % p, p + 1
    lo, hi = max(c - p, 0), min(c + p, p * n)
    return lo, hi - lo + 1


def crs(nel, p=2):
    """Positions of all entries: {(row node, column node): position}, x fastest."""
    nn = [p * n + 1 for n in nel]
    pos, k = {}, 0
    for Z, Y, X in itertools.product(*(range(m) for m in reversed(nn))):
        box = [range(lo, lo + ln) for lo, ln in (axis_row(c, n, p) for c, n in zip((X, Y, Z), nel))]
        for z, y, x in itertools.product(*reversed(box)):
            pos[((X, Y, Z), (x, y, z))] = k
            k += 1
    return pos


def q2_prefix(X):
    e = X >> 1
    return (3 if e == 0 else 8 * e + 3) if X & 1 else (0 if e == 0 else 8 * e - 2)


def q2box_writes(nel, seg):
    """Writes of k_q2box: [(CRS position, contributing elements)], [(row node, contributing elements)]."""
    n0, n1, n2 = nel
    N1, N2 = 2 * n1 + 1, 2 * n2 + 1
    T0, T1 = 8 * n0 + 1, 8 * n1 + 1
    nseg, cn1, cn2 = -(-n0 // seg), (n1 + 2) // 2, (n2 + 2) // 2
    jw, rw = [], []
    # elements of an axis that an assembled pair 0..7 of block e sums: vertex row
    # 2e against columns 2e-2 .. 2e+2, interior row 2e+1 against 2e .. 2e+2
    pair_elems = lambda e, q, n: [v for v in ((e - 1,), (e - 1,), (e - 1, e), (e,), (e,), (e,), (e,), (e,))[q]  # noqa: E731
                                  if 0 <= v < n]
    for block in range(nseg * cn1 * cn2):
        bq = block // nseg
        x0 = (block - bq * nseg) * seg
        x1 = min(x0 + seg, n0)
        ey0, ez0 = 2 * (bq % cn1), 2 * (bq // cn1)
        for wv in range(4):
            ey, ez = ey0 + (wv & 1), ez0 + (wv >> 1)
            if ey > n1 or ez > n2:
                continue
            EYv, EYm = (5 if 0 < ey < n1 else 3), (3 if ey < n1 else 0)
            EZv, EZm = (5 if 0 < ez < n2 else 3), (3 if ez < n2 else 0)
            nr = [EYv * EZv, EYm * EZv, EYv * EZm, EYm * EZm]
            lb = [sum(nr[:j]) for j in range(5)]
            assert lb[4] <= 64
            zs, ys = [q2_prefix(2 * ez + k) * T1 * T0 for k in (0, 1)], [q2_prefix(2 * ey + k) * T0 for k in (0, 1)]
            line = [zs[j >> 1] + (EZm if j >> 1 else EZv) * ys[j & 1] for j in range(4)]
            carry = [None] * 64
            for e in range(max(x0 - 1, 0), x1):
                staged = {}  # LDS slot -> elements of the sum
                width = 8 if e > 0 else 6
                last = {}
                for lane in range(lb[4]):
                    j = sum(lane >= lb[k] for k in (1, 2, 3))
                    pt = lane - lb[j]
                    EY = 3 if j & 1 else EYv
                    iy, iz = pt % EY, pt // EY
                    yp = 5 + iy if j & 1 else (2 + iy if ey == 0 else iy)
                    zp = 5 + iz if j >> 1 else (2 + iz if ez == 0 else iz)
                    yz = list(itertools.product(pair_elems(ey, yp, n1), pair_elems(ez, zp, n2)))
                    own = [(e, y, z) for y, z in yz]
                    if e > 0:
                        c = carry[lane] or []
                        for k in range(5):
                            staged[8 * lb[j] + 5 * pt + k] = (c if k < 2 else c + own if k == 2 else own)
                        for k in range(3):
                            staged[8 * lb[j] + 5 * nr[j] + 3 * pt + k] = own
                    else:
                        for k in range(3):
                            staged[6 * lb[j] + 3 * pt + k] = own
                            staged[6 * lb[j] + 3 * nr[j] + 3 * pt + k] = own
                    for k in range(3):
                        last[3 * lane + k] = own
                    carry[lane] = own
                if e >= x0:
                    assert sorted(staged) == list(range(width * lb[4]))
                    for idx, els in staged.items():
                        j = sum(idx >= width * lb[k] for k in (1, 2, 3))
                        at = idx - width * lb[j]
                        jw.append((line[j] + at + (8 * nr[j] * e - 2 * nr[j] if e > 0 else 0), els))
                    if e + 1 == n0:
                        for idx, els in last.items():
                            j = sum(idx >= 3 * lb[k] for k in (1, 2, 3))
                            jw.append((line[j] + nr[j] * (8 * n0 - 2) + idx - 3 * lb[j], els))
            # residual rows of the block (16 lanes of the workgroup, four a block)
            for e in range(x0, x1):
                for j in range(4):
                    Y, Z = 2 * ey + (j & 1), 2 * ez + (j >> 1)
                    if Y >= N1 or Z >= N2:
                        continue
                    es = [(ey,) if j & 1 else (ey - 1, ey), (ez,) if j >> 1 else (ez - 1, ez)]
                    yz = [(y, z) for y, z in itertools.product(*es) if 0 <= y < n1 and 0 <= z < n2]
                    for k in range(3 if e + 1 == n0 else 2):
                        xs = ([e - 1] if e > 0 else []) + [e] if k == 0 else [e]
                        rw.append(((2 * e + k, Y, Z), [(x, y, z) for x in xs for y, z in yz]))
    return jw, rw


@pytest.mark.parametrize("seg", [2, 4, 12])
@pytest.mark.parametrize("nel", [(5, 4, 3), (7, 3, 2), (8, 1, 1), (1, 1, 1), (2, 5, 7), (13, 2, 3)])
def test_row_owned_schedule(nel, seg):
    jw, rw = q2box_writes(nel, seg)
    pos = crs(nel)
    assert {k for k, _ in pos.items()} == pattern_entries(3, 2, nel)
    at = {p: ent for ent, p in pos.items()}
    assert sorted(p for p, _ in jw) == list(range(len(pos))), "entries not written exactly once"
    for p, els in jw:
        r, c = at[p]
        assert sorted(els) == sorted(set(node_elems(r, nel)) & set(node_elems(c, nel))), (r, c, els)
    assert len(rw) == len({r for r, _ in rw}) == (2 * nel[0] + 1) * (2 * nel[1] + 1) * (2 * nel[2] + 1)
    for r, els in rw:
        assert sorted(els) == node_elems(r, nel), (r, els)


@pytest.mark.parametrize("walk", [1, 2, 5, 48])
@pytest.mark.parametrize("nel", [(1, 1, 1), (6, 7, 1), (7, 6, 2), (8, 8, 3), (14, 13, 9), (15, 1, 4)])
def test_residual_tiles_own_every_row_once(nel, walk):
    """k_q2res: 8 x 8 lanes of elements, 7 x 7 of them own the rows 2e and 2e + 1
    of block e per axis and take the lower neighbour's share from the lane (x,
    y) or the layer (z) before."""
    n0, n1, n2 = nel
    tx, ty, nb = (n0 + 7) // 7, (n1 + 7) // 7, n2 + 1
    rows = {}
    for bx, by, bz in itertools.product(range(tx), range(ty), range(-(-nb // walk))):
        z0, z1 = bz * walk, min((bz + 1) * walk, nb)
        layers = list(range(max(z0 - 1, 0), z1))
        for lx, ly in itertools.product(range(8), range(8)):
            ex, ey = 7 * bx + lx - 1, 7 * by + ly - 1
            if not (lx > 0 and ly > 0 and ex <= n0 and ey <= n1):
                continue
            for z in range(z0, z1):
                for i, j, k in itertools.product(range(2), range(2), range(2)):
                    r = (2 * ex + i, 2 * ey + j, 2 * z + k)
                    if any(c > 2 * n for c, n in zip(r, nel)):
                        continue
                    assert z == 0 or k or z - 1 in layers
                    els = itertools.product((ex - 1, ex) if i == 0 else (ex,), (ey - 1, ey) if j == 0 else (ey,),
                                            (z - 1, z) if k == 0 else (z,))
                    els = sorted(e for e in els if all(0 <= c < n for c, n in zip(e, nel)))
                    assert r not in rows, f"row {r} owned twice"
                    rows[r] = els
    assert set(rows) == set(itertools.product(*(range(2 * n + 1) for n in nel)))
    for r, els in rows.items():
        assert els == node_elems(r, nel), (r, els)


@pytest.mark.parametrize("dim,p,nel", [(2, 1, (5, 3)), (2, 2, (3, 4)), (2, 3, (2, 3)), (2, 6, (1, 2)), (3, 1, (3, 2, 4)),
                                       (3, 2, (2, 3, 1))])
def test_row_gather(dim, p, nel):
    """k_gather_rows: each element around a row adds its row of element matrix
    into the row's image at the columns' places, in the order of the element
    colours (the even one of two along an axis first)."""
    nel3 = list(nel) + [1] * (3 - dim)
    p1, nn = p + 1, [p * n + 1 if d < dim else 1 for d, n in enumerate(nel3)]
    for X, Y, Z in itertools.product(*(range(m) for m in nn)):
        row = (X, Y, Z)
        lo, ln, el, il, po, two = ([0] * 3, [1] * 3, [[0, 0] for _ in range(3)], [[0, 0] for _ in range(3)],
                                   [[0, 0] for _ in range(3)], [False] * 3)
        for d in range(dim):
            e = row[d] // p
            elo, ehi = (e - 1 if row[d] % p == 0 and e > 0 else e), min(e, nel3[d] - 1)
            two[d], lo[d], ln[d] = elo != ehi, p * elo, p * (ehi - elo + 1) + 1
            el[d][0] = ehi if two[d] and elo & 1 else elo
            el[d][1] = elo + ehi - el[d][0]
            for t in range(2):
                il[d][t], po[d][t] = row[d] - p * el[d][t], p * (el[d][t] - elo)
            assert (lo[d], ln[d]) == axis_row(row[d], nel3[d], p)
        image = {}
        for k in range(1 << dim):
            bit = [k >> d & 1 for d in range(3)]
            if any(bit[d] and not two[d] for d in range(3)):
                continue
            ec = tuple(el[d][bit[d]] for d in range(3))
            assert all(0 <= il[d][bit[d]] <= p for d in range(dim))
            for jl in itertools.product(range(p1), range(p1), range(p1 if dim == 3 else 1)):
                slot = sum((jl[d] + po[d][bit[d]]) * m for d, m in enumerate((1, ln[0], ln[0] * ln[1])))
                col = tuple(p * ec[d] + jl[d] if d < dim else 0 for d in range(3))
                want = sum((col[d] - lo[d]) * m for d, m in enumerate((1, ln[0], ln[0] * ln[1])))
                assert slot == want
                image.setdefault(col, []).append(ec)
        colour = lambda e: (e[0] & 1) + 2 * (e[1] & 1) + 4 * (e[2] & 1)  # noqa: E731
        assert len(image) == ln[0] * ln[1] * ln[2]
        for col, els in image.items():
            near = [set(node_elems(c, nel3, p)) if dim == 3 else {e + (0,) for e in node_elems(c[:2], nel, p)}
                    for c in (row, col)]
            assert sorted(els) == sorted(near[0] & near[1]), (row, col)
            assert els == sorted(els, key=colour), (row, col, els)
