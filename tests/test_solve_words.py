"""The pipelined solve's word exchanges on quads, as a model on the CPU that runs by the kernels' own
rules (natray_faces.h, compiled for the host): no order of its waves' steps loses a word.

A replacement of the residual makes four exchanges (x, u, p, q) over two word buffers with no
reduction between them. A word that is written over before its reader has seen it never comes again,
so the model walks through every order the waves can run in and looks for one in which no wave can go
on. With waits for the water cells' words alone there is one (a dry block beside a wet one), which
shows that the model finds such faults.
"""
import ctypes as C
import itertools
import subprocess

import numpy as np
import pytest

from natray_amd.build import CSRC, HIPCC

SOURCE = r"""
#include "natray_faces.h"
using namespace natray;
// Lane `ln` of a set: its links as blocks, face flags and words (out: x, y, m, p links, flags,
// exchange's wants, a reduction's wants, faces published in an exchange and beside a reduction).
extern "C" void lane_rules(const uint32_t* nbm, const uint32_t* block_nb, uint32_t b, uint32_t b0, uint32_t b1, uint32_t ln,
                           uint32_t* out) {
  const QuadLane l = quad_lane(ln);
  uint32_t nb[6];
  for (int f = 0; f < 6; ++f) {
    const uint32_t n = block_nb[6 * b + f];
    nb[f] = n == QUAD_NONE ? QUAD_NONE : (n >= b0 && n < b1 ? n - b0 : n | QUAD_FAR);
  }
  const QuadLinks k = {l.x3 ? nb[0] : (l.x0 ? nb[1] : QUAD_NONE), l.y3 ? nb[2] : (l.y0 ? nb[3] : QUAD_NONE), nb[4], nb[5]};
  const uint32_t w = quad_flags(nbm, nb, k, l, b0), links[4] = {k.x, k.y, k.m, k.p};
  for (int f = 0; f < 4; ++f)
    out[f] = links[f] == QUAD_NONE ? QUAD_NONE : ((links[f] & QUAD_FAR) ? links[f] & ~QUAD_FAR : b0 + links[f]);
  out[4] = w;
  out[5] = quad_exchange(k);
  out[6] = quad_want(w, false);
  out[7] = quad_want(w, true);
  out[8] = quad_faces(w, false);
  out[9] = quad_faces(w, true);
}
"""
NONE = 0xFFFFFFFF


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("words")
    src, lib = d / "rules.cpp", d / "rules.so"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-shared", f"-I{CSRC}", str(src),
                    "-o", str(lib)], check=True)
    fn = C.CDLL(str(lib)).lane_rules
    fn.restype = None

    def lane(nbm, nb, b, b0, b1, ln):
        out = (C.c_uint32 * 10)()
        fn(nbm.ctypes.data_as(C.c_void_p), nb.ctypes.data_as(C.c_void_p), b, b0, b1, ln, out)
        return list(out)

    return lane


def layout(coords, water):
    """Blocks in slot order (z fastest): Dev::nbm's water bit per cell and each block's face
    neighbours. water(x, y, z): whether the cell at these global coordinates is water."""
    coords = sorted(coords)
    at = {c: k for k, c in enumerate(coords)}
    nb = np.full((len(coords), 6), NONE, np.uint32)
    nbm = np.zeros((len(coords), 64), np.uint32)
    for k, c in enumerate(coords):
        for f in range(6):
            o = list(c)
            o[f // 2] += 1 if f & 1 else -1
            nb[k, f] = at.get(tuple(o), NONE)
        for i in range(64):
            if water(4 * c[0] + i // 16, 4 * c[1] + i // 4 % 4, 4 * c[2] + i % 4):
                nbm[k, i] = 64
    return nb, nbm


def words(lane, nb, nbm, groups):
    """Per wave of four blocks: the words it publishes, {(block, face, cell)}, and those it waits
    for, in an exchange and (with other workgroups) beside a reduction, and the water cells' words
    of an exchange. groups: each workgroup's blocks [b0, b1)."""
    waves = []
    for b0, b1 in groups:
        for first in range(b0, b1, 4):
            w = {"pub": set(), "pub_far": set(), "all": set(), "water": set(), "far": set()}
            for ln in range(64):
                b, col = first + ln // 16, ln % 16
                if b >= b1:
                    continue
                x, y = col // 4, col % 4
                o = lane(nbm, nb, b, b0, b1, ln)
                # The words of this lane's four halo links, by their bits.
                read = {}
                if o[0] != NONE:
                    read.update({z: (o[0], 1 if x == 3 else 0, 4 * y + z) for z in range(4)})
                if o[1] != NONE:
                    read.update({4 + z: (o[1], 3 if y == 3 else 2, 4 * x + z) for z in range(4)})
                if o[2] != NONE:
                    read[8] = (o[2], 5, col)
                if o[3] != NONE:
                    read[9] = (o[3], 4, col)
                for name, want in (("all", o[5]), ("water", o[6]), ("far", o[7])):
                    for bit in range(10):
                        if want >> bit & 1:
                            w[name].add(read[bit])  # KeyError: a word of a block that is not there
                own = [[(b, 1 if x == 3 else 0, 4 * y + z) for z in range(4)], [(b, 3 if y == 3 else 2, 4 * x + z) for z in range(4)],
                       [(b, 4, col)], [(b, 5, col)]]
                for name, faces in (("pub", o[8]), ("pub_far", o[9])):
                    for f in range(4):
                        if faces >> f & 1:
                            w[name].update(own[f])
            waves.append(w)
    return waves


def program(w, rule, iterations):
    """A wave's steps: ("pub", buffer, tag, words), ("wait", buffer, tag, words), ("sum", t): the
    workgroup's share of reduction t, ("total", t, buffer, tag, words): everyone's shares and the
    halo's m."""
    out = []
    for t in range(1, iterations + 1):
        a, b = t & 1, (t + 1) & 1
        out += [("sum", t), ("pub", a, 8 * t, w["pub_far"]), ("total", t, a, 8 * t, w["far"])]
        for k, buf in ((1, b), (2, a), (3, b), (4, a)):
            out += [("pub", buf, 8 * t + k, w["pub"]), ("wait", buf, 8 * t + k, w[rule])]
    return out


def stuck(waves, rule, iterations=2):
    """An order of the waves' steps after which none can go on though not all have ended, or None.
    What a word holds follows from how far its owner has run."""
    progs = [program(w, rule, iterations) for w in waves]
    n = len(waves)
    owner = {}
    for k, w in enumerate(waves):
        for x in w["pub"]:
            owner[x] = k
    # last[k][pc]: what wave k's words hold there, {(buffer, word): tag}.
    last = [[{} for _ in range(len(p) + 1)] for p in progs]
    for k, p in enumerate(progs):
        cur = {}
        for pc, op in enumerate(p):
            last[k][pc] = dict(cur)
            if op[0] == "pub":
                for x in op[3]:
                    cur[op[1], x] = op[2]
        last[k][len(p)] = dict(cur)

    def there(buf, tag, want, pcs):
        return all(last[owner[x]][pcs[owner[x]]].get((buf, x)) == tag for x in want)

    # Words are many and waits few: a wait's answer depends on the owners' places alone.
    memo = {}

    def can(k, pcs):
        op = progs[k][pcs[k]]
        if op[0] in ("pub", "sum"):
            return True
        if op[0] == "total":
            t, buf, tag, want = op[1:]
            at = next(i for i, o in enumerate(progs[k]) if o[0] == "sum" and o[1] == t)
            if any(pc <= at for pc in pcs):
                return False
        else:
            buf, tag, want = op[1:]
        owners = tuple(sorted({owner[x] for x in want}))
        key = (k, pcs[k], tuple(pcs[o] for o in owners))
        if key not in memo:
            memo[key] = there(buf, tag, want, pcs)
        return memo[key]

    # (A workgroup's own barriers are left out: that only adds orders.)
    def steps(pcs):
        for k in range(n):
            if pcs[k] < len(progs[k]) and can(k, pcs):
                yield pcs[:k] + (pcs[k] + 1,) + pcs[k + 1:]

    seen, todo = {(0,) * n}, [(0,) * n]
    end = tuple(len(p) for p in progs)
    while todo:
        pcs = todo.pop()
        nxt = list(steps(pcs))
        if not nxt and pcs != end:
            return [(k, progs[k][pcs[k]][:3]) for k in range(n) if pcs[k] < len(progs[k])]
        for s in nxt:
            if s not in seen:
                seen.add(s)
                todo.append(s)
    return None


def ball(c, r):
    return lambda x, y, z: (x + 0.5 - c[0]) ** 2 + (y + 0.5 - c[1]) ** 2 + (z + 0.5 - c[2]) ** 2 < r * r


BOX = list(itertools.product(range(2), range(1), range(4)))  # eight blocks: two sets
TALL = list(itertools.product(range(3), range(1), range(4)))  # twelve: three sets


@pytest.mark.parametrize("groups", [[(0, 4), (4, 8)], [(0, 8)]])
def test_a_dry_block_beside_a_wet_one(rules, groups):
    """Water on one side of a face alone, in two workgroups and within one."""
    nb, nbm = layout(BOX, lambda x, y, z: x < 4)
    waves = words(rules, nb, nbm, groups)
    assert stuck(waves, "water") is not None
    assert stuck(waves, "all") is None


@pytest.mark.parametrize("coords,groups,water", [
    (BOX, [(0, 4), (4, 8)], lambda x, y, z: True),
    (BOX, [(0, 4), (4, 8)], ball((4, 2, 8), 5.0)),
    (TALL, [(0, 4), (4, 12)], lambda x, y, z: 4 <= x < 8),
    (TALL, [(0, 8), (8, 12)], ball((2, 2, 3), 3.7)),
    (TALL[:9] + TALL[10:], [(0, 5), (5, 11)], ball((6, 2, 6), 6.1)),
])
def test_no_order_loses_a_word(rules, coords, groups, water):
    """Wet and dry fringes, a block missing, sets that are not full (three waves, or four)."""
    nb, nbm = layout(coords, water)
    waves = words(rules, nb, nbm, groups)
    assert stuck(waves, "all", 2 if len(waves) < 4 else 1) is None


@pytest.mark.parametrize("seed", range(4))
def test_waits_are_mutual_and_published(rules, seed):
    """Random blocks and water: every word waited for is published by its owner, every word whose value
    is used is waited for, and a wave that waits for another's words is waited for by it."""
    rng = np.random.default_rng(seed)
    coords = [c for c in itertools.product(range(3), range(4), range(5)) if rng.random() < 0.8]
    wet = rng.random((12, 16, 20)) < rng.choice([0.05, 0.4])
    nb, nbm = layout(coords, lambda x, y, z: wet[x, y, z])
    n = len(coords)
    cuts = sorted(rng.choice(np.arange(1, n), 3, replace=False).tolist())
    waves = words(rules, nb, nbm, list(zip([0] + cuts, cuts + [n])))
    pub, pub_far = set().union(*(w["pub"] for w in waves)), set().union(*(w["pub_far"] for w in waves))
    owner = {x: k for k, w in enumerate(waves) for x in w["pub"]}
    for k, w in enumerate(waves):
        assert w["all"] <= pub and w["far"] <= pub_far and w["water"] <= w["all"]
        for o in {owner[x] for x in w["all"]} - {k}:
            assert any(owner[x] == k for x in waves[o]["all"])
