"""Where the Cholesky's workgroups go (no GPU needed): the map from launch index to role that the kernels use, and a model
of its dispatch. A factorisation's flag waits need all its workgroups resident at once, and the launches of two streams
share the XCDs' compute units in any interleaving, so every launch must be able to finish whatever part of the others is
resident."""
import ctypes
import random

import pytest

from spanqr_amd import _lib

NXCD, CUS = 8, 32   # XCDs, compute units of each (a workgroup's LDS leaves room for one per unit)


def workgroups(nb, w, first=4):
    """workgroups of one factorisation: workgroup 0 and the parts (of at most w tiles) of tile rows first..nb-1"""
    return 1 + sum((i + w) // w for i in range(first, nb))


def launch(grid, nz, m, slot, solves):
    """the roles by launch index: ('one', z, b), ('spread', z, b), ('solve', rank) or None, up to the index after which
    no role is left"""
    out, idx, want = [], 0, (2 if m == NXCD else 1) * nz * grid + solves
    three = (ctypes.c_int * 3)()
    while want:
        _lib.check(_lib.lib().spanqr_debug_chol_role(idx, grid, nz, m, slot, three))
        b, z, local = three
        role = ("one" if local else "spread", z, b) if b >= 0 else ("solve", z) if z < solves else None
        want -= role is not None
        out.append(role)
        idx += 1
        assert idx < 64 * (2 * nz * grid + solves + 8), "roles missing"
    return out


LAUNCHES = [(7, 1, 218), (7, 1, 16), (27, 1, 48), (27, 1, 128), (30, 1, 0), (32, 1, 0), (29, 1, 0), (1, 1, 3),
            (27, 2, 96), (24, 7, 0), (28, 7, 0), (28, 8, 0), (13, 12, 0), (13, 16, 0), (7, 17, 0), (3, 32, 90),
            (31, 5, 0)]


@pytest.mark.parametrize("grid,nz,solves", LAUNCHES)
def test_every_role_once_and_in_order(grid, nz, solves):
    for m, slots in ((NXCD, range(NXCD)), (1, [0])):
        for slot in slots:
            roles = launch(grid, nz, m, slot, solves)
            real = [r for r in roles if r is not None]
            want = {("spread", z, b) for z in range(nz) for b in range(grid)} | {("solve", i) for i in range(solves)}
            if m == NXCD:
                want |= {("one", z, b) for z in range(nz) for b in range(grid)}
            assert len(real) == len(set(real)) and set(real) == want
            for x in range(NXCD):
                mine = [r for r in roles[x::NXCD] if r is not None]
                kinds = ["one", "spread", "solve"]
                assert [r[0] for r in mine] == sorted((r[0] for r in mine), key=kinds.index)
                assert all((r[1] + slot) % NXCD == x for r in mine if r[0] == "one")
                # the spread set needs no more of any XCD than an even share
                assert sum(r[0] == "spread" for r in mine) <= -(-nz * grid // NXCD)


def finishes(launches, rng, spread_set=True):
    """Dispatch the launches (role lists) with an adversary's choices: each XCD starts any launch's next workgroup where a
    unit is free. A factorisation runs on one XCD if that set is resident before anyone settles for spread. True if all
    workgroups end."""
    pend = [[[r for r in roles[x::NXCD] if r is not None and (spread_set or r[0] != "spread")] for x in range(NXCD)]
            for roles in launches]
    place, done = {}, set()                # (launch, z) -> 'one' / 'spread'; factorisations that have ended
    need = [{} for _ in launches]          # workgroups of one set of matrix z
    for a, roles in enumerate(launches):
        sets = {r[0] for r in roles if r is not None}
        for r in roles:
            if r is not None and r[0] == ("one" if "one" in sets else "spread"):
                need[a][r[1]] = need[a].get(r[1], 0) + 1
                if "one" not in sets:
                    place[a, r[1]] = "spread"
    held = [[] for _ in range(NXCD)]       # (launch, role) resident

    def settle():
        moved = True
        while moved:
            moved = False
            for a in range(len(launches)):
                for z, n in need[a].items():
                    have = {s: sum(r[:2] == (s, z) for x in held for l, r in x if l == a) for s in ("one", "spread")}
                    if (a, z) not in place and have["one"] == n:
                        place[a, z] = "one"
                    if (a, z) not in done and (a, z) in place and have[place[a, z]] == n:
                        done.add((a, z))
                        moved = True
            for x in range(NXCD):
                def ends(l, r):
                    if r[0] == "solve":
                        return all((l, z) in done for z in need[l])
                    return (l, r[1]) in done or ((l, r[1]) in place and place[l, r[1]] != r[0])
                keep = [(l, r) for l, r in held[x] if not ends(l, r)]
                moved |= len(keep) != len(held[x])
                held[x] = keep

    while True:
        settle()
        can = [(a, x) for a in range(len(launches)) for x in range(NXCD) if pend[a][x] and len(held[x]) < CUS]
        if can:
            # runs of one launch on one XCD, so that the launches fill different XCDs first
            a, x = rng.choice(can)
            for _ in range(rng.choice((1, 4, CUS))):
                if pend[a][x] and len(held[x]) < CUS:
                    held[x].append((a, pend[a][x].pop(0)))
            continue
        if not any(pend[a][x] for a in range(len(launches)) for x in range(NXCD)) and not any(held):
            return True
        # nothing moves: any resident workgroup of an undecided factorisation settles for spread when its time is up
        late = [(l, r[1]) for x in held for l, r in x if r[0] != "solve" and (l, r[1]) not in place]
        if not spread_set or not late:
            return False
        place[rng.choice(late)] = "spread"


# grid and solves of 768x512, 2048x512, 17408x256, a 512- and a 608-column factorisation alone, the fp64 one of 512 columns
# and 608, and a batch of twelve 512-column factorisations
CALLS = [(27, 1, 48), (27, 1, 128), (7, 1, 218), (27, 1, 0), (30, 1, 0), (29, 1, 0), (32, 1, 0), (13, 12, 0)]


def test_grids_are_the_plans():
    assert [workgroups(16, 6), workgroups(8, 6), workgroups(19, 8), workgroups(16, 16)] == [27, 7, 30, 13]
    assert [workgroups(16, 6, 2), workgroups(19, 8, 2)] == [29, 32]


@pytest.mark.parametrize("a", range(len(CALLS)))
def test_two_streams_always_finish(a):
    for b in range(a, len(CALLS)):
        if CALLS[a][1] + CALLS[b][1] > 13:
            continue   # two batches: more workgroups than the device holds, in any placement
        for seed in range(12):
            rng = random.Random(1000 * a + 100 * b + seed)
            calls = [launch(*CALLS[i][:2], NXCD, rng.randrange(NXCD) if seed % 2 else 0, CALLS[i][2]) for i in (a, b)]
            assert finishes(calls, rng), (CALLS[a], CALLS[b], seed)


def test_three_streams_of_768x512_always_finish():
    for seed in range(12):
        rng = random.Random(seed)
        assert finishes([launch(27, 1, NXCD, rng.randrange(NXCD), 48) for _ in range(3)], rng), seed


def test_the_model_sees_the_starvation_without_the_spread_set():
    """two factorisations of 27 workgroups on the same XCD, each resident in part, and on XCDs of their own with the
    other's solve in the way"""
    for slots in ((0, 0), (0, 1)):
        assert not all(finishes([launch(27, 1, NXCD, s, 48) for s in slots], random.Random(seed), spread_set=False)
                       for seed in range(40)), slots


def test_two_of_the_widest_calls_must_be_ordered():
    """the limit that spanqr.h states: 2048x1024 beside itself (99 workgroups and 128 of the solve, always spread) may
    starve; beside a 768x512 call it does not"""
    wide, call = launch(workgroups(32, 6), 1, 1, 0, 128), launch(27, 1, NXCD, 0, 48)
    assert not all(finishes([wide, wide], random.Random(seed)) for seed in range(60))
    assert all(finishes([wide, call], random.Random(seed)) for seed in range(12))
