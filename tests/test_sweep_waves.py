"""Sweeps overlapped on up to eight waves: a CPU model of the protocol (wave s mod N
runs sweep s and waits on the wave before it), and on the GPU the overlapped steps
against sequential ones, bit for bit, with fixed iteration counts and in the residual
mode, whose waves keep velocities and impulses of their own, since sweeps run past the
one that ends the step."""
import os
import random
import subprocess

import numpy as np
import pytest

from dbox_amd import native, scenes
from tests.test_overlap_protocol import _levels

DT = 1.0 / 60.0


def _run(seed, waves, short=False):
    R = random.Random(seed)
    nb, n = R.randint(2, 30), R.randint(1, 60)
    cons = [(R.randrange(nb), R.randrange(nb), R.choice([1, 2, 3, 3, 3])) for _ in range(n)]
    lvl, llast = _levels(cons)
    N = max(lvl) + 1
    need = [0] * N
    for (a, b, dm), l in zip(cons, lvl):
        need[l] = max(need[l], llast[a] if dm & 1 else 0, llast[b] if dm & 2 else 0)
    if short:
        need = [max(x - 1, 0) for x in need]
    ns = R.randint(1, 20)
    levels = [[i for i in range(n) if lvl[i] == l] for l in range(N)]
    ref, got = {x: [] for x in range(nb)}, {x: [] for x in range(nb)}

    def level(s, l, out):
        for i in levels[l]:
            a, b, dm = cons[i]
            if dm & 1:
                out[a].append((s, i))
            if dm & 2:
                out[b].append((s, i))

    for s in range(ns):
        for l in range(N):
            level(s, l, ref)
    inf = 10 ** 9
    pub, pos = [0] * waves, [0] * waves
    plans = [[(s, l) for s in range(w, ns, waves) for l in range(N)] for w in range(waves)]
    while True:
        open_ = [w for w in range(waves) if pos[w] < len(plans[w])]
        if not open_:
            return None if got == ref else "order"
        ready = []
        for w in open_:
            s, l = plans[w][pos[w]]
            if s == 0 or pub[(w - 1) % waves] >= (s - 1) * N + need[l] + 1:
                ready.append(w)
        if not ready:
            return "deadlock"
        w = R.choice(ready)
        s, l = plans[w][pos[w]]
        level(s, l, got)
        pos[w] += 1
        pub[w] = s * N + l + 1 if l + 1 < N else ((s + waves) * N if s + waves < ns else inf)


@pytest.mark.parametrize("waves", [2, 3, 5, 8])
def test_protocol_keeps_every_body_in_order_and_finishes(waves):
    bad = [(k, r) for k in range(600) if (r := _run(k, waves))]
    assert not bad, bad[:5]
    assert sum(_run(k, waves, short=True) == "order" for k in range(300)) > 50


def _run_owned(seed, waves, shared=False):
    """The residual mode's protocol: every wave with values of its own, a sweep that ends the
    step, later ones that give up at random or not at all.  None when the values of the
    sweep that ends it are the sequential sweeps'."""
    R = random.Random(seed)
    nb, n = R.randint(2, 20), R.randint(1, 40)
    dyn = [True] + [R.random() < 0.8 for _ in range(nb - 1)]
    cons = []
    while len(cons) < n:
        a, b = R.randrange(nb), R.randrange(nb)
        if a != b and (dyn[a] or dyn[b]):
            cons.append((a, b, (1 if dyn[a] else 0) | (2 if dyn[b] else 0)))
    lvl, llast = _levels(cons)
    N = max(lvl) + 1
    need = [0] * N
    lfirst = {}
    for (a, b, dm), l in zip(cons, lvl):
        need[l] = max(need[l], llast[a] if dm & 1 else 0, llast[b] if dm & 2 else 0)
        for body, bit in ((a, 1), (b, 2)):
            if dm & bit:
                lfirst[body] = min(lfirst.get(body, N), l)
    ns = R.randint(1, 20)
    stops = sorted(R.sample(range(ns), R.randint(0, min(3, ns))))  # sweeps whose residual is small enough
    levels = [[i for i in range(n) if lvl[i] == l] for l in range(N)]
    base_v, base_i = [("v", b) for b in range(nb)], [("i", k) for k in range(n)]

    def solve(i, s, va, vb, im):
        return hash((va, vb, im, i)), hash((vb, va, im, -i - 1)), hash((im, va, vb, s))

    ref_v, ref_i = list(base_v), list(base_i)
    want = None
    for s in range(ns):
        for l in range(N):
            for i in levels[l]:
                a, b, dm = cons[i]
                va, vb, im = solve(i, s, ref_v[a], ref_v[b], ref_i[i])
                ref_i[i] = im
                if dm & 1:
                    ref_v[a] = va
                if dm & 2:
                    ref_v[b] = vb
        want = (s, list(ref_v), list(ref_i))
        if s in stops:
            break
    vel = [[("?", w, b) for b in range(nb)] for w in range(waves)]
    imp = [[("?", w, k) for k in range(n)] for w in range(waves)]
    if shared:  # one set of values for all waves
        vel, imp = [list(base_v)] * waves, [list(base_i)] * waves
    inf, stop = 10 ** 9, 10 ** 9
    pub, at = [0] * waves, [(w, 0) if w < ns else None for w in range(waves)]
    while any(x is not None for x in at):
        ready = [w for w in range(waves) if at[w] and (at[w][0] == 0 or at[w][0] > stop or
                                                       pub[(w - 1) % waves] >= (at[w][0] - 1) * N + need[at[w][1]] + 1)]
        if not ready:
            return "deadlock"
        w = R.choice(ready)
        s, l = at[w]
        if s > stop and (R.random() < 0.5 or not pub[(w - 1) % waves] >= (s - 1) * N + need[l] + 1):
            at[w], pub[w] = None, inf  # gives up
            continue
        p = (w - 1) % waves
        for i in levels[l]:
            a, b, dm = cons[i]

            def body(x, bit):
                if not dm & bit:
                    return base_v[x]
                if lfirst[x] < l:
                    return vel[w][x]
                return base_v[x] if s == 0 else vel[p][x]

            va, vb, im = solve(i, s, body(a, 1), body(b, 2), base_i[i] if s == 0 else imp[p][i])
            imp[w][i] = im
            if dm & 1:
                vel[w][a] = va
            if dm & 2:
                vel[w][b] = vb
        if l + 1 < N:
            at[w], pub[w] = (s, l + 1), s * N + l + 1
            continue
        if s in stops:
            stop = min(stop, s)
        more = s + waves < ns and s not in stops
        at[w], pub[w] = ((s + waves, 0), (s + waves) * N) if more else (None, inf)
    last = min(stop, ns - 1)
    got_v = [vel[last % waves][b] if b in llast else base_v[b] for b in range(nb)]
    return None if (last, got_v, imp[last % waves]) == want else "values"


@pytest.mark.parametrize("waves", [2, 3, 4, 8])
def test_residual_protocol_ends_with_the_values_of_the_sweep_that_ends_it(waves):
    bad = [(k, r) for k in range(600) if (r := _run_owned(k, waves))]
    assert not bad, bad[:5]
    assert sum(_run_owned(k, waves, shared=True) == "values" for k in range(300)) > 50


RULES = """#include <cstdio>
#include <cstdlib>
#include "%s"
int main(int, char **v) {
    const int levels = atoi(v[1]), lag = atoi(v[2]);
    for (int most = 2; most <= 8; ++most)
        for (int always = 0; always < 2; ++always) {
            // the largest sweep count that still overlaps, by bisection over dbx_step's range
            long long lo = 1, hi = (1ll << 31) + 1;
            while (hi - lo > 1) {
                const long long mid = (lo + hi) / 2;
                (dbx::far_waves(mid, most, lag, levels, always) > 0 ? lo : hi) = mid;
            }
            printf("%%d %%lld %%d %%d\\n", most, lo, dbx::far_waves(lo, most, lag, levels, always),
                   dbx::far_waves((1ll << 31) - 1, most, lag, levels, always));
        }
}
"""


@pytest.mark.parametrize("levels,lag", [(2, 2), (59, 4), (2371, 1518), (3017, 900), (60000, 2), (1 << 22, 5)])
def test_overlap_rule_keeps_the_progress_count_in_an_int(levels, lag, tmp_path):
    header = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dbox_amd", "csrc", "dbx_sweeps.h")
    src, exe = tmp_path / "rules.cpp", tmp_path / "rules"
    src.write_text(RULES % header)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe), str(levels), str(lag)], capture_output=True, text=True, check=True).stdout
    overlapped = 0
    for most, sweeps, waves, at_limit in (map(int, ln.split()) for ln in out.splitlines()):
        assert at_limit == 0 and waves <= most
        # the largest value published, the start of a sweep past the last, and the largest waited for
        assert (sweeps + waves) * levels + levels < 2 ** 31
        overlapped += waves > 0
    assert overlapped or lag >= levels


def _handles(ws):
    out = {}
    for m in ("default", "always", "sequential"):
        h = native.StepWorlds()
        for s in ws:
            h.add_scene(s)
        h.finalize()
        out[m] = h
    return out


ENV = {"default": {}, "always": {"DBX_SWEEPS_OVERLAP_ALWAYS": "1"}, "sequential": {"DBX_SWEEPS_SEQUENTIAL": "1"}}


def _step(hs, monkeypatch, vel, pos, flags):
    for m, env in ENV.items():
        for var in ("DBX_SWEEPS_OVERLAP_ALWAYS", "DBX_SWEEPS_SEQUENTIAL"):
            monkeypatch.delenv(var, raising=False)
        for var, val in env.items():
            monkeypatch.setenv(var, val)
        hs[m].step(DT, vel, pos, flags)


def _same(hs, label):
    for w in range(hs["sequential"].world_count):
        for m in ("default", "always"):
            assert hs[m].bodies(w).tobytes() == hs["sequential"].bodies(w).tobytes(), f"{label}, {m}, world {w}: bodies"
            assert hs[m].contacts(w).tobytes() == hs["sequential"].contacts(w).tobytes(), f"{label}, {m}, world {w}"


def _worlds():
    return ([scenes.stacks_world(k) for k in range(6)] + [scenes.pyramid(n, seed=n) for n in (1, 2, 3, 9, 20)] +
            [scenes.mixed_container(n, 14.0, 30.0, n) for n in (8, 60, 250)] + [scenes.hello_world()])


@pytest.mark.gpu
@pytest.mark.parametrize("vel,pos,warm", [(8, 3, True), (8, 3, False), (1, 3, True), (20, 2, True), (0, 3, True)])
def test_overlapped_sweeps_equal_sequential(vel, pos, warm, monkeypatch):
    print(f"case: sweeps on several waves, {vel} / {pos} iterations, warm {warm}", flush=True)
    hs = _handles(_worlds())
    flags = native.SLEEP | native.ORDERED | (native.WARM if warm else 0)
    for i in range(90):
        _step(hs, monkeypatch, vel, pos, flags)
        if i % 30 == 29:
            _same(hs, f"step {i + 1}")


@pytest.mark.gpu
@pytest.mark.parametrize("pos", [0, 2, 4])
def test_overlapped_residual_sweeps_at_other_position_iterations(pos, monkeypatch):
    print(f"case: residual sweeps on several waves, {pos} position iterations", flush=True)
    hs = _handles(_worlds())
    for h in hs.values():
        h.set_residual(1e-2, 40)
    for i in range(24):
        _step(hs, monkeypatch, 8, pos, native.WARM | native.SLEEP | native.ORDERED | native.RESIDUAL)
        its = {m: h.solver_stats()[0] for m, h in hs.items()}
        for m in ("default", "always"):
            assert np.array_equal(its[m], its["sequential"]), (i, m)
    _same(hs, "step 24")


@pytest.mark.gpu
@pytest.mark.parametrize("tol,most", [(1e-3, 100), (1e-1, 13), (1e-3, 1), (-1.0, 8), (-1.0, 9), (-1.0, 17), (1e9, 50)])
def test_overlapped_residual_sweeps_equal_sequential(tol, most, monkeypatch):
    print(f"case: residual sweeps on several waves, tolerance {tol}, at most {most}", flush=True)
    hs = _handles(_worlds())
    for h in hs.values():
        h.set_residual(tol, most)
    flags = native.WARM | native.SLEEP | native.ORDERED | native.RESIDUAL
    seen = set()
    for i in range(40):
        _step(hs, monkeypatch, 8, 3, flags)
        its = {m: h.solver_stats()[0] for m, h in hs.items()}
        res = {m: h.residuals() for m, h in hs.items()}
        for m in ("default", "always"):
            assert np.array_equal(its[m], its["sequential"]) and res[m].tobytes() == res["sequential"].tobytes(), (i, m)
        seen |= set(its["sequential"].tolist())
        if i % 20 == 19:
            _same(hs, f"step {i + 1}")
    if tol == 1e-3 and most == 100:
        assert len(seen) > 8  # ends on every wave
