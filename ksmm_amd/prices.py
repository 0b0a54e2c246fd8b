"""Makes ``csrc/ksmm_cost.inc``, the prices the library chooses a kernel by where the measured table does
not apply (small and medium batches, ragged ones): measures every kernel instance on drawn problems and fits the
model of ``csrc/ksmm_choose.hip`` to the times.

    python -m ksmm_amd.prices --measure OUT.json [--problems 400] [--seed 0] [--made-for] [--combos 0,1,2,3]   (on the GPU)
    python -m ksmm_amd.prices --fit A.json B.json ... --emit ksmm_amd/csrc/ksmm_cost.inc [--keep OLD.inc [--families 13,14,15]]
    python -m ksmm_amd.prices --check A.json ...          how good the choice by the present table is

A problem is a factor pattern, a batch, an element-type combination (0 = fp32, 1 = fp16, 2 = e4m3 -> fp16,
3 = e4m3 weights on fp16 input) and a layout.  Its instances are timed as launches of a HIP graph on one set of
buffers, the way a layer finds its input: just written.  A quarter of the problems is held back from the fit; what
is printed for them is the geometric mean of (time of the cheapest priced instance) / (time of the fastest).

``--keep`` leaves the prices that a table has as they are, and with them the choices among those instances, except
for the families named (0 .. 5 the tile sub-families, 13 generic, 14 wave, 15 row kernels); instances without one
get the fitted price.

Instances with fewer than ``ENOUGH`` measured problems get no price and are listed at the end of the file: they are
never offered, and only run where the measured table or a family's own choice names them.
"""
import argparse
import ctypes
import json
import math
import os
import random
import re
import sys
import time

import numpy as np

from . import _lib
from .kernel import _COMBO_DTYPES, variant_id

FAM_SPLIT, FAM_GENERIC, FAM_WAVE, FAM_ROWS = 5, 13, 14, 15
SIZE = {_lib.KSMM_F32: 4, _lib.KSMM_F16: 2, _lib.KSMM_FP8_E4M3: 1}
ENOUGH = 12  # problems a price is fitted to
TERMS = 9
MOST = 1 << 27  # elements of a problem's input or output
ROW = re.compile(r"^\{(\d+), (\d+), (\d+), (\d+)u, \{([^}]*)\}\}")


# ---- problems ---------------------------------------------------------------------------------------------------
def draw(rng, made_for=False):
    """(a, b, c, d, batch): blocks from a few elements to 1536, aspect ratios and strides of layers, a third of them
    (made_for: all) blocks that kernels are made for; batches of 1 to 16384 rows, half of them whole vectors."""
    while True:
        kind = 0.3 if made_for else rng.random()
        if kind < 0.15:  # small blocks
            b, c = rng.choice((1, 2, 4, 6, 8, 12, 16, 24)), rng.choice((1, 2, 4, 8, 12, 16, 24))
            a, d = int(2 ** rng.uniform(0, 10)), int(2 ** rng.uniform(0, 7))
        elif kind < 0.5:
            b, c = rng.choice(((16, 16), (32, 32), (48, 48), (64, 64), (96, 96), (128, 128), (192, 192), (48, 192), (192, 48)))
            a, d = rng.choice((1, 2, 4, 8, 16, 32, 64)), rng.choice((1, 1, 2, 3, 4, 6, 8, 12, 16, 32, 64))
        else:
            side = rng.choice((16, 16, 32, 48, 48, 64, 64, 96, 128, 192, 256, 384))
            b, c = rng.choice(((side, side), (side, side), (4 * side, side), (side, 4 * side), (2 * side, side), (side, 2 * side)))
            if rng.random() < 0.12:
                b += rng.randint(1, 15)
            elif rng.random() < 0.08:
                c += rng.randint(1, 15)
            a, d = rng.choice((1, 1, 2, 3, 4, 6, 12, 16)), rng.choice((1, 1, 2, 3, 4, 6, 8, 12, 16, 32, 64))
        batch = int(round(2 ** rng.uniform(0, 14)))
        if rng.random() < 0.5:
            batch = max(1, batch // 16) * 16
        widest = a * d * max(b, c)
        if 16 <= widest <= 24576 and max(b, c) <= 1536 and a * b * c * d <= 1 << 24 and widest * batch <= MOST:
            return a, b, c, d, batch


def instances(combo, bs_last):
    """(family, id, algo, variant) of everything that may be priced."""
    def count(algo, make):
        n = 0
        while True:
            try:
                variant_id(algo, make(n), combo, bs_last)
            except _lib.KsmmError:
                return n
            n += 1

    out = [(FAM_GENERIC, v, _lib.ALGO_GENERIC, v) for v in (0, 1)]
    first = 0 if bs_last else 1000
    out += [(FAM_WAVE if bs_last else FAM_ROWS, variant_id(2, first + i, combo, bs_last)[0], 2, first + i)
            for i in range(count(2, lambda i: first + i))]
    for sub in range(6):
        def make(i, sub=sub):
            return (sub << 24) | i
        for i in range(count(3, make)):
            iid = variant_id(3, make(i), combo, bs_last)[0]
            for w in ((1, 2, 4, 8, 16) if sub == FAM_SPLIT else (0,)):
                out.append((sub, iid, 3, make(i) | (w << 8)))
    return out


def query(problem, combo, bs_last, algo, variant):
    """The tile the library reports, or None where it refuses."""
    t = _lib.KsmmTile()
    a, b, c, d, batch = problem
    rc = _lib.load().ksmm_query_tile_variant(batch, a, b, c, d, *_COMBO_DTYPES[combo], int(bs_last), algo, variant, ctypes.byref(t))
    return t if rc == 0 else None


def features(problem, combo, bs_last, family, t):
    """The terms of the model (csrc/ksmm_choose.hip, price())."""
    a, b, c, d, batch = problem
    ex, ew, ey = (SIZE[v] for v in _COMBO_DTYPES[combo])
    up = lambda p, q: -(-p // q)
    blocks = up(a * d, t.tile_d) if family == FAM_ROWS else a * (d // t.tile_d)
    groups = blocks * up(b, t.tile_m) * up(batch, t.tile_n)
    s, cu = float(up(c, t.tile_k)), up(groups, 256)
    if family == FAM_SPLIT:
        ks = t.threads // 64
        s, cu = float(up(int(s), ks)), up(groups * ks, 1024)
    elif family in (FAM_WAVE, FAM_ROWS):
        waves = t.grid * (t.threads // 64)
        s = t.tile_m * t.tile_n * t.tile_d * c / 65536. * up(groups, waves if family == FAM_WAVE else t.grid)
        cu = up(waves, 1024)
    elif family == FAM_GENERIC:
        s, cu = c / 8., up(t.grid, 256)
    by = (batch * a * d * (c * ex + b * ey) + a * d * b * c * ew) / 5e6
    w = 1.
    if not bs_last and t.tile_d < d:
        w = max(1., min(d * ex, 64.) / (t.tile_d * ex))
    return [1., s, cu * s, s * w, cu * s * w, float(cu), by, by * w, max(0., by - 25.)]


# ---- measuring --------------------------------------------------------------------------------------------------
class Clock:
    """Time of one launch: launches of a graph on one set of buffers."""

    def __init__(self, combo):
        import torch

        self.torch, self.lib = torch, _lib.load()
        xd, wd, yd = _COMBO_DTYPES[combo]
        types = {_lib.KSMM_F32: torch.float32, _lib.KSMM_F16: torch.float16, _lib.KSMM_FP8_E4M3: torch.float8_e4m3fn}
        rand = lambda n, dt: torch.randn(n, device="cuda", dtype=torch.float16).to(types[dt])
        self.x, self.w = rand(MOST, xd), rand(1 << 24, wd)
        self.y = torch.empty(MOST, device="cuda", dtype=types[yd])
        self.dtypes = _COMBO_DTYPES[combo]
        self.stream = torch.cuda.Stream()

    def __call__(self, problem, bs_last, algo, variant, best):
        a, b, c, d, batch = problem
        assert max(b, c) * a * d * batch <= MOST and a * b * c * d <= self.w.numel()
        cuda, s = self.torch.cuda, self.stream
        args = (self.x.data_ptr(), self.w.data_ptr(), self.y.data_ptr(), batch, a, b, c, d, *self.dtypes, int(bs_last), 1.0,
                algo, variant, ctypes.c_void_p(s.cuda_stream))

        def launch(n):
            for _ in range(n):
                _lib.check(self.lib.ksmm_factor_forward_algo(*args))

        t0, t1 = cuda.Event(enable_timing=True), cuda.Event(enable_timing=True)
        with cuda.stream(s):
            launch(1)
            t0.record(s)
            launch(1)
            t1.record(s)
            s.synchronize()
            once = t0.elapsed_time(t1) * 1e3
            if once > 20 * best + 100:  # out of the question: a rough time will do
                return once
            n = int(min(20, max(4, 400 / once)))
            graph = cuda.CUDAGraph()
            graph.capture_begin()
            launch(n)
            graph.capture_end()
            times = []
            graph.replay()
            for _ in range(3):
                t0.record(s)
                graph.replay()
                t1.record(s)
                s.synchronize()
                times.append(t0.elapsed_time(t1) * 1e3 / n)
        return min(times)


def measure(path, combos, problems, seed, made_for):
    out, t_start = [], time.time()
    for combo in combos:
        clock = Clock(combo)
        for bs_last in (True, False):
            insts, rng = instances(combo, bs_last), random.Random("%d %d %d" % (seed, combo, bs_last))
            for k in range(problems):
                problem = draw(rng, made_for)
                times, seen, best = [], set(), 1e30
                for family, iid, algo, variant in insts:
                    t = query(problem, combo, bs_last, algo, variant)
                    if t is None or (t.algo, t.variant) in seen:
                        continue
                    seen.add((t.algo, t.variant))
                    us = clock(problem, bs_last, algo, variant, best)
                    best = min(best, us)
                    times.append((family, iid, algo, t.variant, round(us, 3)))
                out.append({"combo": combo, "bs_last": bs_last, "problem": problem, "times": times})
                if k % 50 == 49:
                    print("combo %d bs_last %d: %d problems, %.0f s" % (combo, bs_last, k + 1, time.time() - t_start), flush=True)
            with open(path, "w") as f:
                json.dump(out, f)
        del clock
    return out


def load(paths):
    """Entries of measured files, with the terms of each instance as the library reports it now, and whether
    it is among those the choice is made from: of the wave and row kernels the family's own choice, of the
    generic ones that of full batches, if it is one."""
    entries = [e for p in paths for e in json.load(open(p))]
    for e in entries:
        problem, times = tuple(e["problem"]), []
        own = query(problem, e["combo"], e["bs_last"], _lib.ALGO_WAVE, -1)
        full = query(problem[:4] + (16384 + problem[4] % 16,), e["combo"], e["bs_last"], _lib.ALGO_AUTO, -3)
        for family, iid, algo, variant, us in e["times"]:
            t = query(problem, e["combo"], e["bs_last"], algo, variant)
            if family == FAM_GENERIC:
                offered = full is not None and full.algo == _lib.ALGO_GENERIC and (full.variant == 1) == (variant == 1)
            else:
                offered = family < FAM_GENERIC or (own is not None and own.variant == variant)
            times.append((family, iid, us, features(problem, e["combo"], e["bs_last"], family, t), offered))
        e["times"] = times
    return entries


# ---- fitting ----------------------------------------------------------------------------------------------------
def nnls(A, y, sweeps=3000):
    """argmin |A f - y| over f >= 0, by coordinate descent."""
    G, h = A.T @ A, A.T @ y
    f = np.zeros(A.shape[1])
    for _ in range(sweeps):
        before = f.copy()
        for i in range(len(f)):
            if G[i, i] > 0:
                f[i] = max(0., f[i] + (h[i] - G[i] @ f) / G[i, i])
        if np.abs(f - before).max() <= 1e-9 * (1 + f.max()):
            break
    return f


def held_back(entry):
    return sum(entry["problem"]) % 4 == 0


def fit(entries, whole=True):
    """{(family, combo, bs_last, id): coefficients}: relative errors weigh the same."""
    data = {}
    for e in entries:
        if not whole and held_back(e):
            continue
        for family, iid, us, v, offered in e["times"]:
            if family == FAM_GENERIC and not offered:
                continue  # (large blocks on these kernels say little about the small ones they run on)
            data.setdefault((family, e["combo"], int(e["bs_last"]), iid), []).append((us, v))
    rows = {}
    for key, samples in data.items():
        if len(samples) < ENOUGH:
            continue
        us = np.array([s[0] for s in samples])
        A = np.array([s[1] for s in samples]) / us[:, None]
        top = A.max(axis=0)
        top[top == 0] = 1.
        rows[key] = nnls(A / top, np.ones(len(us))) / top
    return rows


def read(path):
    rows = {}
    for line in open(path):
        m = ROW.match(line)
        if m:
            terms = [float(v.rstrip("f")) for v in m.group(5).split(", ")]
            rows[tuple(int(g) for g in m.groups()[:4])] = np.array(terms + [0.] * (TERMS - len(terms)))
    return rows


def unpriced(rows):
    """(sub-family, id) of the instances of the library no row prices, in any combination or layout."""
    have = {(k[0], k[3]) for k in rows}
    every = {(f, i) for combo in range(4) for last in (True, False) for f, i, _, _ in instances(combo, last)}
    return sorted(every - have)


def emit(rows, path):
    def num(v):
        text = "%.4g" % (v if v >= 1e-6 else 0.)
        return text + ("f" if "." in text or "e" in text else ".f")

    with open(path, "w") as f:
        f.write("// Generated by `python -m ksmm_amd.prices` on MI355X (gfx950): microseconds per term of the model in\n"
                "// ksmm_choose.hip.  {family, combo, bs_last, instance id, {terms}}\n")
        for key in sorted(rows):
            f.write("{%d, %d, %d, %du, {%s}},\n" % (*key, ", ".join(num(v) for v in rows[key])))
        for family, iid in unpriced(rows):
            f.write("// no price: %d %du\n" % (family, iid))


def choice(entry, rows):
    """Time of the instance the prices choose, of the fastest one."""
    best = None
    for family, iid, us, v, offered in entry["times"]:
        f = rows.get((family, entry["combo"], int(entry["bs_last"]), iid)) if offered else None
        if f is not None and (best is None or f @ np.array(v) < best[0]):
            best = (f @ np.array(v), us)
    return best and best[1], min(t[2] for t in entry["times"])


def check(entries, rows, only=held_back):
    """Geometric means of chosen / fastest by combination and layout."""
    groups = {}
    for e in entries:
        if only(e):
            got, fastest = choice(e, rows)
            groups.setdefault((e["combo"], e["bs_last"]), []).append(got / fastest if got else math.nan)
    for key in sorted(groups):
        r = np.array(groups[key])
        ok = r[~np.isnan(r)]
        print("combo %d bs_last %d: %4d problems, chosen / fastest %.3f (90th percentile %.2f, largest %.2f), without a price %d" % (
            key[0], key[1], len(r), np.exp(np.log(ok).mean()), np.percentile(ok, 90), ok.max(), len(r) - len(ok)))


def main():
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("--measure")
    ap.add_argument("--problems", type=int, default=400, help="per combination and layout")
    ap.add_argument("--seed", type=int, default=0)
    ap.add_argument("--made-for", action="store_true", help="only blocks that kernels are made for")
    ap.add_argument("--combos", default="0,1,2,3")
    ap.add_argument("--fit", nargs="*")
    ap.add_argument("--emit")
    ap.add_argument("--keep", help="a table whose prices stay")
    ap.add_argument("--families", default="", help="families that --keep does not hold for")
    ap.add_argument("--check", nargs="*")
    args = ap.parse_args()
    if args.measure:
        measure(args.measure, [int(c) for c in args.combos.split(",")], args.problems, args.seed, args.made_for)
    if args.fit:
        entries = load(args.fit)
        again = {int(f) for f in args.families.split(",") if f}
        kept = {k: f for k, f in read(args.keep).items() if k[0] not in again} if args.keep else {}
        check(entries, {**fit(entries, whole=False), **kept})
        rows = {**fit(entries), **kept}
        print("%d prices, %d instances without one" % (len(rows), len(unpriced(rows))))
        if args.emit:
            emit(rows, args.emit)
    if args.check:
        check(load(args.check), read(os.path.join(os.path.dirname(__file__), "csrc", "ksmm_cost.inc")),
              only=lambda e: True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
