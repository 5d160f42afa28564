"""The plan rule of csrc/api.hip against measured candidates: what its picks cost, its constants fitted anew, and the
range rows of the plan table. Reads the candidate times that `tune.py --data` writes (CSV: kind, N, K, M, tile, splitk,
one_launch, us; kind | 4 = packed weights). Needs no GPU.

    python open-jev-fast_amd/planfit.py DATA.csv [DATA.csv ...]       # costs of the plan rule and of the plan table
    python open-jev-fast_amd/planfit.py DATA.csv --fit [--rule-out open-jev-fast_amd/csrc/plan_rule.inc]
    python open-jev-fast_amd/planfit.py DATA.csv --ranges             # range rows, to go into csrc/plan_table.inc
    python open-jev-fast_amd/planfit.py DATA.csv --thin OUT.csv       # only what the fit and the picks need

The cost of a pick at one point (kind, N, K, M) is its measured time over the best measured two-launch candidate's.
The fit minimises the squared log errors of the estimate over the candidates within 30% of the best at each point.
"""
import argparse
import csv
import os
import re
import sys
from collections import defaultdict

HERE = os.path.dirname(os.path.abspath(__file__))
RULE_INC = os.path.join(HERE, "csrc", "plan_rule.inc")
CUS = 256
SPLITS = (1, 2, 3, 4, 6, 8)
CONSTANTS = {  # name in plan_rule.inc -> what it is
    "kHbmBytesPerUs": "weights from HBM",
    "kTileUs": "persistent tile: prologue and epilogue",
    "kPieceLaunchUs": "stream-K: launch of the split-tile pass",
    "kPieceBytesPerUs": "and the rate its pieces are written and read at",
    "kRoundUs": "other tiles: prologue and epilogue of a round",
    "kPlaneLaunchUs": "K splits: launch of the reduction",
    "kPlaneBytesPerUs": "and the rate its planes are written and read at",
}


def cdiv(a, b):
    return -(-a // b)


def read_rule(path=RULE_INC):
    """(stage cost by tile, constants by name) of a plan_rule.inc."""
    text = open(path).read()
    stage = {int(t): float(us) for t, us in re.findall(r"\{(\d+), ([0-9.]+)\}", text)}
    const = {n: float(re.search(rf"double {n} = ([0-9.e]+);", text).group(1)) for n in CONSTANTS}
    return stage, const


def write_rule(path, stage, const):
    head = open(RULE_INC).read().split("constexpr")[0]
    items = [f"{{{t}, {stage[t]:.3f}}}" for t in sorted(stage)]
    rows = ",\n    ".join(", ".join(items[i:i + 8]) for i in range(0, len(items), 8))
    with open(path, "w") as f:
        f.write(f"{head}constexpr StageCost kStageCost[] = {{\n    {rows}}};\n")
        for n, what in CONSTANTS.items():
            v = f"{const[n] / 1e6:.2f}e6" if n.endswith("BytesPerUs") else f"{const[n]:.2f}"
            line = f"constexpr double {n} = {v};"
            f.write(f"{line:<46}// {what}\n")


def plan_us(info, stage, const, M, N, K, residual, S):
    """The estimate of api.hip's plan_us (us)."""
    bn, bm = info["bn"], info["bm"]
    tm = cdiv(M, bm)
    tiles = cdiv(N, bn) * tm

    def rate(running):
        return max(stage, min(running, CUS) / tm * bn * 128.0 / const["kHbmBytesPerUs"])

    if info["family"] == 5:
        ipt = cdiv(K, 64)
        full, rem = divmod(tiles, CUS)
        gs = min(rem * S, rem * ipt)
        its = full * ipt + (cdiv(rem * ipt, gs) if rem else 0)
        us = its * rate(CUS if full else gs) + const["kTileUs"] * (full + (rem > 0))
        if gs > rem:
            us += 0.0 if residual else const["kPieceLaunchUs"]
            us += 2.0 * (gs + rem) * bn * bm * 4.0 / const["kPieceBytesPerUs"]
        return us
    nk, wgs = cdiv(cdiv(K, S), 64), tiles * S
    us = cdiv(wgs, CUS) * (nk * rate(wgs) + const["kRoundUs"])
    if S > 1:
        us += 0.0 if residual else const["kPlaneLaunchUs"]
        us += 2.0 * S * M * N * 4.0 / const["kPlaneBytesPerUs"]
    return us


def skinny(M, N):
    """Calls that the rule plans for weight streaming, without an estimate."""
    return M <= 32 and not (M > 16 and cdiv(N, 144) >= 200)


def rule_candidates(tiles, stage, M, N, K, residual):
    """The (tile, split) pairs that the rule estimates (packed limits and rows out of reach aside)."""
    for t in stage:
        n = cdiv(N, tiles[t]["bn"]) * cdiv(M, tiles[t]["bm"])
        rem = n % CUS
        for S in SPLITS:
            persistent = tiles[t]["family"] == 5
            if S > 1 and ((rem == 0 or rem * S > CUS) if persistent else (K // S < 512 or (residual and N > 8192))):
                break
            yield t, S


def rule_pick(tiles, rule, M, N, K, kind):
    """(tile, split) of the rule for M > 32 or a wide N, None where it does not estimate."""
    if skinny(M, N):
        return None
    stage, const = rule
    res = (kind & 3) == 2
    return min(rule_candidates(tiles, stage, M, N, K, res),
               key=lambda c: plan_us(tiles[c[0]], stage[c[0]], const, M, N, K, res, c[1]))


def read_data(paths):
    """{(kind, N, K, M): {(tile, split): us}} of the two-launch candidates."""
    pts = defaultdict(dict)
    for p in paths:
        for r in csv.DictReader(open(p)):
            if int(r["one_launch"]) == 0:
                key = tuple(int(r[c]) for c in ("kind", "N", "K", "M"))
                pts[key][int(r["tile"]), int(r["splitk"])] = float(r["us"])
    return dict(pts)


def cost_summary(pts, pick):
    """(points, mean, 90th percentile and largest cost - 1, points whose pick was not measured) of pick(point)."""
    cost, missing = [], 0
    for key, c in pts.items():
        p = pick(key)
        if p is None:
            continue
        if p not in c:
            missing += 1
            continue
        cost.append(c[p] / min(c.values()) - 1.0)
    cost.sort()
    if not cost:
        return 0, 0.0, 0.0, 0.0, missing
    return len(cost), sum(cost) / len(cost), cost[int(0.9 * len(cost))], cost[-1], missing


def fit(pts, tiles, rule):
    """Stage costs and constants fitted from the given ones (log parameters, least squares)."""
    import numpy as np
    from scipy.optimize import least_squares
    stage, const = rule
    ts, ns = sorted(stage), list(CONSTANTS)
    obs = []
    for (kind, N, K, M), c in pts.items():
        if skinny(M, N):
            continue
        res = (kind & 3) == 2
        known = set(rule_candidates(tiles, stage, M, N, K, res))
        obs += [(t, M, N, K, res, S, us) for (t, S), us in c.items() if us <= 1.3 * min(c.values()) and (t, S) in known]

    def unpack(v):
        e = np.exp(v)
        return dict(zip(ts, e)), dict(zip(ns, e[len(ts):]))

    def err(v):
        s, c = unpack(v)
        return [np.log(plan_us(tiles[t], s[t], c, M, N, K, r, S) / us) for t, M, N, K, r, S, us in obs]

    sol = least_squares(err, np.log([stage[t] for t in ts] + [const[n] for n in ns]), loss="soft_l1", f_scale=0.05)
    return unpack(sol.x), len(obs)


def ranges(pts, tiles, rule, least=0.05):
    """Range rows: per (kind, N, K), intervals of the measured row counts and one measured plan each, so that the time
    saved against the rule is largest, a row saving `least` or more of the rule's time summed over its row counts."""
    shapes = defaultdict(list)
    for (kind, N, K, M) in pts:
        shapes[kind, N, K].append(M)
    out = []
    for (kind, N, K), Ms in shapes.items():
        Ms = sorted(m for m in Ms if rule_pick(tiles, rule, m, N, K, kind) in pts[kind, N, K, m])
        at = [pts[kind, N, K, m] for m in Ms]
        base = [c[rule_pick(tiles, rule, m, N, K, kind)] for m, c in zip(Ms, at)]
        best = [(0.0, None)]  # best[j]: saving over the first j row counts, and how
        for j in range(1, len(Ms) + 1):
            b = (best[j - 1][0], None)
            for i in range(max(0, j - 8), j):
                total = sum(base[i:j])
                for cand in set.intersection(*(set(c) for c in at[i:j])):
                    us = sum(c[cand] for c in at[i:j])
                    if total - us >= least * total and best[i][0] + total - us > b[0]:
                        b = (best[i][0] + total - us, (i, cand, at[j - 1][cand]))
            best.append(b)
        j = len(Ms)
        while j > 0:
            how = best[j][1]
            if how is None:
                j -= 1
                continue
            i, (t, S), us = how
            lo = Ms[i - 1] + 1 if i > 0 else Ms[i]
            out.append((Ms[j - 1], N, K, kind, t, S, lo, us))
            j = i
    return sorted(out, key=lambda r: (-(r[3] & 4), r[1], r[2], r[3], r[0]))


def main():
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("data", nargs="+")
    ap.add_argument("--fit", action="store_true")
    ap.add_argument("--rule-out", default="")
    ap.add_argument("--ranges", action="store_true")
    ap.add_argument("--thin", default="")
    args = ap.parse_args()
    sys.path.insert(0, os.path.dirname(HERE))
    import __graft_entry__
    lib = __graft_entry__.load_package()._lib
    tiles = {t: lib.tile_info(t) for t in range(lib.lib().ojx_num_tiles())}
    pts, rule = read_data(args.data), read_rule()

    def table(key):
        kind, N, K, M = key
        c = lib.plan(M, N, K, kind)
        return (c.tile, c.splitk) if c.tail_rows == 0 and c.one_launch == 0 else None

    def show(what, pick):
        n, mean, p90, worst, missing = cost_summary(pts, pick)
        print(f"{what}: {n} points, mean cost {100 * mean:.1f}%, 90th percentile {100 * p90:.1f}%, largest "
              f"{100 * worst:.1f}% ({missing} picks not measured)", flush=True)

    print(f"{sum(map(len, pts.values()))} candidates at {len(pts)} points")
    show("rule", lambda k: rule_pick(tiles, rule, k[3], k[1], k[2], k[0]))
    show("table and rule, two-launch plans", table)
    if args.fit:
        rule, n = fit(pts, tiles, rule)
        print(f"fitted to {n} candidates: {({k: round(float(v), 3) for k, v in {**rule[0], **rule[1]}.items()})}")
        show("fitted rule", lambda k: rule_pick(tiles, rule, k[3], k[1], k[2], k[0]))
        if args.rule_out:
            write_rule(args.rule_out, *rule)
    if args.thin:  # the candidates within 30% of the best at their point, and the picks
        with open(args.thin, "w") as f:
            f.write("kind,N,K,M,tile,splitk,one_launch,us\n")
            for key, c in sorted(pts.items()):
                kind, N, K, M = key
                picks = (rule_pick(tiles, rule, M, N, K, kind), table(key))
                for (t, S), us in sorted(c.items()):
                    if us <= 1.3 * min(c.values()) or (t, S) in picks:
                        f.write(f"{kind},{N},{K},{M},{t},{S},0,{us:.2f}\n")
    if args.ranges:
        for M, N, K, kind, t, S, lo, us in ranges(pts, tiles, rule):
            print(f"{{{M}, {N}, {K}, {kind}, {t}, {S}, 0, 1, 0, 0, {lo}}},  // {us:.1f} us")


if __name__ == "__main__":
    main()
