"""C-ABI checks that need no GPU: the library loads, exports every function include/ojx.h declares, and its host
logic (plan table, candidate list, workspace sizes, argument validation and error messages) behaves."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def header_functions():
    text = open(os.path.join(ROOT, "include", "ojx.h")).read()
    return sorted(set(re.findall(r"^\s*(?:const\s+)?\w+\*?\s+\**(ojx_\w+)\s*\(", text, re.M)))


def test_header_symbols_exported(pkg):
    names = header_functions()
    assert len(names) >= 19
    L = ctypes.CDLL(pkg._lib.LIB_PATH)
    for n in names:
        assert hasattr(L, n), n
    assert set(names) == set(pkg._lib.EXPORTS), "ctypes table out of sync with include/ojx.h"


def test_version_and_tiles(pkg):
    L = pkg._lib.lib()
    assert b"gfx950" in L.ojx_version()
    from importlib import import_module
    build = import_module("open_jev_fast_amd.build")
    # the loaded binary was compiled from this tree's sources (digest of csrc/ and include/ojx.h)
    assert L.ojx_version().decode().endswith("src:" + build.source_digest())
    n = L.ojx_num_tiles()
    assert n >= 8
    live = 0
    for t in range(n):
        info = pkg._lib.tile_info(t)
        if info["family"] < 0:  # a retired id: never planned, fitted or launched
            assert all(c.tile != t for c in pkg._lib.candidates(288, 1024, 2048, 0))
            continue
        live += 1
        assert info["bn"] % 16 == 0 and info["bm"] % 16 == 0 and info["bk"] % 32 == 0
        assert info["threads"] == 64 * info["wn"] * info["wm"]
    assert live >= 8 and pkg._lib.tile_info(52)["family"] == -1
    with pytest.raises(RuntimeError, match="out of range"):
        pkg._lib.tile_info(n)


SHAPES = [(M, N, K) for M in (1, 7, 16, 64, 128, 288, 539, 1024, 2048)
          for N, K in ((14336, 5120), (34816, 5120), (5120, 17408), (5120, 6144), (16384, 5120), (16480, 5120))]


def test_plan_table_names_live_tiles(pkg):
    """Every tile id stored in the plan table (main and tail) is a live tile: a retired id reports family -1."""
    import os
    import re
    src = os.path.join(os.path.dirname(pkg.__file__), "csrc", "plan_table.inc")
    rows = [list(map(int, m.group(1).split(","))) for m in re.finditer(r"^\{([^}]*)\}", open(src).read(), re.M)]
    assert len(rows) > 100
    for r in rows:
        for t in (r[4], r[6]):
            assert pkg._lib.tile_info(t)["family"] >= 0, f"plan row {r} names tile {t}"


def _plan_kinds(N, K):
    return [k | p for k in (0, 1, 2) for p in (0, 4) if not p or (N % 16 == 0 and K % 64 == 0)]


def test_plan_rule_off_the_table(pkg):
    """Calls that no row covers: over sizes from one row and eight columns up, every plan is a configuration that the
    library itself accepts (ojx_workspace_bytes checks it), names a live tile, has no tail and no one-launch
    reduction, and leaves a residual projection wider than 8192 columns without planes (its row pass cannot read
    them back without an RMSNorm output)."""
    import random
    rng = random.Random(3)
    sizes = [(1, 8, 8), (17, 8, 8), (33, 16, 64), (2049, 5120, 5120), (65536, 256, 64), (300, 65536, 128)]
    for _ in range(400):
        M = int(2 ** rng.uniform(0, 13))
        N = 16 * int(2 ** rng.uniform(0, 11)) if rng.random() < 0.5 else 8 * rng.randint(1, 4000)
        K = 64 * rng.randint(1, 300) if rng.random() < 0.5 else 8 * rng.randint(1, 2500)
        sizes.append((M, N, K))
    for M, N, K in sizes:
        for kind in _plan_kinds(N, K):
            if kind & 4 and N * K * 2 >= 2 ** 31:
                continue
            c = pkg._lib.plan(M, N, K, kind)
            what = (M, N, K, kind, c)
            assert pkg._lib.tile_info(c.tile)["family"] in (0, 5, 6), what
            assert pkg._lib.lib().ojx_workspace_bytes(M, N, K, kind, ctypes.byref(c)) >= 0, what
            assert c.tail_rows == 0 and c.one_launch == 0 and 1 <= c.splitk <= 8, what
            if kind & 3 == 2 and N > 8192 and pkg._lib.tile_info(c.tile)["family"] != 5:
                assert c.splitk == 1, what


# 64-row tiles reach to K = 2^24, 32-row tiles to 2^25
@pytest.mark.parametrize("M,N,K", [(300, 64, 1 << 22), (33, 128, 1 << 23), (2048, 1024, 3_500_032), (24, 65536, 1 << 22),
                                   (24, 64, 20_000_000), (300, 64, (1 << 25) - 64), (16, 8, 1 << 25)])
@pytest.mark.parametrize("kind", [0, 2])
def test_plan_rule_keeps_rows_in_reach(pkg, M, N, K, kind):
    """Tiles address their rows with 32-bit offsets through descriptors of less than 2^31 bytes: a plan's tile rows
    that exist span no more than that, however long a row is."""
    t = pkg._lib.tile_info(pkg._lib.plan(M, N, K, kind).tile)
    assert max(min(t["bm"], M), min(t["bn"], N)) * K * 2 < 2 ** 31, t


@pytest.mark.parametrize("kind", [0, 1, 2, 4, 5, 6])
def test_plan_refuses_empty_and_negative_sizes(pkg, kind):
    """An empty or negative dimension ends in the shape error before any plan arithmetic (which divides by tile
    counts and K stages), from ojx_plan, ojx_workspace_bytes and the Python entry points' workspace and tuning calls;
    M = 0 is a plan as before (the launch is then a no-op)."""
    import torch
    from importlib import import_module
    ext = import_module("open_jev_fast_amd.ext")
    L, c = pkg._lib.lib(), pkg._lib.OjxCfg()
    given = pkg._lib.cfg(0, 1)
    bad = [(M, *nk) for M in (0, 7, 24, 64, 300) for b in (0, -8, -64, 1 << 31)
           for nk in ((b, 5120), (5120, b), (b, b), (b, 64))] + [(-1, 5120, 5120), (-64, 64, 64), (1 << 31, 64, 64)]
    for M, N, K in bad:
        assert L.ojx_plan(M, N, K, kind, ctypes.byref(c)) == 2, (M, N, K)
        assert b"shape" in L.ojx_last_error()
        for cfg in (None, ctypes.byref(given)):
            assert L.ojx_workspace_bytes(M, N, K, kind, cfg) == -1, (M, N, K)
        with pytest.raises(RuntimeError, match="shape"):
            ext._workspace(M, N, K, kind, None, torch.device("cpu"))
    assert L.ojx_plan(0, 5120, 5120, kind, ctypes.byref(c)) == 0
    proj = import_module("open_jev_fast_amd.fastproj").FastProjections()
    e = lambda *s: torch.empty(*s, dtype=torch.bfloat16)  # noqa: E731
    for x, w in ((e(64, 0), e(5120, 0)), (e(7, 5120), e(0, 5120))):
        with pytest.raises(RuntimeError, match="bad shape"):
            proj._tune(x, w)
        with pytest.raises(RuntimeError, match="bad shape"):
            proj._tune_sk(x, w, 2)


def test_rows_out_of_reach_are_refused_before_a_launch(pkg):
    """Where no tile reaches the rows of the call (or the given one does not), every entry point returns the shape
    error instead of multiplying zeros: planned and explicit configurations, splits, strides, one-launch, planes, the
    fused prep. The sizes below the limits pass the same check and end at the launch, so this needs a machine without
    a GPU (the buffers are host memory)."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("hands host buffers to launches that must fail for want of a GPU")
    L = pkg._lib.lib()
    buf = ctypes.create_string_buffer(1 << 12)
    p = ctypes.cast(ctypes.addressof(buf) + (-ctypes.addressof(buf)) % 16, ctypes.c_void_p)
    f = ctypes.cast(p, ctypes.POINTER(ctypes.c_float))
    ws = 1 << 62
    cfgp = lambda c: None if c is None else ctypes.byref(pkg._lib.cfg(*c))  # noqa: E731

    def refused(rc):
        assert rc == 2 and b"2 GiB" in L.ojx_last_error(), (rc, L.ojx_last_error())

    def in_reach(rc):  # passes the check: what fails is the launch, for want of a GPU
        assert rc == 5 and b"2 GiB" not in L.ojx_last_error(), (rc, L.ojx_last_error())

    for M, N, K in ((24, 128, 1 << 25), (300, 64, 1 << 25), (16, 1024, 1 << 25), (1, 64, 1 << 26), (1, 8, 1 << 30)):
        for c in (None, (0, 1), (90, 2), (73, 4), (80, 3), (0, 2, 0, 1, 0, 1)):
            refused(L.ojx_gemm_bf16(p, p, p, M, N, K, K, K, N, p, ws, cfgp(c), None))
            refused(L.ojx_gemm_silu_mul(p, p, p, M, N // 2, K, p, ws, cfgp(c), None))
            refused(L.ojx_gemm_residual_rmsnorm(p, p, p, p, None, 1e-6, p, p, M, N, K, p, ws, cfgp(c), None))
        for tile in (-1, 0, 80):
            refused(L.ojx_gemm_splitk_f32(p, p, p, M, N, K, K, K, 2, tile, None))
    refused(L.ojx_gemm_qkv_fullattn_prep(p, p, 0, f, f, p, p, p, p, p, p, 4, 1 << 24, 2, 1, 256, 64, 1e-6, None))
    for ld in ((1 << 30) + 8, 1 << 40, 1 << 62):  # row strides: two rows or more
        refused(L.ojx_gemm_bf16(p, p, p, 2, 64, 64, ld, 64, 64, p, ws, None, None))
        refused(L.ojx_gemm_bf16(p, p, p, 1, 64, 64, 64, ld, 64, p, ws, None, None))
        refused(L.ojx_gemm_splitk_f32(p, p, p, 2, 64, 64, ld, 64, 1, -1, None))
        refused(L.ojx_gemm_bf16_pk(p, p, p, 2, 64, 64, ld, 64, p, ws, None, None))
    in_reach(L.ojx_gemm_bf16(p, p, p, 1, 64, 64, 1 << 40, 64, 64, p, ws, None, None))  # one row: its stride is not used
    in_reach(L.ojx_gemm_bf16(p, p, p, 2, 64, 64, (1 << 30) - 64 - 8, 64, 64, p, ws, None, None))
    in_reach(L.ojx_gemm_bf16(p, p, p, 24, 64, 20_000_000, 20_000_000, 20_000_000, 64, p, ws, None, None))


def test_ragged_cases_reach_every_family(pkg):
    """The GPU cases with a partial last K stage are planned on the families and splits that they name: split and
    unsplit tiles of families 0 and 6, persistent tiles with a spread, all three kinds."""
    from tests.test_gpu_random_shapes import RAGGED_PLANS
    for kind, M, N, K, family, split in RAGGED_PLANS:
        c = pkg._lib.plan(M, N, K, ("plain", "silu", "residual").index(kind))
        got = (pkg._lib.tile_info(c.tile)["family"], c.splitk > 1)
        assert K % 64 and got == (family, split), (kind, M, N, K, c)


def test_plan_rule_is_a_function_of_its_arguments(pkg):
    """The rule's plans come through a small table per thread: the same sizes in another order, with others in
    between and from another thread, give the same plans."""
    import threading
    args = [(M, N, K, k) for M in (33, 100, 515, 3000) for N in (512, 4096, 5120) for K in (1024, 4160)
            for k in _plan_kinds(N, K)]
    ask = lambda a: (lambda c: (c.tile, c.splitk, c.one_launch, c.tail_rows))(pkg._lib.plan(*a))  # noqa: E731
    first = {a: ask(a) for a in args}
    got = {}
    t = threading.Thread(target=lambda: got.update({a: ask(a) for a in args[::-1]}))
    t.start()
    t.join()
    assert got == first and all(ask(a) == first[a] for a in args[::3] + args[::2])


def test_planfit_restates_the_rule(pkg, tmp_path):
    """The Python restatement that judges and fits the rule picks what the library's rule picks, over random calls that
    no table row covers; its constants file reads back as written."""
    import random
    from importlib import import_module
    fit = import_module("open_jev_fast_amd.planfit")
    tiles = {t: pkg._lib.tile_info(t) for t in range(pkg._lib.lib().ojx_num_tiles())}
    rule = fit.read_rule()
    fit.write_rule(tmp_path / "rule.inc", *rule)
    assert (tmp_path / "rule.inc").read_text() == open(fit.RULE_INC).read()
    rng = random.Random(4)
    for _ in range(600):
        M, N, K = int(2 ** rng.uniform(4.2, 12)), 8 * rng.randint(4, 5000), 8 * rng.randint(8, 2500)
        kind = rng.choice([0, 1, 2])
        c = pkg._lib.plan(M, N, K, kind)
        pick = fit.rule_pick(tiles, rule, M, N, K, kind)
        assert pick is None or pick == (c.tile, c.splitk), (M, N, K, kind, c)


def test_planfit_costs_and_ranges(pkg):
    """Costs and range rows from a made-up measured set: the rule's pick is 10% behind one plan at M = 96 and 112 and the
    best one elsewhere, so that one range row covers 65 (after the measured 64) to 112."""
    from importlib import import_module
    fit = import_module("open_jev_fast_amd.planfit")
    tiles = {t: pkg._lib.tile_info(t) for t in range(pkg._lib.lib().ojx_num_tiles())}
    rule, N, K = fit.read_rule(), 7168, 4096
    pts = {}
    for M in (48, 64, 96, 112, 160):
        p = fit.rule_pick(tiles, rule, M, N, K, 0)
        pts[0, N, K, M] = {p: 110.0, (6, 1): 100.0 if M in (96, 112) else 200.0}
    n, mean, p90, worst, missing = fit.cost_summary(pts, lambda k: fit.rule_pick(tiles, rule, k[3], k[1], k[2], k[0]))
    assert (n, missing) == (5, 0) and abs(mean - 0.04) < 1e-9 and abs(worst - 0.1) < 1e-9
    assert fit.ranges(pts, tiles, rule) == [(112, N, K, 0, 6, 1, 65, 100.0)]


def test_tuner_keeps_the_rows_it_did_not_measure(pkg):
    """tune.py --out changes the measured single rows only: ranges, comments and the other rows stay, new calls go to
    their shape's rows."""
    from importlib import import_module
    tune = import_module("open_jev_fast_amd.tune")
    text = open(os.path.join(os.path.dirname(pkg.__file__), "csrc", "plan_table.inc")).read()
    assert tune.merge_table(text, []) == text
    new = tune.merge_table(text, [(288, 34816, 5120, 1, (73, 2, 0, 1, 0, 0), 1e-4), (300, 34816, 5120, 1, (80, 1, 0, 1, 0, 0), 2e-4),
                                  (5, 512, 512, 0, (0, 1, 0, 1, 0, 0), 3e-6)])
    old, got = text.splitlines(), new.splitlines()
    assert len(got) == len(old) + 2
    assert set(got) - set(old) == {"{288, 34816, 5120, 1, 73, 2, 0, 1, 0, 0, 0},  // 100.0 us",
                                   "{300, 34816, 5120, 1, 80, 1, 0, 1, 0, 0, 0},  // 200.0 us",
                                   "{5, 512, 512, 0, 0, 1, 0, 1, 0, 0, 0},  // 3.0 us"}
    assert [l for l in old if l not in got] == [l for l in old if l.startswith("{288, 34816, 5120, 1,")]
    assert [l for l in got if l in set(old)] == [l for l in old if l in set(got)]
    assert got.index("{300, 34816, 5120, 1, 80, 1, 0, 1, 0, 0, 0},  // 200.0 us") < next(
        i for i, l in enumerate(got) if l.startswith("// ---- ranges"))


def test_plan_table_ranges(pkg):
    """Range rows (m_lo > 0): ordered, disjoint per shape and kind, two-launch, and the plan of every row count in
    them; a row for a single count inside a range goes first."""
    src = os.path.join(os.path.dirname(pkg.__file__), "csrc", "plan_table.inc")
    rows = [list(map(int, m.group(1).split(","))) for m in re.finditer(r"^\{([^}]*)\}", open(src).read(), re.M)]
    single = {tuple(r[:4]): (r[4], r[5], r[9]) for r in rows if len(r) < 11 or r[10] == 0}
    last = {}
    for r in rows:
        if len(r) < 11 or r[10] == 0:
            continue
        hi, N, K, kind, lo = r[0], r[1], r[2], r[3], r[10]
        assert 1 < lo <= hi and lo > last.get((N, K, kind), 0) and r[8] == 0 and r[9] == 0
        last[(N, K, kind)] = hi
        for M in (lo, (lo + hi) // 2, hi):
            c = pkg._lib.plan(M, N, K, kind)
            assert (c.tile, c.splitk, c.one_launch) == single.get((M, N, K, kind), (r[4], r[5], 0))


@pytest.mark.parametrize("kind", [0, 1, 2, 4, 5, 6])
def test_plan_valid_for_every_contract_shape(pkg, kind):
    L = pkg._lib.lib()
    for M, N, K in SHAPES:
        c = pkg._lib.plan(M, N, K, kind)
        assert 0 <= c.tile < L.ojx_num_tiles() and 1 <= c.splitk <= 16
        live = lambda t: pkg._lib.tile_info(t)["family"] >= 0  # noqa: E731
        assert live(c.tile) and (c.tail_rows == 0 or live(c.tail_tile))
        ws = pkg._lib.workspace_bytes(M, N, K, kind)
        # each launch's data one after the other: split-K planes (rounded up to 256 bytes) or, for the persistent
        # family, partial-tile slots (or nothing)
        parts = [(c.tile, c.splitk, N - c.tail_rows)] + ([(c.tail_tile, c.tail_splitk, c.tail_rows)] if c.tail_rows else [])
        data, sk = 0, False
        for tile, S, n in parts:
            if pkg._lib.tile_info(tile)["family"] == 5:
                sk = True
            elif S > 1:
                data += -(-S * M * n * 4 // 256) * 256
                if c.one_launch:  # the per-tile row sums of squares follow the planes
                    data += -(-(-(-n // pkg._lib.tile_info(tile)["bn"])) * M * 4 // 256) * 256
        if sk:
            assert ws >= data
        else:
            assert ws == data


def test_candidates(pkg):
    cands = pkg._lib.candidates(288, 5120, 5120)
    assert len(cands) > 10
    assert len({(c.tile, c.splitk, c.one_launch) for c in cands}) == len(cands)
    ol = [c for c in cands if c.one_launch]
    assert ol and all(pkg._lib.tile_info(c.tile)["family"] in (0, 6) and c.splitk >= 2 for c in ol)
    assert all(c.one_launch == 1 for c in ol)  # the RMSNorm fold (2) is a residual candidate only
    fold = [c for c in pkg._lib.candidates(7, 5120, 6144, 2) if c.one_launch == 2]
    assert fold and all(pkg._lib.tile_info(c.tile)["family"] == 0 for c in fold)
    # no tile whose x rows are mostly padding at M = 7
    for c in pkg._lib.candidates(7, 5120, 5120):
        assert pkg._lib.tile_info(c.tile)["bm"] == 16
    L = pkg._lib.lib()
    c = pkg._lib.OjxCfg()
    assert L.ojx_candidate(7, 5120, 5120, 0, 10 ** 6, ctypes.byref(c)) == 4
    assert b"out of range" in L.ojx_last_error()


def test_argument_validation_without_gpu(pkg):
    """These return before any HIP call, so they run on a machine without a GPU."""
    L = pkg._lib.lib()
    buf = ctypes.create_string_buffer(1 << 12)
    p = ctypes.cast(ctypes.addressof(buf) + (-ctypes.addressof(buf)) % 16, ctypes.c_void_p)
    # N not a multiple of 8
    assert L.ojx_gemm_bf16(p, p, p, 4, 60, 64, 64, 64, 60, None, 0, None, None) == 2
    assert b"multiples of 8" in L.ojx_last_error()
    # null operand
    assert L.ojx_gemm_bf16(None, p, p, 4, 64, 64, 64, 64, 64, None, 0, None, None) == 1
    # misaligned
    mis = ctypes.c_void_p(p.value + 2)
    assert L.ojx_gemm_bf16(mis, p, p, 4, 64, 64, 64, 64, 64, None, 0, None, None) == 1
    # stride smaller than K
    assert L.ojx_gemm_bf16(p, p, p, 4, 64, 64, 32, 64, 64, None, 0, None, None) == 1
    # bad config
    bad = pkg._lib.OjxCfg(999, 1)
    assert L.ojx_gemm_bf16(p, p, p, 4, 64, 64, 64, 64, 64, None, 0, ctypes.byref(bad), None) == 4
    bad = pkg._lib.OjxCfg(0, 17)
    assert L.ojx_gemm_bf16(p, p, p, 4, 64, 64, 64, 64, 64, None, 0, ctypes.byref(bad), None) == 4
    # split-K without workspace
    sk = pkg._lib.OjxCfg(0, 2)
    assert L.ojx_gemm_bf16(p, p, p, 4, 64, 64, 64, 64, 64, None, 0, ctypes.byref(sk), None) == 3
    assert b"workspace" in L.ojx_last_error()
    # RMSNorm row limit (H/8 <= 1024), as the reference's TORCH_CHECK (src/kernels.cu:757)
    assert L.ojx_add_rmsnorm(p, None, p, None, 1e-6, None, p, 4, 8200, None) == 2
    assert L.ojx_add_rmsnorm_sk(p, p, 17, p, None, 1e-6, p, p, 4, 64, None) == 4
    # silu_mul needs I % 8 == 0
    assert L.ojx_silu_mul(p, p, 4, 12, None) == 2
    assert L.ojx_gemm_silu_mul(p, p, p, 4, 6, 64, None, 0, None, None) == 2
    assert L.ojx_pack_gate_up(p, p, p, 6, 64, None) == 2
    # M == 0 is a no-op
    assert L.ojx_gemm_bf16(p, p, p, 0, 64, 64, 64, 64, 64, None, 0, None, None) == 0
    # scoring head: H % 8, null operands, misalignment; R == 0 is a no-op
    assert L.ojx_head_scores(p, 4, 60, p, 3, p, None, p, None) == 2
    assert L.ojx_head_scores(None, 4, 64, p, 3, p, None, p, None) == 1
    assert L.ojx_head_scores(mis, 4, 64, p, 3, p, None, p, None) == 1
    assert L.ojx_head_scores(p, 4, 64, p, 0, p, None, p, None) == 0


def test_prep_argument_validation_without_gpu(pkg):
    """The prep entry points reject what their kernels do not handle before any HIP call (head dims, rotary dims,
    head-count ratios, sizes, alignment); empty inputs are no-ops."""
    L = pkg._lib.lib()
    buf = ctypes.create_string_buffer(1 << 12)
    p = ctypes.cast(ctypes.addressof(buf) + (-ctypes.addressof(buf)) % 16, ctypes.c_void_p)
    mis = ctypes.c_void_p(p.value + 2)
    f = ctypes.cast(p, ctypes.POINTER(ctypes.c_float))
    fa = lambda N, HQ, HKV, D, RD, proj=p: L.ojx_fullattn_prep(proj, N, HQ, HKV, D, RD, 1e-6, f, f, p, p, p, p, p,  # noqa: E731
                                                                p, None)
    assert fa(3, 2, 1, 128, 64) == 2 and b"head_dim 256" in L.ojx_last_error()
    assert fa(3, 2, 1, 256, 48) == 2 and b"rotary" in L.ojx_last_error()   # 48 / 16 = 3, not a power of two
    assert fa(3, 2, 1, 256, 8) == 2                                          # below 16
    assert fa(3, 2, 1, 256, 512) == 2                                        # above D
    assert fa(3, 0, 1, 256, 64) == 2
    assert fa(3, 2, 1, 256, 64, proj=mis) == 1
    assert fa(0, 2, 1, 256, 64, proj=None) == 0                              # no tokens: nothing to do
    q = lambda M, K, RD, w=p: L.ojx_gemm_qkv_fullattn_prep(p, w, 0, f, f, p, p, p, p, p, p, M, K, 2, 1, 256, RD,  # noqa: E731
                                                           1e-6, None)
    assert q(4, 256, 32) == 2 and b"RD = 64" in L.ojx_last_error()
    assert q(4, 260, 64) == 2                                                # K not a multiple of 8
    assert q(4, 256, 64, w=None) == 1
    la = lambda N, R, L2, KD, VD, HV, HK, HD, rq, proj=p: L.ojx_linattn_prep(  # noqa: E731
        proj, p, p, p, N, R, L2, p, p, p, KD, VD, HV, HK, HD, rq, p, p, p, f, p, None)
    assert la(5, 32, 16, 256, 768, 6, 2, 64, 0) == 2 and b"head_dim 128" in L.ojx_last_error()
    assert la(5, 32, 16, 384, 768, 6, 2, 128, 0) == 2                       # KD != HK HD
    assert la(5, 30, 16, 256, 768, 6, 2, 128, 0) == 2                       # R not a multiple of L2
    assert la(5, 32, 16, 256, 768, 8, 2, 128, 1) == 2 and b"HV / HK = 3" in L.ojx_last_error()
    assert la(5, 32, 16, 256, 768, 300, 2, 128, 0) == 2                     # HV > 256
    assert la(5, 32, 16, 256, 768, 6, 2, 128, 0, proj=mis) == 1
    assert la(5, 0, 16, 256, 768, 6, 2, 128, 0, proj=None) == 0             # no slots: nothing to do


def test_linattn_prep_channel_limits(pkg):
    """Channel counts past the 28672 that an earlier kernel held in LDS pass the checks (and end at the launch, for
    want of a GPU); sizes whose products leave 32 bits are refused."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("hands host buffers to launches that must fail for want of a GPU")
    L = pkg._lib.lib()
    buf = ctypes.create_string_buffer(1 << 12)
    p = ctypes.cast(ctypes.addressof(buf) + (-ctypes.addressof(buf)) % 16, ctypes.c_void_p)
    f = ctypes.cast(p, ctypes.POINTER(ctypes.c_float))
    la = lambda KD, VD, HK, N=5: L.ojx_linattn_prep(p, p, p, p, N, 32, 16, p, p, p, KD, VD, 6, HK, 128, 0, p, p,  # noqa: E731
                                                    p, f, p, None)
    assert la(256, 28160, 2) == 5 and la(256, 28168, 2) == 5 and la(16384, 32768, 128) == 5
    assert la(256, 768, 2, N=1 << 24) == 5
    assert la(0, 768, 1 << 25) == 2 and la(128, 768, (1 << 25) + 1) == 2   # HK HD wraps to KD in 32 bits
    assert la(1 << 30, 768, 1 << 23) == 2 and la(256, (1 << 31) - 8, 2) == 2


def test_python_mirror_errors_without_gpu(pkg):
    import torch
    from importlib import import_module
    ext = import_module("open_jev_fast_amd.ext")
    x = torch.zeros(4, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="contiguous CUDA"):
        ext.mm(x, x)
    with pytest.raises(RuntimeError, match="S must be 2..4"):
        ext.add_rmsnorm_sk2(x, torch.zeros(5, 4, 64), torch.ones(64), None, 1e-6)
    lt = import_module("open_jev_fast_amd.lt_ext").load()
    assert lt.lt_setup(288, 5120, 5120, 8) == 8
    with pytest.raises(RuntimeError, match="lt_setup not called"):
        lt.lt_matmul(torch.zeros(3, 64, dtype=torch.bfloat16), torch.zeros(64, 64, dtype=torch.bfloat16), 0)
    with pytest.raises(RuntimeError, match="fp32"):
        lt.lt2_plan(288, 5120, 6144, 2, 0, 1)
    h = lt.lt2_plan(288, 5120, 6144, 2, 1, 1)
    n = lt.lt2_search(h, 400, 3)
    assert n >= 1 and lt.lt2_info(h, 0)[1] == 2
    raw = lt.lt2_raw(h, 0)
    assert lt.lt2_add_raw(h, raw) == n


def test_unsplit_weight_argument_validation(pkg):
    L = pkg._lib.lib()
    buf = ctypes.create_string_buffer(1 << 12)
    p = ctypes.cast(ctypes.addressof(buf) + (-ctypes.addressof(buf)) % 16, ctypes.c_void_p)
    assert L.ojx_unsplit_weight(p, p, 64, 96, 5, None) == 2  # K % S != 0
    assert b"multiple of S" in L.ojx_last_error()
    assert L.ojx_unsplit_weight(p, p, 60, 96, 2, None) == 2  # N not a multiple of 8
    assert L.ojx_unsplit_weight(None, p, 64, 96, 2, None) == 1
    assert L.ojx_unsplit_weight(p, ctypes.c_void_p(p.value + 2), 64, 96, 2, None) == 1


C_HOST = r"""
#include <stdio.h>
#include "ojx.h"
int main(void) {
  ojx_cfg c;
  if (ojx_plan(288, 34816, 5120, OJX_KIND_SILU_MUL | OJX_KIND_PACKED, &c) != OJX_OK) return 1;
  long long ws = (long long)ojx_workspace_bytes(288, 34816, 5120, OJX_KIND_SILU_MUL | OJX_KIND_PACKED, &c);
  printf("%s|%d|%d|%d|%lld\n", ojx_version(), ojx_num_tiles(), c.tile, c.splitk, ws);
  return ws < 0;
}
"""


def test_c_host_compiles_links_and_plans(pkg, tmp_path):
    """include/ojx.h is plain C (C99) and C++; a C host links libojx.so and uses its host-side calls (the plan
    lookup and workspace size need no GPU), as the C / C++ integration path does."""
    import shutil
    import subprocess
    inc = os.path.join(ROOT, "include")
    for comp, std, lang in (("gcc", "-std=c99", "c"), ("g++", "-std=c++17", "c++")):
        if shutil.which(comp) is None:
            pytest.skip(f"{comp} not installed")
        r = subprocess.run([comp, std, "-Wall", "-Werror", "-fsyntax-only", "-x", lang, os.path.join(inc, "ojx.h")],
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
    src = tmp_path / "host.c"
    src.write_text(C_HOST)
    exe = tmp_path / "host"
    libdir = os.path.dirname(pkg._lib.LIB_PATH)
    r = subprocess.run(["gcc", "-std=c99", "-Wall", "-Werror", "-I", inc, str(src), "-o", str(exe), pkg._lib.LIB_PATH,
                        "-Wl,-rpath," + libdir, "-Wl,--allow-shlib-undefined"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    version, ntiles, tile, splitk, ws = r.stdout.strip().split("|")
    c = pkg._lib.plan(288, 34816, 5120, 1 | 4)
    assert version == pkg._lib.lib().ojx_version().decode()
    assert int(ntiles) == pkg._lib.lib().ojx_num_tiles()
    assert (int(tile), int(splitk)) == (c.tile, c.splitk)
    assert int(ws) == pkg._lib.workspace_bytes(288, 34816, 5120, 1 | 4)
