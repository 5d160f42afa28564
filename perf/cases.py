"""Performance cases of the projection path: what a server of the 27B hybrid model has this package do.

A request's prompt and candidate texts are packed into M rows (a multiple of 32 in the server, any number through the
API; 1 to 2048 here). Every layer then runs its in-projection, the attention prep on its output, the out-projection
with residual + RMSNorm, the gate-up projection with SiLU.mul and the down-projection with residual + RMSNorm; the
scoring head ends the forward. The sizes are the model's: hidden 5120, MLP 17408, linear-attention in-projection 16480
(16 q/k heads, 48 value heads of 128), full-attention QKV 14336 (24 + 4 heads of 256), out-projections 5120 x 6144.
Inputs follow the parity tests: activations ~ N(0, 1), weights ~ N(0, 0.02^2), bf16.

A case's "op" says what runs:
  head     ext.head_scores: R gathered rows of the last hidden state
  mm       ext.mm: a plain projection
  res      ext.mm_residual_rmsnorm: out / down projection, residual, RMSNorm
  silu     ext.mm_silu_mul: the fused gate-up
  mlp2     FastProjections._silu_mul(_mm(hn, w_gu)): the gate-up as two calls, the reference's own call site
  qkvprep  ext.mm_fullattn_prep: QKV in-projection and the full-attention prep
  linprep  ext.linattn_prep_dedup2: the linear-attention prep on a packed tree of candidate paths
  layer    a linear-attention layer's projections and prep, recorded once in a HIP graph and replayed, as the server
           replays one graph per request shape
"packed" says whether the weights are in the load-time packed layout (what FastProjections loads) or row-major.
"""
import math

import numpy as np
import torch

from __graft_entry__ import load_package

load_package()
from open_jev_fast_amd import ext, fastproj  # noqa: E402

H, I, KD, VD, HV, HK, HD = 5120, 17408, 2048, 6144, 48, 16, 128   # model sizes (linear attention: HK, HV heads of HD)
HQ, HKV, D, RD = 24, 4, 256, 64                                   # full attention: heads, head size, rotary dims
CONV = 2 * KD + VD
LIN_N, QKV_N, OUT_K = CONV + VD + 2 * HV, (2 * HQ + 2 * HKV) * D, VD
MM_N = (QKV_N, LIN_N, 16384, H)       # in-projections; the square 5120 layer is the generic single linear
RES_K = (OUT_K, I)                    # out-projection, down-projection
EPS = 1e-6


def listed():
    return [
        # the end of a forward: 8 candidates scored out of a 288-row request; the smallest call, launch latency
        {"name": "head_r8", "op": "head", "rows": 288, "R": 8},
        # one short text alone: weight streaming, latency counts
        {"name": "qkv_m7", "op": "mm", "M": 7, "N": QKV_N, "K": H, "packed": True},
        # a request of two row buckets: out-projection, split K, the smallest weight of the layer
        {"name": "oproj_m64", "op": "res", "M": 64, "N": H, "K": OUT_K, "packed": True},
        # the example request's row count, the model's largest projection
        {"name": "gateup_m288", "op": "silu", "M": 288, "K": H, "packed": True},
        # the gate-up as the reference's forward calls it: two calls, weights as loaded (row-major), six buckets
        {"name": "mlp2_m192_rowmajor", "op": "mlp2", "M": 192, "K": H, "packed": False},
        # the linear-attention in-projection at its real width (no multiple of 128), row-major weights
        {"name": "linin_m384_rowmajor", "op": "mm", "M": 384, "N": LIN_N, "K": H, "packed": False},
        # a longer request, not a multiple of any tile: the longest K
        {"name": "down_m539", "op": "res", "M": 539, "N": H, "K": I, "packed": True},
        # full-attention layer entry of a long request: projection and prep
        {"name": "qkvprep_m1024", "op": "qkvprep", "M": 1024, "packed": True},
        # the largest: long context, compute-bound
        {"name": "gateup_m2048", "op": "silu", "M": 2048, "K": H, "packed": True},
        # the tree prep of the example request: 200 shared rows, 8 candidates
        {"name": "linprep_200x8", "op": "linprep", "shared": 200, "paths": 8, "leaf": 11},
        # a layer of a small request and of a middling one, replayed from a graph
        {"name": "layer_m96", "op": "layer", "shared": 60, "paths": 4, "leaf": 8, "packed": True},
        {"name": "layer_m640", "op": "layer", "shared": 560, "paths": 8, "leaf": 9, "packed": True},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _rows(rng):
    m = _log_int(rng, 1, 2048)
    return m if rng.random() < 0.5 else min(2048, -(-m // 32) * 32)  # half the time a server's row bucket


def draw(rng):
    op = rng.choices(("head", "mm", "res", "silu", "mlp2", "qkvprep", "linprep", "layer"),
                     (1, 6, 5, 3, 1, 2, 2, 3))[0]
    packed = rng.random() < 0.75
    if op == "head":
        rows = _log_int(rng, 32, 2048)
        return {"op": op, "rows": rows, "R": _log_int(rng, 1, min(rows, 256))}
    if op == "mm":
        return {"op": op, "M": _rows(rng), "N": rng.choice(MM_N), "K": H, "packed": packed}
    if op == "res":
        return {"op": op, "M": _rows(rng), "N": H, "K": rng.choice(RES_K), "packed": packed}
    if op == "silu":
        return {"op": op, "M": _rows(rng), "K": H, "packed": packed}
    if op == "mlp2":  # one projection and a pass over its output; stays below the largest listed case
        return {"op": op, "M": min(_rows(rng), 1400), "K": H, "packed": False}
    if op == "qkvprep":
        return {"op": op, "M": _rows(rng), "packed": packed}
    paths = _log_int(rng, 1, 16)
    leaf = _log_int(rng, 3, 24)
    shared = _log_int(rng, 16, 1600 if op == "linprep" else 900) - paths * leaf
    return {"op": op, "shared": max(8, shared), "paths": paths, "leaf": leaf,
            **({"packed": packed} if op == "layer" else {})}


# ------------------------------------------------------------------------------------------------ inputs
class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 13)

    def f32(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std + mean

    def bf16(self, *shape, std=1.0):
        return self.f32(*shape, std=std).bfloat16()

    def weight(self, n, k):
        return self.bf16(n, k, std=0.02)


def _tree(shared, paths, leaf):
    """The packed tree of `paths` candidates behind a shared prompt: leaves of leaf - 2 .. leaf + 2 rows, rows padded
    to a multiple of 32, path slots to a multiple of 16. Index fields as the tree layout builds them: hist [N + 1, 4]
    (rows t-3 .. t on the row's path), rep_ptr [N + 2] and rep_pos [paths L2] (row -> slots, group N = padding)."""
    lens = [max(1, leaf - 2 + c * 3 % 5) for c in range(paths)]
    start = shared + np.concatenate([[0], np.cumsum(lens)[:-1]])
    N = -(-(shared + sum(lens)) // 32) * 32
    L2 = -(-(shared + max(lens)) // 16) * 16
    src = np.full((paths, L2), -1, np.int32)
    hist = np.full((N + 1, 4), -1, np.int32)
    for c in range(paths):
        path = np.concatenate([np.arange(shared), start[c] + np.arange(lens[c])])
        src[c, :len(path)] = path
        for i in range(4):
            back = 3 - i
            hist[path[back:], i] = path[:len(path) - back] if back else path
    grp = np.where(src.reshape(-1) >= 0, src.reshape(-1), N)
    rep_pos = np.argsort(grp, kind="stable").astype(np.int32)
    rep_ptr = np.concatenate([[0], np.cumsum(np.bincount(grp, minlength=N + 1))]).astype(np.int32)
    return N, L2, src, hist, rep_ptr, rep_pos


def _tree_rows(case):
    lens = [max(1, case["leaf"] - 2 + c * 3 % 5) for c in range(case["paths"])]
    rows = case["shared"] + sum(lens)
    return -(-rows // 32) * 32, case["paths"] * (-(-(case["shared"] + max(lens)) // 16) * 16)


def _raw(case, seed):
    """The inputs before any layout of this package: what both prepare() and exact() start from."""
    r, op = _Rand(seed), case["op"]
    if op == "head":
        idx = torch.randint(0, case["rows"], (case["R"],), generator=r.g, device="cuda")
        return {"hn": r.bf16(case["rows"], H), "idx": idx, "w": r.f32(H, std=0.02), "bias": r.f32(1)}
    if op == "mm":
        return {"x": r.bf16(case["M"], case["K"]), "w": r.weight(case["N"], case["K"])}
    if op == "res":
        M, N, K = case["M"], case["N"], case["K"]
        return {"x": r.bf16(M, K), "w": r.weight(N, K), "h": r.bf16(M, N), "w1": r.f32(N, std=0.1, mean=1.0)}
    if op in ("silu", "mlp2"):
        return {"x": r.bf16(case["M"], H), "gate": r.weight(I, H), "up": r.weight(I, H)}
    if op == "qkvprep":
        M = case["M"]
        ang = torch.rand(M, RD // 2, generator=r.g, device="cuda") * 6.0
        return {"x": r.bf16(M, H), "w": r.weight(QKV_N, H), "qw1": r.f32(D, std=0.1, mean=1.0),
                "kw1": r.f32(D, std=0.1, mean=1.0), "cos": torch.cat([ang.cos()] * 2, 1).bfloat16(),
                "sin": torch.cat([ang.sin()] * 2, 1).bfloat16()}
    N, L2, src, hist, rep_ptr, rep_pos = _tree(case["shared"], case["paths"], case["leaf"])
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    s = {"L2": L2, "src": dev(src), "hist": dev(hist), "rep_ptr": dev(rep_ptr), "rep_pos": dev(rep_pos),
         "convw": r.bf16(CONV, 4, std=0.5), "A_log": r.bf16(HV), "dt_bias": r.bf16(HV, std=2.0)}
    if op == "linprep":
        return {**s, "proj": r.bf16(N, LIN_N, std=1.5)}
    return {**s, "hn": r.bf16(N, H), "h": r.bf16(N, H), "y": r.bf16(N, OUT_K), "w_in": r.weight(LIN_N, H),
            "w_out": r.weight(H, OUT_K), "gate": r.weight(I, H), "up": r.weight(I, H), "w_down": r.weight(H, I),
            "w1": r.f32(H, std=0.1, mean=1.0)}


def _lin_prep(s, proj):
    return ext.linattn_prep_dedup2(proj, s["hist"], s["rep_ptr"], s["rep_pos"], s["L2"], s["convw"], s["A_log"],
                                   s["dt_bias"], KD, VD, HV, HK, HD, False)


def _layer(s):
    q, k, v, g, beta = _lin_prep(s, ext.mm(s["hn"], s["w_in"]))
    h, hn = ext.mm_residual_rmsnorm(s["h"], s["y"], s["w_out"], s["w1"], None, EPS)
    m = ext.mm_silu_mul(hn, s["w_gu"])
    h, hn = ext.mm_residual_rmsnorm(h, m, s["w_down"], s["w1"], None, EPS)
    return [q, k, v, g, beta, h, hn]


def prepare(case, seed):
    s, op = _raw(case, seed), case["op"]
    layout = ext.pack_weight if case.get("packed") else (lambda w: w)
    s["op"] = op
    for name in ("w", "w_in", "w_out", "w_down"):
        if op != "head" and name in s:
            s[name] = layout(s[name])
    if op in ("silu", "layer"):
        s["w_gu"] = layout(ext.pack_gate_up(s.pop("gate"), s.pop("up")))
    if op == "mlp2":
        s["w_gu"] = torch.cat([s.pop("gate"), s.pop("up")], 0)
        s["proj"] = fastproj.FastProjections(EPS)
        s["proj"]._tune(s["x"], s["w_gu"])
        s["proj"]._silu_tab, s["proj"]._sig_tab = ext.act_tables(s["x"])
    if op == "layer":  # once for the graph's own stream, then recorded
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _layer(s)
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["out"] = _layer(s)
    return s


def run(s):
    op = s["op"]
    if op == "head":
        return ext.head_scores(s["hn"], s["idx"], s["w"], s["bias"])
    if op == "mm":
        return ext.mm(s["x"], s["w"])
    if op == "res":
        return ext.mm_residual_rmsnorm(s["h"], s["x"], s["w"], s["w1"], None, EPS)
    if op == "silu":
        return ext.mm_silu_mul(s["x"], s["w_gu"])
    if op == "mlp2":
        return s["proj"]._silu_mul(s["proj"]._mm(s["x"], s["w_gu"]))
    if op == "qkvprep":
        return ext.mm_fullattn_prep(s["x"], s["w"], s["qw1"], s["kw1"], s["cos"], s["sin"], HQ, HKV, D, EPS)
    if op == "linprep":
        return _lin_prep(s, s["proj"])
    s["graph"].replay()
    return s["out"]


# ------------------------------------------------------------------------------------------------ work
def _gemm_work(m, n, k, out_cols):
    return 2.0 * (m * k + n * k + m * out_cols), 2.0 * m * n * k


def work(case):
    op, M = case["op"], case.get("M")
    if op == "head":
        b, f = case["R"] * (2.0 * H + 12) + 4 * H + 4, 2.0 * case["R"] * H
    elif op == "mm":
        b, f = _gemm_work(M, case["N"], case["K"], case["N"])
    elif op == "res":  # the GEMM's output is h; residual read and hn written besides
        b, f = _gemm_work(M, case["N"], case["K"], 3 * case["N"])
        b += 4 * case["N"]
    elif op in ("silu", "mlp2"):
        b, f = _gemm_work(M, 2 * I, H, I)
    elif op == "qkvprep":  # the projection itself is no output
        b, f = _gemm_work(M, QKV_N, H, (2 * HQ + 2 * HKV) * D)
        b += 4.0 * M * RD + 8 * D
    else:
        N, slots = _tree_rows(case)
        out = slots * (2.0 * CONV + 6 * HV)
        index = 16.0 * (N + 1) + 4 * (N + 2) + 4 * slots + 8 * CONV + 4 * HV
        if op == "linprep":
            b, f = N * 2.0 * (CONV + 2 * HV) + index + out, 16.0 * N * CONV
        else:
            b = 2.0 * (LIN_N * H + H * OUT_K + 2 * I * H + H * I) + 2.0 * N * (2 * H + OUT_K + 2 * H) + index + out
            f = 2.0 * N * (LIN_N * H + H * OUT_K + 2 * I * H + H * I) + 16.0 * N * CONV
    return {"bytes": float(b), "flops": float(f)}


# ------------------------------------------------------------------------------------------------ tolerance, exact
def tolerance(case):
    """Four times what the path shows against itself with its fp32 sums in other orders (other tiles and K splits, up
    to 13 of them per case): bf16 results that fall on the other side of a rounding boundary, in rel 2e-5 to 8.4e-5
    and at most 0.02 of the value or the rms for one projection, 1.1e-3 and 0.022 for a layer, where a rounding step
    of hn travels through gate-up and down. The head is one fp32 sum of 5120 terms."""
    if case["op"] == "head":
        return {"rel": 2e-6, "max": 1e-5}
    if case["op"] == "layer":
        return {"rel": 4.5e-3, "max": 0.09}
    return {"rel": 3.5e-4, "max": 0.08}


def _norm64(h, w1):
    return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * w1.double()


def _prep64(s, proj):
    """The linear-attention prep in 64 bits, from the paths themselves (src [paths, L2], -1 = padding)."""
    src = s["src"].long()
    conv = torch.zeros(*src.shape, CONV, dtype=torch.float64, device="cuda")
    for i in range(4):
        at = torch.nn.functional.pad(src, (3 - i, 0), value=-1)[:, :src.shape[1]]
        conv += proj[at.clamp(min=0), :CONV] * (at >= 0)[..., None] * s["convw"][:, i].double()
    live = (src >= 0)[..., None]
    o = torch.nn.functional.silu(conv).mul_(live)
    q, k, v = o.split([KD, KD, VD], -1)
    unit = lambda t: (lambda u: (u * torch.rsqrt(u.square().sum(-1, keepdim=True) + 1e-6)).reshape(t.shape))(  # noqa: E731
        t.reshape(*t.shape[:-1], HK, HD))
    ba = proj[src.clamp(min=0), CONV + VD:]
    beta = torch.sigmoid(ba[..., :HV]) * live
    g = -torch.exp(s["A_log"].double()) * torch.nn.functional.softplus(ba[..., HV:] + s["dt_bias"].double()) * live
    flat = lambda t: t.reshape(-1, t.shape[-1])  # noqa: E731
    return [flat(unit(q)), flat(unit(k)), flat(v), flat(g), flat(beta)]


def exact(case, seed):
    s, op = _raw(case, seed), case["op"]
    if op in ("linprep", "layer") and _tree_rows(case)[1] > 16384:
        return None  # the 64-bit slots would not fit beside the rest in comfort
    for name, t in s.items():
        if torch.is_tensor(t) and t.dtype == torch.bfloat16 and name not in ("convw", "A_log", "dt_bias"):
            s[name] = t.double()
    if op == "head":
        return s["hn"][s["idx"]] @ s["w"].double() + s["bias"].double()
    if op == "mm":
        return s["x"] @ s["w"].t()
    if op == "res":
        h = s["h"] + s["x"] @ s["w"].t()
        return [h, _norm64(h, s["w1"])]
    if op in ("silu", "mlp2"):
        return torch.nn.functional.silu(s["x"] @ s["gate"].t()) * (s["x"] @ s["up"].t())
    if op == "qkvprep":
        M = case["M"]
        p = s["x"] @ s["w"].t()
        qg, k, v = p.split([2 * HQ * D, HKV * D, HKV * D], -1)
        qg = qg.reshape(M, HQ, 2, D)
        half = RD // 2

        def rope(t, w1):
            t = _norm64(t, w1)
            rot = torch.cat([-t[..., half:RD], t[..., :half]], -1)
            a = t[..., :RD] * s["cos"][:, None] + rot * s["sin"][:, None]
            return torch.cat([a, t[..., RD:]], -1).transpose(0, 1)[None]

        return [rope(qg[:, :, 0], s["qw1"]), rope(k.reshape(M, HKV, D), s["kw1"]),
                v.reshape(M, HKV, D).transpose(0, 1)[None], qg[:, :, 1].reshape(M, HQ * D)]
    if op == "linprep":
        return _prep64(s, s["proj"])
    prep = _prep64(s, s["hn"] @ s["w_in"].t())
    h = s["h"] + s["y"] @ s["w_out"].t()
    hn = _norm64(h, s["w1"])
    h = h + (torch.nn.functional.silu(hn @ s["gate"].t()) * (hn @ s["up"].t())) @ s["w_down"].t()
    return prep + [h, _norm64(h, s["w1"])]
