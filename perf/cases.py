"""The workloads whose speed is measured: what a program that uses gpipes has it do.

Seven families, each through the public entry points of the Python mirror:

  mgn      a MeshGraphNet edge (K 384) or node (K 256) MLP, or a 128-wide one: mgn_mlp_out / mgn_mlp
  gather   the edge update with its gather front end: mgn_edge_gather
  bert     the transformer feed-forward block with residual and LayerNorm: bert_ffn_out / bert_ffn
  addln    attention output projection + add + LayerNorm + feed-forward + add + LayerNorm: bert_addln_ffn_out
  dlrm     the bottom and the top MLP of a DLRM: dlrm_botmlp_out, dlrm_topmlp_out
  nerf     the NeRF MLP, or the NerfA trunk: nerf_full_out / nerf_a_out
  stages   an edge update and a wide projection written with the stage functions, one call a layer

Rows run from a few hundred (one small graph, one sequence, one request batch, one bundle of
rays) to the benchmark sizes (about a million), odd counts among them, in fp16 and bf16.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-pipes_amd"))

import gpipes  # noqa: E402

DEV = "cuda"
TYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # The headline workload: every edge of a batch of large meshes.
        {"name": "edge_mlp_1m", "family": "mgn", "M": 1048576, "K": 384, "dtype": "fp16", "ln": True, "into": True},
        # One small graph in a rollout, a new output each step: latency, not throughput.
        {"name": "edge_mlp_1000", "family": "mgn", "M": 1000, "K": 384, "dtype": "fp16", "ln": True, "into": False},
        # The node MLP of the same batch in bf16, a row count no tile divides.
        {"name": "node_mlp_bf16", "family": "mgn", "M": 262143, "K": 256, "dtype": "bf16", "ln": True, "into": False},
        # The edge update of a mid-size mesh, int64 indices as torch keeps them.
        {"name": "edge_gather_100k", "family": "gather", "E": 100003, "N": 17011, "index": "int64", "ln": True},
        # BERT-large, 128 sequences of 512 tokens.
        {"name": "bert_ffn_65536", "family": "bert", "M": 65536, "H": 1024, "FF": 4096, "dtype": "fp16",
         "act": "gelu_tanh", "into": True},
        # BERT-large, one request of one sequence.
        {"name": "bert_ffn_509", "family": "bert", "M": 509, "H": 1024, "FF": 4096, "dtype": "bf16",
         "act": "gelu_tanh", "into": False},
        # The bert_addln_ffn app at its own batch and width.
        {"name": "bert_addln_32768", "family": "addln", "M": 32768, "H": 128, "FF": 512, "dtype": "fp16",
         "act": "relu"},
        # DLRM at its training batch, inputs padded to whole 16-byte rows.
        {"name": "dlrm_262144", "family": "dlrm", "M": 262144, "K0": 16, "K1": 480, "dtype": "fp16"},
        # DLRM answering one batch of requests, inputs as wide as the features are.
        {"name": "dlrm_2048", "family": "dlrm", "M": 2048, "K0": 13, "K1": 479, "dtype": "bf16"},
        # NeRF over the samples of a large bundle of rays.
        {"name": "nerf_1m", "family": "nerf", "M": 1048576, "trunk": False, "dtype": "fp16"},
        # NeRF over the few rays of an interactive view, 63 samples each.
        {"name": "nerf_4095", "family": "nerf", "M": 4095, "trunk": False, "dtype": "fp16"},
        # The edge update and a projection layer by layer, as a program composes its own model.
        {"name": "stages_50001", "family": "stages", "M": 50001},
    ]


def _rows(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["mgn", "gather", "bert", "addln", "dlrm", "nerf", "stages"])
    dtype = rng.choice(["fp16", "bf16"])
    if family == "mgn":
        return {"family": family, "M": _rows(rng, 200, 1048576), "K": rng.choice([128, 256, 384]), "dtype": dtype,
                "ln": rng.random() < 0.7, "into": rng.random() < 0.5}
    if family == "gather":
        E = _rows(rng, 500, 600000)
        return {"family": family, "E": E, "N": max(8, int(E / rng.uniform(3, 8))),
                "index": rng.choice(["int32", "int64"]), "ln": rng.random() < 0.7}
    if family == "bert":
        H = rng.choice([256, 512, 1024])
        return {"family": family, "M": _rows(rng, 64, 65536), "H": H, "FF": 4 * H, "dtype": dtype,
                "act": rng.choice(["relu", "gelu_tanh"]), "into": rng.random() < 0.5}
    if family == "addln":
        H = rng.choice([128, 256, 512, 1024])
        return {"family": family, "M": _rows(rng, 64, 32768), "H": H, "FF": 4 * H, "dtype": dtype,
                "act": rng.choice(["relu", "gelu_tanh"])}
    if family == "dlrm":
        return {"family": family, "M": _rows(rng, 64, 262144), "K0": rng.choice([13, 16]),
                "K1": rng.choice([479, 480]), "dtype": dtype}
    if family == "nerf":
        return {"family": family, "M": _rows(rng, 256, 1048576), "trunk": rng.random() < 0.4, "dtype": dtype}
    return {"family": family, "M": _rows(rng, 256, 262144)}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

class _Maker:
    """Seeded tensors on the GPU, rounded to the case's element type."""

    def __init__(self, seed, dtype):
        self.g = torch.Generator(device=DEV).manual_seed(seed)
        self.dt = dtype

    def normal(self, *shape, std=1.0):
        return (torch.randn(shape, generator=self.g, device=DEV) * std).to(self.dt)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return (torch.rand(shape, generator=self.g, device=DEV) * (hi - lo) + lo).to(self.dt)

    def linear(self, k, n):
        """nn.Linear's default init, the weight as [in, out]."""
        a = 1.0 / math.sqrt(k)
        return self.uniform(k, n, lo=-a, hi=a), self.uniform(n, lo=-a, hi=a)

    def xavier(self, k, n):
        a = math.sqrt(6.0 / (k + n))
        return self.uniform(k, n, lo=-a, hi=a), self.uniform(n, lo=-1.0 / math.sqrt(k), hi=1.0 / math.sqrt(k))

    def affine(self, n):
        """A trained LayerNorm's gamma and beta: near 1 and near 0."""
        return self.normal(n, std=0.1) + 1, self.normal(n, std=0.1)

    def encoded(self, rows, octaves, width, unit=False):
        """Positional encoding of points in the unit cube (or directions), zero-padded to `width`."""
        p = torch.rand((rows, 3), generator=self.g, device=DEV) * 2 - 1
        if unit:
            p = p / p.norm(dim=1, keepdim=True).clamp_min(1e-6)
        f = [p] + [fn((2.0 ** i) * p) for i in range(octaves) for fn in (torch.sin, torch.cos)]
        out = torch.zeros((rows, width), device=DEV)
        out[:, :3 + 6 * octaves] = torch.cat(f, dim=1)
        return out.to(self.dt)


NERF_KX, NERF_KD = 64, 27


def _nerf_shapes(trunk):
    s = [(NERF_KX, 256)] + [(256, 256)] * 4 + [(256 + NERF_KX, 256), (256, 256), (256, 256)]
    return s if trunk else s + [(256, 1), (256, 256), (256 + NERF_KD, 128), (128, 3)]


DLRM_BOT, DLRM_TOP = (512, 256, 128), (1024, 1024, 512, 256, 1)


def _inputs(case, seed):
    f = case["family"]
    m = _Maker(seed, TYPES[case.get("dtype", "fp16")])
    s = {"family": f, "case": case}
    if f == "mgn":
        s["x"] = m.normal(case["M"], case["K"])
        s["wb"] = [t for k in (case["K"], 128, 128) for t in m.linear(k, 128)]
        s["affine"] = m.affine(128) if case["ln"] else (None, None)
    elif f == "gather":
        it = torch.int32 if case["index"] == "int32" else torch.int64
        s["nf"], s["ef"] = m.normal(case["N"], 128), m.normal(case["E"], 128)
        s["src"], s["dst"] = (torch.randint(0, case["N"], (case["E"],), generator=m.g, device=DEV).to(it)
                              for _ in range(2))
        s["wb"] = [t for k in (384, 128, 128) for t in m.linear(k, 128)]
        s["affine"] = m.affine(128) if case["ln"] else (None, None)
    elif f == "bert":
        H, FF = case["H"], case["FF"]
        s["x"] = m.normal(case["M"], H)
        s["wb"] = [m.normal(H, FF, std=0.02), m.normal(FF, std=0.02), m.normal(FF, H, std=0.02), m.normal(H, std=0.02)]
        s["affine"] = m.affine(H)
    elif f == "addln":
        H, FF = case["H"], case["FF"]
        s["attn"], s["x"] = m.normal(case["M"], H), m.normal(case["M"], H)
        s["wb"] = [t for k, n in ((H, H), (H, FF), (FF, H)) for t in m.linear(k, n)]
        s["affine"] = m.affine(H) + m.affine(H)
    elif f == "dlrm":
        M = case["M"]
        s["dense"] = m.uniform(M, case["K0"])
        s["dense"][:, 13:] = 0
        s["x"] = m.normal(M, case["K1"])
        s["x"][:, 479:] = 0
        for key, w in (("bot", (case["K0"],) + DLRM_BOT), ("top", (case["K1"],) + DLRM_TOP)):
            s[key] = [t for k, n in zip(w, w[1:]) for t in m.xavier(k, n)]
    elif f == "nerf":
        s["x"] = m.encoded(case["M"], 10, NERF_KX)
        if not case["trunk"]:
            s["d"] = m.encoded(case["M"], 4, NERF_KD, unit=True)
        s["wb"] = [t for k, n in _nerf_shapes(case["trunk"]) for t in m.linear(k, n)]
    else:
        M = case["M"]
        s["nodes"], s["ef"] = m.normal(M, 256), m.normal(M, 128)
        s["wb"] = [t for k, n in ((384, 128), (128, 128), (128, 128), (128, 512)) for t in m.linear(k, n)]
        s["affine"] = m.affine(128) + m.affine(512)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    f, dt = case["family"], TYPES[case.get("dtype", "fp16")]

    def buf(rows, cols):
        return torch.empty((rows, cols), dtype=dt, device=DEV)

    if f == "mgn" and case["into"]:
        s["out"] = buf(case["M"], 128)
    elif f == "bert" and case["into"]:
        s["out"] = buf(case["M"], case["H"])
    elif f == "addln":
        s["out"] = buf(case["M"], case["H"])
    elif f == "dlrm":
        s["out"] = buf(case["M"], 128), buf(case["M"], 1)
    elif f == "nerf":
        s["out"] = (buf(case["M"], 256),) if case["trunk"] else (buf(case["M"], 1), buf(case["M"], 3))
    return s


def run(s):
    f, case = s["family"], s["case"]
    if f == "mgn":
        if case["into"]:
            return gpipes.mgn_mlp_out(s["x"], *s["wb"], *s["affine"], s["out"])
        return gpipes.mgn_mlp(s["x"], *s["wb"], *s["affine"])
    if f == "gather":
        return gpipes.mgn_edge_gather(s["nf"], s["ef"], s["src"], s["dst"], *s["wb"], *s["affine"])
    if f == "bert":
        if case["into"]:
            return gpipes.bert_ffn_out(s["x"], *s["wb"], *s["affine"], s["out"], eps=1e-12, act=case["act"])
        return gpipes.bert_ffn(s["x"], *s["wb"], *s["affine"], eps=1e-12, act=case["act"])
    if f == "addln":
        return gpipes.bert_addln_ffn_out(s["attn"], s["x"], *s["wb"], *s["affine"], s["out"], act=case["act"])
    if f == "dlrm":
        return [gpipes.dlrm_botmlp_out(s["dense"], *s["bot"], s["out"][0]),
                gpipes.dlrm_topmlp_out(s["x"], *s["top"], s["out"][1], act5="sigmoid")]
    if f == "nerf":
        if case["trunk"]:
            return gpipes.nerf_a_out(s["x"], *s["wb"], s["out"][0])
        return list(gpipes.nerf_full_out(s["x"], s["d"], *s["wb"], *s["out"], rgb_act="sigmoid"))
    w1, b1, w2, b2, w3, b3, wp, bp = s["wb"]
    g1, be1, g2, be2 = s["affine"]
    h = gpipes.concat_out(s["nodes"], s["ef"])
    h = gpipes.linear_out(h, w1, b1, act="relu")
    h = gpipes.linear_out(h, w2, b2, act="relu")
    e = gpipes.add_out(gpipes.linear_layer_norm_out(h, w3, b3, g1, be1), s["ef"])
    p = gpipes.gemm_out(e, wp, bp, act="gelu_tanh")
    return [e, gpipes.layer_norm_out(p, g2, be2)]


# ---------------------------------------------------------------------------
# Work, tolerance and the 64-bit result
# ---------------------------------------------------------------------------

def _chain(M, widths):
    """(16-bit values of the weights and biases, flops) of a dense chain."""
    return (sum(k * n + n for k, n in zip(widths, widths[1:])), sum(2 * M * k * n for k, n in zip(widths, widths[1:])))


def work(case):
    f = case["family"]
    if f == "mgn":
        M, K = case["M"], case["K"]
        p, fl = _chain(M, (K, 128, 128, 128))
        return {"bytes": 2 * (M * (K + 128) + p + 256 * case["ln"]), "flops": fl}
    if f == "gather":
        E = case["E"]
        p, fl = _chain(E, (384, 128, 128, 128))
        return {"bytes": 2 * (256 * E + 128 * case["N"] + p + 256 * case["ln"]) +
                2 * E * (4 if case["index"] == "int32" else 8), "flops": fl}
    if f == "bert":
        M, H, FF = case["M"], case["H"], case["FF"]
        p, fl = _chain(M, (H, FF, H))
        return {"bytes": 2 * (2 * M * H + p + 2 * H), "flops": fl}
    if f == "addln":
        M, H, FF = case["M"], case["H"], case["FF"]
        p, fl = _chain(M, (H, H, FF, H))
        return {"bytes": 2 * (3 * M * H + p + 4 * H), "flops": fl}
    if f == "dlrm":
        M = case["M"]
        p0, f0 = _chain(M, (case["K0"],) + DLRM_BOT)
        p1, f1 = _chain(M, (case["K1"],) + DLRM_TOP)
        return {"bytes": 2 * (M * (case["K0"] + 128 + case["K1"] + 1) + p0 + p1), "flops": f0 + f1}
    if f == "nerf":
        M, shapes = case["M"], _nerf_shapes(case["trunk"])
        io = NERF_KX + (256 if case["trunk"] else NERF_KD + 4)
        return {"bytes": 2 * (M * io + sum(k * n + n for k, n in shapes)),
                "flops": sum(2 * M * k * n for k, n in shapes)}
    # every stage function reads its inputs and writes its output
    M = case["M"]
    shapes = ((384, 128), (128, 128), (128, 128), (128, 512))
    io = 2 * 384 + sum(k + n for k, n in shapes) + 3 * 128 + 2 * 512
    return {"bytes": 2 * (M * io + sum(k * n + n for k, n in shapes) + 2 * (128 + 512)),
            "flops": sum(2 * M * k * n for k, n in shapes)}


def tolerance(case):
    # About four times the distance to exact(): 2.5e-4 to 5e-4 in fp16, 1.9e-3 to 3.3e-3 in bf16.
    return {"rel": 1e-2 if case.get("dtype", "fp16") == "bf16" else 2e-3}


def _act(v, act):
    if act == "relu":
        return torch.relu(v)
    if act == "gelu_tanh":
        return torch.nn.functional.gelu(v, approximate="tanh")
    return torch.sigmoid(v) if act == "sigmoid" else v


def _norm(v, g, b, eps):
    return torch.nn.functional.layer_norm(v, (v.shape[-1],), None if g is None else g.double(),
                                          None if b is None else b.double(), eps)


def _dense(v, wb, acts):
    for w, b, a in zip(wb[::2], wb[1::2], acts):
        v = _act(v @ w.double() + b.double(), a)
    return v


def _exact_rows(s, r):
    """run()'s outputs for rows `r` (a slice), in 64 bits."""
    f, case, R = s["family"], s["case"], ["relu"]
    if f in ("mgn", "gather"):
        if f == "mgn":
            v = s["x"][r].double()
        else:
            v = torch.cat([s["nf"][s["src"][r].long()], s["ef"][r], s["nf"][s["dst"][r].long()]], 1).double()
        v = _dense(v, s["wb"], R * 2 + ["none"])
        return [_norm(v, *s["affine"], 1e-5) if case["ln"] else v]
    if f == "bert":
        x = s["x"][r].double()
        return [_norm(_dense(x, s["wb"], [case["act"], "none"]) + x, *s["affine"], 1e-12)]
    if f == "addln":
        h = _norm(_dense(s["attn"][r].double(), s["wb"][:2], ["none"]) + s["x"][r].double(), *s["affine"][:2], 1e-5)
        return [_norm(_dense(h, s["wb"][2:], [case["act"], "none"]) + h, *s["affine"][2:], 1e-5)]
    if f == "dlrm":
        return [_dense(s["dense"][r].double(), s["bot"], R * 3),
                _dense(s["x"][r].double(), s["top"], R * 4 + ["sigmoid"])]
    if f == "nerf":
        x, wb = s["x"][r].double(), s["wb"]
        h = _dense(x, wb[:10], R * 5)
        h = _dense(torch.cat([h, x], 1), wb[10:16], R * 3)
        if case["trunk"]:
            return [h]
        c = torch.cat([_dense(h, wb[18:20], ["none"]), s["d"][r].double()], 1)
        return [_dense(h, wb[16:18], ["none"]), _dense(c, wb[20:24], ["relu", "sigmoid"])]
    e = _dense(torch.cat([s["nodes"][r], s["ef"][r]], 1).double(), s["wb"][:6], R * 2 + ["none"])
    e = _norm(e, *s["affine"][:2], 1e-5) + s["ef"][r].double()
    return [e, _norm(_dense(e, s["wb"][6:], ["gelu_tanh"]), *s["affine"][2:], 1e-5)]


def exact(case, seed):
    s = _inputs(case, seed)
    M = case["E"] if case["family"] == "gather" else case["M"]
    step = 65536
    parts = [_exact_rows(s, slice(r, min(r + step, M))) for r in range(0, M, step)]
    outs = [torch.cat(p) for p in zip(*parts)]
    return outs if case["family"] in ("dlrm", "nerf", "stages") and len(outs) > 1 else outs[0]
