"""Performance cases of the optimizer step and of what surrounds it, through the public entry points.

A case is a dict of plain values; `kind` selects the entry point:

    minimal   HybridOptimizer with everything at its defaults: fp32 gradients from host arrays, Keller
              coefficients, unguarded, synchronous
    hybrid    HybridOptimizer with resident gradients: global norm, clip, skip guard, Muon, AdamW
    resident  ResidentMuon.step: one weight at a time over a shared scratch
    proj      BatchedProjMuon.step over the projections of a stack of layers
    expert    ExpertOptimizer.step: stacked expert tensors, transposed copies, router
    ns        newton_schulz_resident_e: the bare chain, bf16 in and out
    adamw     StepGuard.compute + AdamW.step over one flat tensor
    dw        gemm_dW: the weight gradients of one layer, or of a single weight
    embed     one step of the input embedding: id groups, catch-up, scatter, row-sparse AdamW
    quant     Mxfp8WeightCache.refresh after a step

Models of more than one layer hold their weights stacked over the layers, [L, K, N] per projection:
the optimizer takes such a tensor as L matrices.
"""
import math

import numpy as np
import torch

import ancora_cutile_amd as anc
from ancora_cutile_amd.adamw import AdamW
from ancora_cutile_amd.embed import IdGroups, RowSparseAdamW, embed_dw_scatter
from ancora_cutile_amd.gradnorm import StepGuard
from ancora_cutile_amd.grads import DwWorkspace, gemm_dW
from ancora_cutile_amd.hybrid import resident_is_muon
from ancora_cutile_amd.moe import ExpertOptimizer
from ancora_cutile_amd.muon_ns import NsWorkspace, newton_schulz_resident_e
from ancora_cutile_amd.quant import Mxfp8WeightCache

DEV = "cuda"


def listed():
    return [
        # The smallest hybrid model: one AdamW matrix, one gain, one Muon matrix, everything default.
        # What a first program does; host time, uploads and launches count.
        dict(name="minimal_1024", kind="minimal", K=1024, N=1024),
        # A small model trained for experiments: short kernels, few matrices per shape.
        dict(name="hybrid_small", kind="hybrid", layers=4, hidden=512, ffn=1536, q=512, kv=256, head_dim=64,
             vocab=8192, experts=0, polar=True, bf16=True, sr=True),
        # The full step of the Qwen3-0.6B parameter set: 596 M parameters, 196 Muon matrices.
        dict(name="hybrid_qwen3_0p6b", kind="hybrid", layers=28, hidden=1024, ffn=3072, q=2048, kv=1024,
             head_dim=128, vocab=151936, experts=0, polar=True, bf16=True, sr=True),
        # One weight, as a layer that steps itself right after its backward does it; Keller's
        # coefficients, which are the default.
        dict(name="resident_1024x3072", kind="resident", K=1024, N=3072, polar=False),
        # The projections of a few layers of a width that is no power of two, in the default chunks.
        dict(name="proj_640", kind="proj", layers=6, hidden=640, ffn=1792, q=640, kv=384, polar=True),
        # One mixture-of-experts layer.
        dict(name="expert_16x1024", kind="expert", E=16, H=1024, Ie=1024, polar=True, muon=True),
        # The bare chain on a stack of wide matrices.
        dict(name="ns_24x1024x2048", kind="ns", E=24, M=1024, N=2048, polar=True),
        # The flat AdamW sweep of a large parameter shard, with norm, clip and stochastic rounding.
        dict(name="adamw_1p2e9", kind="adamw", n=1200000000, bf16=True, sr=True, div=True),
        # The backward's weight gradients: a whole layer in one call at a training batch.
        dict(name="dw_layer_8192", kind="dw", T=8192, hidden=1024, ffn=3072, q=2048, kv=1024, accumulate=True),
        # A single weight at a short and ragged batch, as a small model or the last micro-batch gives it.
        dict(name="dw_one_1504", kind="dw", T=1504, hidden=640, ffn=1792, q=0, kv=0, accumulate=False),
        # The input embedding of a large vocabulary at a training batch.
        dict(name="embed_8192", kind="embed", V=151936, H=1024, M=8192),
        # The fp8 copies of four layers' weights, refreshed before the next forward.
        dict(name="quant_4_layers", kind="quant", layers=4, hidden=1024, ffn=3072, q=2048, kv=1024,
             col_major=False),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _mult(rng, lo, hi, of):
    """A multiple of `of` in lo .. hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(_log(rng, lo, hi) / of)) * of))


def _model(rng, of, widest):
    hidden = _mult(rng, 256, widest, of)
    return dict(hidden=hidden, ffn=_mult(rng, hidden, 3 * hidden, of), q=_mult(rng, hidden, 2 * hidden, of),
                kv=_mult(rng, 256, hidden, of))


def draw(rng):
    kind = rng.choice(("minimal", "hybrid", "hybrid", "resident", "proj", "expert", "ns", "adamw", "dw", "dw",
                       "embed", "quant"))
    polar = rng.random() < 0.5
    if kind == "minimal":
        return dict(kind=kind, K=_mult(rng, 64, 2048, 64), N=_mult(rng, 64, 2048, 64))
    if kind == "hybrid":
        m = _model(rng, 128, 1280)
        experts = rng.choice((0, 0, 8))
        most = max(2, int(2.5e8 / (6 * m["hidden"] * m["ffn"] * (1 + experts // 2))))
        return dict(kind=kind, layers=int(_log(rng, 1, min(24, most))), head_dim=rng.choice((64, 128)),
                    vocab=_mult(rng, 1000, 100000, 8), experts=experts, polar=polar, bf16=rng.random() < 0.7,
                    sr=rng.random() < 0.5, **m)
    if kind == "resident":
        return dict(kind=kind, K=_mult(rng, 128, 4096, 128), N=_mult(rng, 128, 4096, 128), polar=polar)
    if kind == "proj":
        return dict(kind=kind, layers=rng.randint(1, 8), polar=polar, **_model(rng, 128, 1152))
    if kind == "expert":
        H = _mult(rng, 256, 1280, 128)
        return dict(kind=kind, E=rng.randint(2, 16), H=H, Ie=H, polar=polar, muon=rng.random() < 0.7)
    if kind == "ns":
        M = _mult(rng, 128, 1536, 128)
        return dict(kind=kind, E=int(_log(rng, 1, 24)), M=M, N=_mult(rng, M, 3 * M, 128), polar=polar)
    if kind == "adamw":
        return dict(kind=kind, n=_mult(rng, 64, 1000000000, 64), bf16=rng.random() < 0.7,
                    sr=rng.random() < 0.5, div=rng.random() < 0.7)
    if kind == "dw":
        m = _model(rng, 256, 1024)
        if rng.random() < 0.5:
            m.update(q=0, kv=0)
        return dict(kind=kind, T=_mult(rng, 32, 8192, 32), accumulate=rng.random() < 0.5, **m)
    if kind == "embed":
        return dict(kind=kind, V=int(_log(rng, 1000, 151936)), H=_mult(rng, 64, 1024, 64), M=int(_log(rng, 16, 8192)))
    return dict(kind=kind, layers=rng.randint(1, 4), col_major=rng.random() < 0.5, **_model(rng, 128, 1280))


# ---------------------------------------------------------------- parameter sets
def _projections(c, layers):
    h, f, q, kv = c["hidden"], c["ffn"], c["q"], c["kv"]
    return {"q_proj": (layers, h, q), "k_proj": (layers, h, kv), "v_proj": (layers, h, kv),
            "o_proj": (layers, q, h), "gate_proj": (layers, h, f), "up_proj": (layers, h, f),
            "down_proj": (layers, f, h)}


def _hybrid_shapes(c):
    """{name: shape}: with experts, every second layer has an expert FFN in place of the dense one."""
    L, h = c["layers"], c["hidden"]
    moe = L // 2 if c["experts"] else 0
    s = {"embed": (c["vocab"], h), "input_ln": (L, h), "q_norm": (L, c["head_dim"]), "k_norm": (L, c["head_dim"]),
         "post_ln": (L, h), "final_norm": (h,)}
    s.update(_projections(c, L))
    for n in ("gate_proj", "up_proj", "down_proj"):
        s[n] = (L - moe,) + s[n][1:]
    if moe:
        E = c["experts"]
        s["ffn.router"] = (moe, h, E)
        s["ffn.gate_proj"] = s["ffn.up_proj"] = s["ffn.down_proj"] = (moe * E, h, h)
    return s


def _is_gain(name):
    return name.endswith(("ln", "norm"))


def _grad(gen, shape, bf16):
    """A gradient: N(0, 1e-3), 1 % of the rows of a matrix x100."""
    g = 1e-3 * torch.randn(shape, generator=gen, device=DEV)
    if len(shape) > 1:
        rows = g.view(-1, shape[-1])
        k = max(1, rows.shape[0] // 100)
        rows[torch.randperm(rows.shape[0], generator=gen, device=DEV)[:k]] *= 100.0
    return g.to(torch.bfloat16) if bf16 else g


_NP = {torch.float32: np.float32, torch.bfloat16: np.uint16, torch.int32: np.int32, torch.uint8: np.uint8}


def _buf(t):
    """The library's view of a torch tensor (bf16 as bit patterns); the tensor stays the owner."""
    return anc.DevBuf(shape=tuple(t.shape), dtype=_NP[t.dtype], ptr=t.data_ptr())


class _Cai:
    def __init__(self, buf, owners):
        self.owners = owners        # the memory lives as long as a tensor that shows it
        code = "<i2" if buf.dtype == np.uint16 else buf.dtype.str
        self.__cuda_array_interface__ = {"shape": buf.shape, "typestr": code, "data": (buf.ptr, False), "version": 2}


def _tensor(buf, owners=None):
    """torch's view of a library buffer; uint16 buffers hold bf16."""
    t = torch.as_tensor(_Cai(buf, owners), device=DEV)
    return t.view(torch.bfloat16) if buf.dtype == np.uint16 else t


def _fill_master(gen, p32, p16, gain=False):
    """Random weights in a master buffer and its bf16 copy, as a resumed run has them."""
    w = _tensor(p32)
    w.normal_(1.0 if gain else 0.0, 0.05 if gain else 0.02, generator=gen)
    _tensor(p16).copy_(w.view(_tensor(p16).shape))


class Owners:
    """The library objects of a state, given back when the state and its outputs are gone."""

    def __init__(self, *objects):
        self.objects = objects

    def __del__(self):
        torch.cuda.synchronize()
        for o in self.objects:
            o.free()


class State:
    """Whatever a case keeps between passes: `go` makes one, `out` is what it writes."""

    def __init__(self, go, out, *kept):
        self.go, self.out, self.kept = go, out, kept


# ---------------------------------------------------------------- prepare / run per kind
def _hybrid_out(opt, owners):
    out = {}
    for part, keys in ((opt.muon, ("p32", "p16", "buf")), (opt.adamw, ("p32", "p16", "m", "v"))):
        for n, st in part.st.items():
            out[n] = [_tensor(st[k], owners) for k in keys]
    return out


def _prepare_minimal(c, gen):
    K, N = c["K"], c["N"]
    host = {"lm_head": (K, N), "norm": (N,), "w": (K, N)}
    params = {n: (0.02 * torch.randn(sh, generator=gen, device=DEV) + (n == "norm")).cpu().numpy()
              for n, sh in host.items()}
    grads = {n: _grad(gen, sh, False).cpu().numpy() for n, sh in host.items()}
    opt = anc.HybridOptimizer(params)
    return State(lambda: opt.step(grads, 0), _hybrid_out(opt, Owners(opt)))


def _prepare_hybrid(c, gen):
    shapes = _hybrid_shapes(c)
    opt = anc.HybridOptimizer(
        {n: np.zeros(sh, np.float32) for n, sh in shapes.items()}, is_muon=resident_is_muon,
        no_decay=lambda n, p: _is_gain(n) or "router" in n,
        muon_kw=dict(lr=0.02, momentum=0.95, ns_steps=5, schedule=anc.PE_SCHEDULE if c["polar"] else None,
                     sr=c["sr"], seed=1),
        adamw_kw=dict(lr=3e-4, betas=(0.9, 0.95), eps=1e-8, wd=0.1, sr=c["sr"], seed=2),
        max_grad_norm=1.0, grad_dtype=np.uint16 if c["bf16"] else np.float32)
    for part in (opt.muon, opt.adamw):
        for n, st in part.st.items():
            _fill_master(gen, st["p32"], st["p16"], _is_gain(n))
    kept = {n: _grad(gen, sh, c["bf16"]) for n, sh in shapes.items()}
    grads = {n: _buf(t) for n, t in kept.items()}
    return State(lambda: opt.step(grads, 0, sync=False), _hybrid_out(opt, Owners(opt)), kept)


def _prepare_resident(c, gen):
    K, N = c["K"], c["N"]
    p32, p16 = anc.DevBuf.empty((K, N), np.float32), anc.DevBuf.empty((K, N), np.uint16)
    _fill_master(gen, p32, p16)
    scratch = anc.MuonScratch([(K, N)])
    opt = anc.ResidentMuon(p32, p16, K, N, scratch)
    kept = _grad(gen, (K, N), False)
    g = _buf(kept)
    owners = Owners(opt, scratch, p32, p16)
    sched = anc.PE_SCHEDULE if c["polar"] else None
    return State(lambda: opt.step(g, 0, schedule=sched), [_tensor(b, owners) for b in (p32, p16, opt.buf)], kept)


def _prepare_proj(c, gen):
    stacks, recs = {}, []
    for n, (L, K, N) in _projections(c, c["layers"]).items():
        b = dict(p32=anc.DevBuf.empty((L * K, N), np.float32), p16=anc.DevBuf.empty((L * K, N), np.uint16),
                 buf=anc.DevBuf.zeros((L * K, N), np.float32))
        _fill_master(gen, b["p32"], b["p16"])
        b["g"] = _grad(gen, (L * K, N), False)
        stacks[n] = b
    for lid in range(c["layers"]):
        for n, (L, K, N) in _projections(c, c["layers"]).items():
            b = stacks[n]
            recs.append(dict(buf=b["buf"].at_pos(lid * K), p32=b["p32"].at_pos(lid * K),
                             p16=b["p16"].at_pos(lid * K), G=_buf(b["g"]).at_pos(lid * K), K=K, N=N, lid=lid))
    opt = anc.BatchedProjMuon(recs)
    owners = Owners(opt, *[b[k] for b in stacks.values() for k in ("p32", "p16", "buf")])
    sched = anc.PE_SCHEDULE if c["polar"] else None
    return State(lambda: opt.step(0, schedule=sched),
                 {n: [_tensor(b[k], owners) for k in ("p32", "p16", "buf")] for n, b in stacks.items()},
                 [b["g"] for b in stacks.values()])


def _prepare_expert(c, gen):
    E, H, Ie = c["E"], c["H"], c["Ie"]
    shapes = {"gate_proj": (E, H, Ie), "up_proj": (E, H, Ie), "down_proj": (E, Ie, H)}
    opt = ExpertOptimizer({n: np.zeros(sh, np.float32) for n, sh in shapes.items()},
                          router=np.zeros((H, E), np.float32), optimizer="muon" if c["muon"] else "adamw")
    for st in list(opt.st.values()) + [opt.router]:
        _fill_master(gen, st["p32"], st["p16"])
    kept = {n: _grad(gen, sh, False) for n, sh in shapes.items()}
    for t in kept.values():
        t[:E // 4] = 0.0                           # experts that no token reached
    kept["router"] = _grad(gen, tuple(opt.router["p32"].shape), False)
    grads = {n: _buf(t) for n, t in kept.items()}
    owners = Owners(opt)
    out = {n: [_tensor(st[k], owners) for k in ("p32", "p16", "p16T", "buf", "m", "v") if k in st]
           for n, st in list(opt.st.items()) + [("router", opt.router)]}
    sched = anc.PE_SCHEDULE if c["polar"] else None
    return State(lambda: opt.step(grads, 0, router_grad=grads["router"], schedule=sched), out, kept)


def _prepare_ns(c, gen):
    E, M, N = c["E"], c["M"], c["N"]
    ws = NsWorkspace()
    owners = Owners(ws)
    src = torch.randn((E * M, N), generator=gen, device=DEV).to(torch.bfloat16)
    work_buf = torch.empty_like(src)
    x = _buf(work_buf)
    sched = anc.PE_SCHEDULE if c["polar"] else None

    def go():
        work_buf.copy_(src)                        # the chain works in place: a new momentum every step
        newton_schulz_resident_e(x, None, None, None, None, None, E, M, N, 0, schedule=sched, workspace=ws)
    return State(go, [work_buf], owners)


def _prepare_adamw(c, gen):
    n = c["n"]
    opt = AdamW({"flat": np.zeros(n, np.float32)}, lr=3e-4, betas=(0.9, 0.95), eps=1e-8, wd=0.1, sr=c["sr"], seed=3,
                form="div" if c["div"] else "ibc", grad_dtype=np.uint16 if c["bf16"] else np.float32)
    guard = StepGuard(1.0)
    st = opt.st["flat"]
    _fill_master(gen, st["p32"], st["p16"])
    kept = _grad(gen, (n,), c["bf16"])
    g = _buf(kept)
    owners = Owners(opt, guard)

    def go():
        guard.compute([g], 0)
        opt.step({"flat": g}, 0, guard)
    return State(go, [_tensor(st[k], owners) for k in ("p32", "p16", "m", "v")], kept)


def _dw_weights(c):
    if c["q"]:
        return [sh[1:] for sh in _projections(c, 1).values()]
    return [(c["hidden"], c["ffn"])]


def _prepare_dw(c, gen):
    T = c["T"]
    acts, problems, out, workspaces = {}, [], [], []
    for K, N in _dw_weights(c):
        if K not in acts:                          # weights of one input width share the activations
            acts[K] = torch.randn((T, K), generator=gen, device=DEV).to(torch.bfloat16)
        dy = (1e-3 * torch.randn((T, N), generator=gen, device=DEV)).to(torch.bfloat16)
        dW, g16 = torch.zeros((K, N), device=DEV), torch.zeros((K, N), device=DEV, dtype=torch.bfloat16)
        workspaces.append(DwWorkspace())
        out.append([dW, g16])
        problems.append(dict(x=_buf(acts[K]), dy=_buf(dy), dW=_buf(dW), g16=_buf(g16), T=T, K=K, N=N,
                             workspace=workspaces[-1], accumulate=c["accumulate"], kept=(acts[K], dy)))
    return State(lambda: gemm_dW(problems, 0), out, Owners(*workspaces))


def _prepare_embed(c, gen):
    V, H, M = c["V"], c["H"], c["M"]
    opt = RowSparseAdamW(np.zeros((V, H), np.float32), lr=3e-4, wd=0.1, max_steps=1 << 19)
    _fill_master(gen, opt.p32, opt.p16)
    # a few batches in turn: frequent ids come back, rare ones are caught up when they do
    ids = [(V * torch.rand(M, generator=gen, device=DEV) ** 3).long().clamp(max=V - 1).cpu().numpy().astype(np.int32)
           for _ in range(4)]
    dys = [(1e-3 * torch.randn((M, H), generator=gen, device=DEV)).to(torch.bfloat16) for _ in range(4)]
    dy_bufs = [_buf(d) for d in dys]
    rows = torch.zeros((M, H), device=DEV)
    compact = _buf(rows)
    owners = Owners(opt)
    turn = [0]

    def go():
        i = turn[0] % 4
        turn[0] += 1
        opt.catch_up(ids[i], 0)                    # before the forward reads the rows
        groups = IdGroups(ids[i])
        embed_dw_scatter(groups, dy_bufs[i], 0, compact=compact)
        opt.step(groups.gid, groups.n_groups, compact, 0)
        groups.free()
    return State(go, [_tensor(b, owners) for b in (opt.p32, opt.p16, opt.m, opt.v, opt.last)] + [rows], dys)


def _prepare_quant(c, gen):
    w, kept = {}, {}
    for lid in range(c["layers"]):
        for n, (_, K, N) in _projections(c, 1).items():
            t = (0.02 * torch.randn((K, N), generator=gen, device=DEV)).to(torch.bfloat16)
            kept[f"layer{lid}.{n}"] = t
            w[f"layer{lid}.{n}"] = dict(p16=_buf(t), K=K, N=N)
    cache = Mxfp8WeightCache(w, col_major=c["col_major"])
    owners = Owners(cache)

    def go():
        cache.mark_dirty()
        cache.refresh(0)
    return State(go, [[_tensor(cache.fp8(n), owners), _tensor(cache.scale(n), owners)] for n in w], kept)


_PREPARE = dict(minimal=_prepare_minimal, hybrid=_prepare_hybrid, resident=_prepare_resident, proj=_prepare_proj,
                expert=_prepare_expert, ns=_prepare_ns, adamw=_prepare_adamw, dw=_prepare_dw, embed=_prepare_embed,
                quant=_prepare_quant)


def prepare(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    return _PREPARE[case["kind"]](case, gen)


def run(state):
    state.go()
    return state.out


# ---------------------------------------------------------------- work and tolerance
def _chain_flops(M, N, steps=5):
    """A and B are symmetric: half of their entries."""
    M, N = min(M, N), max(M, N)
    return steps * (3.0 * M * M * N + 1.0 * M ** 3)


def work(case):
    c, kind = case, case["kind"]
    if kind == "minimal":
        n = c["K"] * c["N"]
        return {"bytes": 24.0 * n + 30.0 * (n + c["N"]), "flops": _chain_flops(c["K"], c["N"])}
    if kind == "hybrid":
        gb, by, fl = (2 if c["bf16"] else 4), 0.0, 0.0
        for n, sh in _hybrid_shapes(c).items():
            size = float(np.prod(sh))
            if len(sh) == 3 and "router" not in n:
                by += size * (gb + 18)             # buf, p32 read and written, p16 written
                fl += sh[0] * _chain_flops(sh[1], sh[2])
            else:
                by += size * (gb + 26)             # m, v, p32 read and written, p16 written
        return {"bytes": by, "flops": fl}
    if kind == "resident":
        return {"bytes": 22.0 * c["K"] * c["N"], "flops": _chain_flops(c["K"], c["N"])}
    if kind == "proj":
        shapes = _projections(c, c["layers"]).values()
        return {"bytes": sum(22.0 * L * K * N for L, K, N in shapes),
                "flops": sum(L * _chain_flops(K, N) for L, K, N in shapes)}
    if kind == "expert":
        n, r = 3.0 * c["E"] * c["H"] * c["Ie"], 30.0 * c["H"] * c["E"]
        if not c["muon"]:
            return {"bytes": 32.0 * n + r, "flops": 15.0 * n}
        return {"bytes": 24.0 * n + r, "flops": 3 * c["E"] * _chain_flops(c["H"], c["Ie"])}
    if kind == "ns":
        return {"bytes": 4.0 * c["E"] * c["M"] * c["N"], "flops": c["E"] * _chain_flops(c["M"], c["N"])}
    if kind == "adamw":
        return {"bytes": (28.0 if c["bf16"] else 30.0) * c["n"], "flops": 15.0 * c["n"]}
    if kind == "dw":
        ws = _dw_weights(c)
        by = sum(K * N * (10.0 if c["accumulate"] else 6.0) + 2.0 * c["T"] * N for K, N in ws)
        return {"bytes": by + sum(2.0 * c["T"] * K for K in set(K for K, _ in ws)),
                "flops": sum(2.0 * c["T"] * K * N for K, N in ws)}
    if kind == "embed":
        # distinct ids of the batch (u^3 over V): their rows' state, the gradient rows, the compact rows
        n, edge = 0.0, np.linspace(0.0, 1.0, 4097)
        p = (edge ** (1.0 / 3.0))[1:] - (edge ** (1.0 / 3.0))[:-1]
        per = c["V"] / 4096.0
        n = float(np.sum(per * -np.expm1(-c["M"] * p / per)))
        return {"bytes": c["H"] * (2.0 * c["M"] + n * (4.0 + 26.0)) + 20.0 * c["M"], "flops": c["H"] * (c["M"] + 15.0 * n)}
    n = sum(K * N for _, K, N in _projections(c, 1).values()) * float(c["layers"])
    return {"bytes": n * (3.0 + 1.0 / 32.0), "flops": 2.0 * n}


def tolerance(case):
    kind = case["kind"]
    if kind == "quant":
        return "exact"
    if kind == "ns":
        # bf16 matrix-core chain: each result within 2e-3 of the exact one, then rounded to bf16
        return {"rel": 4e-3, "max": 0.1}
    if kind == "adamw" or kind == "embed" or kind == "dw" or (kind == "expert" and not case["muon"]):
        # fp32 arithmetic; a bf16 copy may round to its other neighbour now and then
        return {"rel": 3e-5, "max": 1e-2}
    # weights after a Muon update: the orthogonalised step is within 2e-3 and small beside the weight
    return {"rel": 1e-3, "max": 1.6e-2}
