"""The work this framework is measured on: its public operators over the sizes they are used at.

Every case goes through an entry point of ``pto_fuser_amd`` the way a program calls it: operands
resident on the GPU, outputs allocated by the call, workspaces kept by the package.  Distributions
are the benchmark's: q, k L2-normalised Gaussian rows, v ~ N(0,1), beta = sigmoid(N(0,1)),
log-decay g = -softplus(N(0,1)) times 0.1 (per token) or 0.05 (per channel), h0 ~ N(0, 0.02).

``exact`` evaluates the same mathematics in float64 with plain torch: the delta rule as its
token-by-token recurrence (no chunks), the stage operators from their definitions.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "pto-fuser_amd"))

import pto_fuser_amd as pf                                              # noqa: E402
from pto_fuser_amd.forwards import (build_gdn_program, make_gdn_inputs,  # noqa: E402
                                    prepare_gdn_bindings)

D = 128
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
ESIZE = {"bf16": 2, "fp32": 4}


# ------------------------------------------------------------------------------------------
#  The cases
# ------------------------------------------------------------------------------------------
def _gdn(dtype, B, H, T, gated=True, h0=False, C=64):
    return {"op": "gdn", "dtype": dtype, "B": B, "H": H, "T": T, "C": C, "gated": gated, "h0": h0}


def _kda(dtype, B, H, T, h0=False, C=64):
    return {"op": "kda", "dtype": dtype, "B": B, "H": H, "T": T, "C": C, "h0": h0}


def listed():
    return [
        # one more 64-token chunk of a running sequence: 16 heads, the state carried in and out
        dict(_gdn("bf16", 1, 16, 64, h0=True), name="gdn_stream_step"),
        # a few sequences of uneven length and head count (15 chains, 23 chunks)
        dict(_gdn("bf16", 3, 5, 1472), name="gdn_ragged"),
        # a training or prefill layer: the benchmark's headline
        dict(_gdn("bf16", 4, 16, 4096), name="gdn_layer"),
        # long-context prefill of one sequence, continued from a state
        dict(_gdn("bf16", 1, 32, 32768, h0=True), name="gdn_long_context"),
        # full-precision DeltaNet (no gate): a short check-sized forward
        dict(_gdn("fp32", 1, 4, 512, gated=False), name="deltanet_fp32"),
        # a per-channel-gate layer: the KDA benchmark
        dict(_kda("bf16", 2, 32, 8192), name="kda_layer"),
        # the same in full precision, at a validation size
        dict(_kda("fp32", 2, 16, 2048), name="kda_fp32"),
        # gated kkt + (I + A)^-1 alone over 4096 chunks
        {"name": "kkt_inverse", "op": "kkt", "dtype": "fp32", "M": 4096},
        # the compile stack's fused nodes, on its C = D = 128 tiles: the gated score of a token
        # layout [T, H, D], the resident-state scan, and the chunk output
        {"name": "gated_score", "op": "score", "dtype": "bf16", "nc": 32, "H": 16, "C": 128,
         "causal": False},
        {"name": "chunk_scan", "op": "scan", "dtype": "bf16", "B": 8, "H": 32, "nc": 16, "C": 128,
         "perdim": False},
        {"name": "chunk_output", "op": "flash", "dtype": "bf16", "M": 1024, "C": 128},
        # a GDN program lowered by the compile stack and replayed as a captured graph
        {"name": "compiled_gdn", "op": "compiled", "dtype": "bf16", "B": 1, "H": 16, "nc": 8,
         "C": 128},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.999)))))))


def _chains(rng, rows, max_T, C):
    """(B, H, T): T a multiple of C, B*H*T <= rows, both spread over their logarithm."""
    T = C * _log_int(rng, 1, max_T // C)
    BH = _log_int(rng, 1, max(1, min(512, rows // T)))
    B = rng.choice([b for b in range(1, 9) if BH // b >= 1])
    return B, max(1, BH // B), T


def draw(rng):
    op = rng.choice(["gdn", "gdn", "gdn", "gdn_fp32", "kda", "kda", "kda_fp32", "kkt", "score",
                     "scan", "flash"])
    C = rng.choice([64, 64, 128])
    if op == "gdn":
        B, H, T = _chains(rng, 960000, 32768, C)
        return _gdn("bf16", B, H, T, gated=rng.random() < 0.8, h0=rng.random() < 0.5, C=C)
    if op == "gdn_fp32":
        B, H, T = _chains(rng, 1 << 17, 4096, C)
        return _gdn("fp32", B, H, T, gated=rng.random() < 0.5, h0=rng.random() < 0.5, C=C)
    if op == "kda":
        B, H, T = _chains(rng, 1 << 19, 16384, C)
        return _kda("bf16", B, H, T, h0=rng.random() < 0.5, C=C)
    if op == "kda_fp32":
        B, H, T = _chains(rng, 1 << 16, 4096, C)
        return _kda("fp32", B, H, T, h0=rng.random() < 0.5, C=C)
    dtype = rng.choice(["bf16", "bf16", "fp32"])
    if op == "kkt":
        return {"op": "kkt", "dtype": dtype, "M": _log_int(rng, 1, 8192)}
    C = rng.choice([32, 64, 128, 128])
    if op == "score":
        H = rng.choice([1, 3, 4, 8, 16, 32])
        return {"op": "score", "dtype": dtype, "nc": _log_int(rng, 1, 2048 // H), "H": H, "C": C,
                "causal": rng.random() < 0.5}
    if op == "scan":
        BH = _log_int(rng, 1, 256)
        B = rng.choice([b for b in (1, 2, 3, 4, 8) if BH // b >= 1])
        H = max(1, BH // B)
        return {"op": "scan", "dtype": dtype, "B": B, "H": H,
                "nc": _log_int(rng, 1, min(64, max(1, 2048 // (B * H)))), "C": C,
                "perdim": rng.random() < 0.4}
    return {"op": "flash", "dtype": dtype, "M": _log_int(rng, 1, 2048), "C": C}


# ------------------------------------------------------------------------------------------
#  What a program has in hand before the call
# ------------------------------------------------------------------------------------------
def _gen(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)
    return gen


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda")


def _unit_rows(gen, *shape):
    return torch.nn.functional.normalize(_randn(gen, *shape), dim=-1)


def _decay(gen, scale, *shape):
    return -torch.nn.functional.softplus(_randn(gen, *shape)) * scale


def _within_chunk(g, C):
    """Cumulative sum along dim 0 inside chunks of C rows."""
    return g.reshape(-1, C, *g.shape[1:]).cumsum(1).reshape(g.shape).contiguous()


def _inputs(case, seed):
    """The operands, from the seed alone."""
    gen, op = _gen(seed), case["op"]
    dt = DTYPES[case["dtype"]]
    if op in ("gdn", "kda"):
        B, H, T = case["B"], case["H"], case["T"]
        x = {"q": _unit_rows(gen, B, H, T, D).to(dt), "k": _unit_rows(gen, B, H, T, D).to(dt),
             "v": _randn(gen, B, H, T, D).to(dt), "beta": torch.sigmoid(_randn(gen, B, H, T)),
             "g": None}
        if op == "kda":
            x["g"] = _decay(gen, 0.05, B, H, T, D)
        elif case["gated"]:
            x["g"] = _decay(gen, 0.1, B, H, T)
        x["h0"] = _randn(gen, B, H, D, D) * 0.02 if case["h0"] else None
        return x
    if op == "kkt":
        n = case["M"] * 64
        return {"k": _unit_rows(gen, n, D).to(dt), "g": _decay(gen, 0.1, n),
                "beta": torch.sigmoid(_randn(gen, n))}
    if op == "score":
        n, H = case["nc"] * case["C"], case["H"]
        return {"k": _unit_rows(gen, n, H, D).to(dt),
                "q": _unit_rows(gen, n, H, D).to(dt) if case["causal"] else None,
                "g": _within_chunk(_decay(gen, 0.1, n, H), case["C"]),
                "beta": torch.sigmoid(_randn(gen, n, H))}
    if op == "scan":
        # contractive magnitudes, as the stage's own inputs (forwards.make_scan_inputs) draw them
        B, H, nc, C = case["B"], case["H"], case["nc"], case["C"]
        dshape = (B, H, nc, D) if case["perdim"] else (B, H, nc)
        return {"w": (_randn(gen, B, nc, C, H, D) * 0.02).to(dt),
                "u": (_randn(gen, B, nc, C, H, D) * 0.05).to(dt),
                "k": (_randn(gen, B, nc, C, H, D) * 0.02).to(dt),
                "decay": 0.7 + 0.2 * torch.rand(*dshape, generator=gen, device="cuda")}
    if op == "flash":
        M, C = case["M"], case["C"]
        return {"q": _unit_rows(gen, M, C, D).to(dt), "k": _unit_rows(gen, M, C, D).to(dt),
                "v": _randn(gen, M, C, D).to(dt), "g": _decay(gen, 0.1, M, C).cumsum(1)}
    raise ValueError(f"unknown op {op!r}")


def _compiled_inputs(case, seed):
    """The program's operands as its own input maker draws them (on the host, then moved)."""
    return make_gdn_inputs(case["B"], case["H"], case["nc"], case["C"], D, device="cuda",
                           dtype=DTYPES[case["dtype"]], seed=int(seed) % (1 << 31))


def prepare(case, seed):
    if case["op"] != "compiled":
        return {"case": case, "x": _inputs(case, seed)}
    B, H, nc, C = case["B"], case["H"], case["nc"], case["C"]
    work = DTYPES[case["dtype"]]
    bindings = prepare_gdn_bindings(**_compiled_inputs(case, seed), work=work)
    program = build_gdn_program(B, H, nc, C, D, D ** -0.5, work=work)
    lowered = pf.compile_program(program, pf.Features(B=B, H=H, nc=nc, C=C, D=D), verify=False)
    graph = pf.GraphReplayExecutor().capture(lowered.program, bindings)
    return {"case": case, "x": bindings, "graph": graph}


# ------------------------------------------------------------------------------------------
#  One pass
# ------------------------------------------------------------------------------------------
def run(state):
    case, x = state["case"], state["x"]
    op = case["op"]
    if op == "gdn":
        return pf.gdn_chunk_forward(x["q"], x["k"], x["v"], x["beta"], x["g"], h0=x["h0"],
                                    chunk_size=case["C"])
    if op == "kda":
        return pf.kda_chunk_forward(x["q"], x["k"], x["v"], x["beta"], x["g"], h0=x["h0"],
                                    chunk_size=case["C"])
    if op == "kkt":
        return pf.kkt_inverse(x["k"], x["g"], x["beta"])
    if op == "score":
        a = x["q"] if case["causal"] else x["k"]
        return pf.gated_qk(a, x["k"], x["g"], x["beta"], chunk_size=case["C"], heads=case["H"],
                           causal=case["causal"], out_dtype=DTYPES[case["dtype"]])
    if op == "scan":
        return pf.chunk_scan(x["w"], x["u"], x["k"], x["decay"], out_dtype=DTYPES[case["dtype"]])
    if op == "flash":
        return pf.qkv_flash(x["q"], x["k"], x["v"], x["g"], chunk_size=case["C"])
    return state["graph"].replay(x)["o"]


# ------------------------------------------------------------------------------------------
#  What a pass cannot do without
# ------------------------------------------------------------------------------------------
def _forward_work(n, chains, esize, gate_floats, h0):
    """q, k, v, beta and the gate in, o and the final state out (fp32); the chunked products of
    64-token chunks: kkt, (I + A)^-1, T r, k S, q S, q k^T, P v and the update."""
    state = chains * D * D * 4
    nbytes = n * (3 * D * esize + 4 + 4 * gate_floats + 4 * D) + state * (2 if h0 else 1)
    c = 64
    flops = n // c * (2 * (2 * c * c * D) + c ** 3 // 3 + 2 * (2 * c * c * D) + 3 * (2 * c * D * D))
    return {"bytes": nbytes, "flops": flops}


def work(case):
    op = case["op"]
    e = ESIZE[case["dtype"]]
    if op in ("gdn", "kda"):
        chains = case["B"] * case["H"]
        gate = D if op == "kda" else (1 if case["gated"] else 0)
        return _forward_work(chains * case["T"], chains, e, gate, case["h0"])
    if op == "kkt":
        n = case["M"] * 64
        return {"bytes": n * (D * e + 8) + n * 64 * 4,
                "flops": case["M"] * (2 * 64 * 64 * D + 64 ** 3 // 3)}
    if op == "score":
        n, C = case["nc"] * case["C"] * case["H"], case["C"]
        return {"bytes": n * (D * e * (2 if case["causal"] else 1) + 8) + n * C * e,
                "flops": n * C * D}
    if op == "scan":
        m, C = case["B"] * case["H"] * case["nc"], case["C"]
        dec = m * 4 * (D if case["perdim"] else 1)
        return {"bytes": 3 * m * C * D * e + dec + m * D * D * e + case["B"] * case["H"] * D * D * 4,
                "flops": 2 * m * (2 * C * D * D)}
    if op == "flash":
        m, C = case["M"], case["C"]
        return {"bytes": m * C * (3 * D * e + 4 + 4 * D), "flops": m * 2 * C * C * D}
    n = case["B"] * case["H"] * case["nc"] * case["C"]
    return _forward_work(n, case["B"] * case["H"], e, 1, False)


# ------------------------------------------------------------------------------------------
#  The same in 64 bits
# ------------------------------------------------------------------------------------------
def _recurrence(q, k, v, beta, g, h0):
    """S <- e^g S;  S <- S + k (beta (v - k^T S))^T;  o = scale q S, token by token.  q, k, v
    [N, T, D], beta [N, T], g [N, T] or [N, T, D] or None, all float64.  Returns o, S."""
    N, T, _ = q.shape
    S = torch.zeros(N, D, D, dtype=torch.float64, device=q.device) if h0 is None else h0.clone()
    o = torch.empty(N, T, D, dtype=torch.float64, device=q.device)
    gate = None
    if g is not None:
        gate = torch.exp(g if g.dim() == 3 else g.unsqueeze(-1)).unsqueeze(-1)   # [N, T, D | 1, 1]
    for t in range(T):
        kt = k[:, t].unsqueeze(-1)
        if gate is not None:
            S *= gate[:, t]
        r = beta[:, t, None] * (v[:, t] - (kt * S).sum(1))
        S += kt * r.unsqueeze(1)
        o[:, t] = (q[:, t].unsqueeze(-1) * S).sum(1)
    return o * D ** -0.5, S


def _f64(x):
    return {n: (None if t is None else t.double()) for n, t in x.items()}


def _exact_forward(case, x):
    N, T = case["B"] * case["H"], case["T"]
    flat = {n: (None if t is None else t.reshape(N, *t.shape[2:])) for n, t in x.items()}
    o, S = _recurrence(flat["q"], flat["k"], flat["v"], flat["beta"], flat["g"], flat["h0"])
    lead = (case["B"], case["H"])
    return o.reshape(*lead, T, D), S.reshape(*lead, D, D)


def _unit_lower_inverse(A):
    """(I + A)^-1, A strictly lower, row by row."""
    C = A.shape[-1]
    T = torch.eye(C, dtype=A.dtype, device=A.device).repeat(A.shape[0], 1, 1)
    for i in range(1, C):
        T[:, i, :] -= (A[:, i, :i].unsqueeze(1) @ T[:, :i, :]).squeeze(1)
    return T


def _gated(score, G, log_beta):
    return score * torch.exp(torch.clamp(G.unsqueeze(-1) + log_beta - G.unsqueeze(-2), max=0.0))


def exact(case, seed):
    op = case["op"]
    if op == "compiled":
        i = _f64(_compiled_inputs(case, seed))
        N, T = case["B"] * case["H"], case["nc"] * case["C"]
        o, _ = _recurrence(i["q"].reshape(N, T, D), i["k"].reshape(N, T, D),
                           i["v"].reshape(N, T, D), i["beta"].reshape(N, T),
                           i["g_in"].reshape(N, T), None)
        return o.reshape(case["B"], case["H"], case["nc"], case["C"], D)
    x = _f64(_inputs(case, seed))
    if op in ("gdn", "kda"):
        return _exact_forward(case, x)
    if op == "kkt":
        M = case["M"]
        k, beta = x["k"].reshape(M, 64, D), x["beta"].reshape(M, 64)
        G = x["g"].reshape(M, 64).cumsum(1)
        A = (beta.unsqueeze(-1) * torch.exp(G.unsqueeze(-1) - G.unsqueeze(-2)).tril(-1)
             * (k @ k.transpose(1, 2).contiguous()))
        return _unit_lower_inverse(A)
    if op == "score":
        nc, H, C = case["nc"], case["H"], case["C"]

        def heads_out(t):
            return t.reshape(nc, C, H, -1).permute(0, 2, 1, 3).reshape(nc * H, C, -1)

        k = heads_out(x["k"])
        a = heads_out(x["q"]) if case["causal"] else k
        G, lb = heads_out(x["g"]).squeeze(-1), heads_out(x["beta"]).log()
        L = _gated(a @ k.transpose(1, 2).contiguous(), G, lb).tril(0 if case["causal"] else -1)
        return L.reshape(nc, H, C, C).permute(0, 2, 1, 3).reshape(nc * C, H, C).contiguous()
    if op == "scan":
        B, H, nc = case["B"], case["H"], case["nc"]
        S = torch.zeros(B, H, D, D, dtype=torch.float64, device="cuda")
        snaps = []
        for c in range(nc):
            snaps.append(S)
            w, u, k = (x[n][:, c].transpose(1, 2).contiguous() for n in ("w", "u", "k"))
            dec = x["decay"][:, :, c]
            dec = dec.unsqueeze(-1) if case["perdim"] else dec.reshape(B, H, 1, 1)
            S = dec * S + k.transpose(2, 3).contiguous() @ (u - w @ S)
        return torch.stack(snaps, 1), S
    P = _gated(x["q"] @ x["k"].transpose(1, 2).contiguous(), x["g"], 0.0).tril()
    return P @ x["v"]


# ------------------------------------------------------------------------------------------
#  How far two correct implementations may lie apart
# ------------------------------------------------------------------------------------------
def tolerance(case):
    """About four times the distance to float64 measured: 2.9e-3 (GDN) and 3.8e-3 (KDA) for the bf16
    forwards, whose state, r and v_new are rounded to 8 bits before each product, 2.3e-3 for the
    bf16 stages (one or two such roundings), up to 3e-7 for fp32 at these lengths, where a sum in
    another order over 4096 tokens may lie further off."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    return {"rel": 1e-2 if case["op"] in ("score", "scan", "flash") else 1.6e-2}
