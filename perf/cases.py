"""What is timed to see whether the library got faster: the calls a structure-prediction program makes on one GPU.

A case is one call of a public entry point on device tensors, with a plan, weights and workspace that such a program
keeps from call to call.  Lengths are what proteins have: any number of residues, seldom a multiple of a tile.

  op                       entry point
  gating                   kutacc_af2_gating_attention (tensor handles): triangle, MSA-row and extra-MSA-row attention
  triangle_attention       kutacc_hip_triangle_attention: the whole block, starting or ending node, in place
  triangle_multiplication  kutacc_hip_triangle_multiplication: the whole block, outgoing or incoming edges, in place
  msa_attention            kutacc_hip_msa_attention: the whole block, row-wise with pair bias or column-wise, in place
  transition               kutacc_hip_transition_block: LayerNorm, two products and residual, in place
  global_attention         kutacc_af2_global_attention (tensor handles): the extra-MSA column attention
  linear                   kutacc_af2_linear (tensor handles): the pair-bias projection and other Linears of a caller
"""
import math

import torch

from kutacc_amd import capi

HEAD = 32      # head size of the blocks
C_PAIR = 128   # channels of the pair activation
C_MSA = 256    # channels of the MSA activation
EPS = 1e-5


def listed():
    return [
        # The smallest operator call, in fp32 storage: sixteen short sequences, where the launches and the host count.
        dict(name="msa_row_fp32_16x64", op="gating", dtype="fp32", batch=16, seq=64, heads=8, head_size=32, padded=False),
        # A short peptide: one block of the pair stack at 77 residues, latency and an odd length.
        dict(name="tri_att_start_77", op="triangle_attention", n=77, ending=False, padded=False),
        # The operator by itself at the usual crop of 384 residues.
        dict(name="tri_att_op_384", op="gating", dtype="bf16", batch=384, seq=384, heads=4, head_size=32, padded=False),
        # A long chain padded by a few residues, past the longest row of the fused kernels: the largest case.
        dict(name="tri_att_end_2048", op="triangle_attention", n=2048, ending=True, padded=True),
        # The other half of the pair stack at the usual crop ...
        dict(name="tri_mul_out_384", op="triangle_multiplication", n=384, incoming=False, padded=False),
        # ... and on a whole chain, whose length is odd.
        dict(name="tri_mul_in_691", op="triangle_multiplication", n=691, incoming=True, padded=True),
        # MSA stack: 508 clustered sequences of a protein of 259 residues, row-wise ...
        dict(name="msa_row_508x259", op="msa_attention", n_seq=508, n_res=259, column=False, padded=False),
        # ... column-wise over 1024 sequences, a tenth of them padding ...
        dict(name="msa_col_1024x384", op="msa_attention", n_seq=1024, n_res=384, column=True, padded=True),
        # ... and its transition, 256 -> 1024 -> 256 channels.
        dict(name="msa_transition_508x384", op="transition", rows=508 * 384, c_o=256, c_i=1024),
        # Extra-MSA stack (64 channels, heads of 8): row attention of 1024 sequences of an odd length ...
        dict(name="extra_row_1024x301", op="gating", dtype="bf16", batch=1024, seq=301, heads=8, head_size=8, padded=False),
        # ... and the global column attention over all 5120 sequences.
        dict(name="extra_global_5120x384", op="global_attention", n_seq=5120, n_res=384, heads=8, padded=True),
        # The pair-bias Linear of a caller that follows the operator-by-operator API: eight heads from the pair channels.
        dict(name="pair_bias_linear_384", op="linear", rows=384 * 384, n=8, k=C_PAIR, bias=False),
    ]


def _size(rng, low, high):
    """A size between low and high, even over the logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    op = rng.choice(["gating", "triangle_attention", "triangle_multiplication", "msa_attention", "transition", "global_attention",
                     "linear"])
    padded = rng.random() < 0.5
    if op == "gating":
        kind = rng.choice(["triangle", "msa", "extra", "fp32"])
        if kind == "triangle":
            n = _size(rng, 48, 1280)
            return dict(op=op, dtype="bf16", batch=n, seq=n, heads=4, head_size=32, padded=padded)
        if kind == "msa":
            return dict(op=op, dtype="bf16", batch=_size(rng, 16, 512), seq=_size(rng, 48, 1024), heads=8, head_size=32, padded=padded)
        if kind == "extra":
            return dict(op=op, dtype="bf16", batch=_size(rng, 64, 5120), seq=_size(rng, 48, 512), heads=8, head_size=8, padded=padded)
        return dict(op=op, dtype="fp32", batch=_size(rng, 4, 64), seq=_size(rng, 16, 200), heads=rng.choice([4, 8]), head_size=32,
                    padded=padded)
    if op == "triangle_attention":
        return dict(op=op, n=_size(rng, 48, 1536), ending=rng.random() < 0.5, padded=padded)
    if op == "triangle_multiplication":
        return dict(op=op, n=_size(rng, 48, 1280), incoming=rng.random() < 0.5, padded=padded)
    if op == "msa_attention":
        return dict(op=op, n_seq=_size(rng, 32, 1024), n_res=_size(rng, 48, 768), column=rng.random() < 0.5, padded=padded)
    if op == "transition":
        c = rng.choice([64, 128, 256])  # extra-MSA or template, pair, MSA
        return dict(op=op, rows=_size(rng, 2048, 512 * 1024), c_o=c, c_i=rng.choice([2, 4]) * c)
    if op == "global_attention":
        return dict(op=op, n_seq=_size(rng, 128, 5120), n_res=_size(rng, 48, 512), heads=8, padded=padded)
    return dict(op=op, rows=_size(rng, 2048, 512 * 1024), n=rng.choice([4, 8, 32, 64, 128, 256]), k=rng.choice([64, 128, 256]),
                bias=rng.random() < 0.5)


# ---- inputs ----

class _Draw:
    """Seeded values on the GPU with the distributions of the network: activations N(0, 1), weights N(0, 1 / fan_in), LayerNorm
    parameters around 1 and 0, gating bias around 1, other biases around 0."""

    def __init__(self, seed, dtype=torch.bfloat16):
        self.g = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = dtype

    def normal(self, *shape, scale=1.0):
        return (torch.randn(*shape, device="cuda", generator=self.g) * scale).to(self.dtype)

    def weight(self, fan_out, fan_in):
        return self.normal(fan_out, fan_in, scale=fan_in ** -0.5)

    def around(self, centre, size):
        return centre + 0.1 * torch.randn(size, device="cuda", generator=self.g)

    def normalised(self, *shape):
        return torch.nn.functional.layer_norm(torch.randn(*shape, device="cuda", generator=self.g), shape[-1:]).to(self.dtype)

    def kept(self, size, padded):
        """1 for positions that are there, 0 for padding: up to a tenth of them at the end."""
        m = torch.ones(size, device="cuda")
        if padded and size > 1:
            cut = int(torch.randint(1, max(2, size // 10 + 1), (1,), device="cuda", generator=self.g))
            m[size - cut:] = 0
        return m


def _attention_weights(d, c):
    w = {k: d.weight(c, c) for k in ("wq", "wk", "wv", "wg", "wo")}
    w["bg"], w["bo"] = d.around(1.0, c), d.around(0.0, c)
    return w


def prepare(case, seed):
    capi.set_blocking(False)  # calls return once they are enqueued, on torch's default stream
    op = case["op"]
    d = _Draw(seed, torch.float32 if case.get("dtype") == "fp32" else torch.bfloat16)
    dt = d.dtype
    if op == "gating":
        B, S, H = case["batch"], case["seq"], case["heads"]
        C = H * case["head_size"]
        w = _attention_weights(d, C)
        bias = ((d.kept(S, case["padded"]) - 1.0) * 1e9).to(dt).expand(B, S).contiguous()
        nb = d.normal(H, S, S)
        out = torch.empty(B, S, C, device="cuda", dtype=dt)
        scratch = {k: torch.empty(B, S, H, case["head_size"], device="cuda", dtype=dt) for k in ("q", "k", "gate", "avg")}
        scratch["v"] = torch.empty(H, case["head_size"], B, S, device="cuda", dtype=dt)
        call = capi.GatedAttention(d.normalised(B, S, C), w["wq"], w["wk"], w["wv"], w["wg"], w["bg"], w["wo"], w["bo"], bias, nb, H,
                                   out, scratch)
        return dict(run=call.run, out=out)
    if op == "triangle_attention":
        n, H = case["n"], C_PAIR // HEAD
        act = d.normal(n, n, C_PAIR)
        keep = d.kept(n, case["padded"])
        w = _attention_weights(d, C_PAIR)
        block = capi.TriangleAttentionBlock(act, torch.outer(keep, keep).to(dt), d.around(1.0, C_PAIR), d.around(0.0, C_PAIR),
                                            d.weight(H, C_PAIR), w["wq"], w["wk"], w["wv"], w["wg"], w["bg"], w["wo"], w["bo"], H,
                                            case["ending"], EPS)
        return dict(run=_checked(block.run), out=act)
    if op == "triangle_multiplication":
        n, c = case["n"], C_PAIR
        act = d.normal(n, n, c)
        keep = d.kept(n, case["padded"])
        w = {}
        for side in ("left", "right"):
            w[f"{side}_proj_w"], w[f"{side}_gate_w"] = d.weight(c, c), d.weight(c, c)
            w[f"{side}_proj_b"], w[f"{side}_gate_b"] = d.around(0.0, c), d.around(1.0, c)
        for norm in ("ln_in", "ln_center"):
            w[f"{norm}_gamma"], w[f"{norm}_beta"] = d.around(1.0, c), d.around(0.0, c)
        w["output_w"], w["output_b"], w["gating_w"], w["gating_b"] = d.weight(c, c), d.around(0.0, c), d.weight(c, c), d.around(1.0, c)
        block = capi.TriangleMultiplicationBlock(act, torch.outer(keep, keep).to(dt), w, case["incoming"], EPS)
        return dict(run=_checked(block.run), out=act)
    if op == "msa_attention":
        n_seq, n_res, H = case["n_seq"], case["n_res"], C_MSA // HEAD
        act = d.normal(n_seq, n_res, C_MSA)
        # padding: of the sequences where they are attended over, of the residues where those are
        mask = (d.kept(n_seq, case["padded"])[:, None] if case["column"] else d.kept(n_res, case["padded"])[None, :])
        w = _attention_weights(d, C_MSA)
        w["ln_gamma"], w["ln_beta"] = d.around(1.0, C_MSA), d.around(0.0, C_MSA)
        pair = None
        if not case["column"]:
            pair = dict(pair_act=d.normal(n_res, n_res, C_PAIR), pair_ln_gamma=d.around(1.0, C_PAIR),
                        pair_ln_beta=d.around(0.0, C_PAIR), bias_w=d.weight(H, C_PAIR))
        block = capi.MsaAttentionBlock(act, mask.expand(n_seq, n_res).to(dt).contiguous(), w, H, pair, EPS)
        return dict(run=_checked(block.run), out=act)
    if op == "transition":
        rows, c_o, c_i = case["rows"], case["c_o"], case["c_i"]
        act = d.normal(rows, c_o)
        keep = [d.around(1.0, c_o), d.around(0.0, c_o), d.weight(c_i, c_o), d.around(0.0, c_i), d.weight(c_o, c_i), d.around(0.0, c_o)]
        gamma, beta, w1, b1, w2, b2 = keep
        L = capi.lib()
        size = max(0, L.kutacc_hip_transition_block_workspace(rows, c_o, c_i))
        workspace = torch.empty(max(size, 1), dtype=torch.uint8, device="cuda")
        keep.append(workspace)
        args = (act.data_ptr(), gamma.data_ptr(), beta.data_ptr(), EPS, w1.data_ptr(), b1.data_ptr(), w2.data_ptr(), b2.data_ptr(),
                workspace.data_ptr(), size, rows, c_o, c_i, capi.K_BF16, None)
        return dict(run=_checked(lambda: L.kutacc_hip_transition_block(*args)), out=act, keep=keep)
    if op == "global_attention":
        B, S, H, C = case["n_res"], case["n_seq"], case["heads"], 64
        x = d.normalised(B, S, C)
        mask = d.kept(S, case["padded"]).to(dt).expand(B, S)[..., None].contiguous()
        hs = C // H
        out = torch.empty(B, S, C, device="cuda", dtype=dt)
        avg = torch.empty(B, C, device="cuda", dtype=dt)
        small = torch.empty(1, C, device="cuda", dtype=dt)  # scratch of the reference that the device library leaves alone
        scratch = dict(q=small, k=small, v=small, gate=small, avg=avg)
        call = capi.GlobalAttention(x, mask, d.weight(C, C), d.weight(hs, C), d.weight(hs, C), d.weight(C, C), d.around(1.0, C),
                                    d.weight(C, C), d.around(0.0, C), H, out, scratch)
        return dict(run=call.run, out=(out, avg))
    rows, n, k = case["rows"], case["n"], case["k"]
    act, weight = d.normalised(rows, k), d.weight(n, k)
    bias = d.around(0.0, n) if case["bias"] else None
    out = torch.empty(rows, n, device="cuda", dtype=dt)
    handles = [capi.tensor(t) for t in (act, weight, out)]
    a, w, r = (h.handle for h in handles)
    L = capi.lib()
    b = bias.data_ptr() if bias is not None else None
    return dict(run=lambda: L.kutacc_af2_linear(a, w, b, r, 0), out=out, keep=(handles, bias))


def _checked(call):
    def run():
        rc = call()
        if rc != 0:
            raise RuntimeError(f"the library returned {rc}")
    return run


def run(state):
    state["run"]()
    return state["out"]


# ---- what a pass cannot do without ----

def work(case):
    op = case["op"]
    if op == "gating":
        B, S, H, e = case["batch"], case["seq"], case["heads"], 4 if case["dtype"] == "fp32" else 2
        C = H * case["head_size"]
        return dict(bytes=(2 * B * S * C + H * S * S + B * S + 5 * C * C) * e + 8 * C,
                    flops=10 * B * S * C * C + 4 * B * S * S * C)
    if op == "triangle_attention":
        n, C, H = case["n"], C_PAIR, C_PAIR // HEAD
        return dict(bytes=2 * (2 * n * n * C + n * n + 5 * C * C + H * C) + 16 * C,
                    flops=10 * n * n * C * C + 4 * n ** 3 * C + 2 * n * n * C * H)
    if op == "triangle_multiplication":
        n, C = case["n"], C_PAIR
        return dict(bytes=2 * (2 * n * n * C + n * n + 6 * C * C) + 40 * C, flops=12 * n * n * C * C + 2 * n ** 3 * C)
    if op == "msa_attention":
        s, r, C, H = case["n_seq"], case["n_res"], C_MSA, C_MSA // HEAD
        row = not case["column"]
        keys = r if row else s
        return dict(bytes=2 * (2 * s * r * C + s * r + 5 * C * C + (r * r * C_PAIR + H * C_PAIR) * row) + 16 * C,
                    flops=10 * s * r * C * C + 4 * s * r * keys * C + 2 * r * r * C_PAIR * H * row)
    if op == "transition":
        rows, c_o, c_i = case["rows"], case["c_o"], case["c_i"]
        return dict(bytes=2 * (2 * rows * c_o + 2 * c_o * c_i) + 4 * (c_i + 3 * c_o), flops=4 * rows * c_o * c_i)
    if op == "global_attention":
        m, hs = case["n_seq"] * case["n_res"], 64 // case["heads"]
        return dict(bytes=2 * (2 * m * 64 + m + 64 * case["n_res"] + 3 * 64 * 64 + 2 * hs * 64) + 512,
                    flops=m * (4 * 64 * hs + 4 * 64 * 64 + 4 * 64))
    rows, n, k = case["rows"], case["n"], case["k"]
    return dict(bytes=2 * (rows * k + n * k + rows * n) + 4 * n * case["bias"], flops=2 * rows * n * k)


def tolerance(case):
    """fp32: sums of a few hundred terms.  bf16: results, and the operands of every product, are rounded to eight bits."""
    if case.get("dtype") == "fp32":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 1e-2, "max": 6e-2}
