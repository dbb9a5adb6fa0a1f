"""The work a binder-design program has this library do, as timed cases.

A case is one pass of a layer, a block stack or a whole design step through
bindcraft2_amd.ops, forward and (unless it says otherwise) backward, on
random-init AF2 multimer weights and N(0, 1) activations resident in HBM:

  triattn     one triangle attention with its dropout table and residual
  trimul      one triangle multiplication, likewise
  transition  the pair transition over rows x n tokens
  evoformer   `depth` Evoformer blocks over the MSA and pair carries
  template    the template pair stack (2 blocks, c_t = 64)
  design      the one-call design step from the designed logits

Lengths are total complex lengths (target + binder), padded to 32 as the
layers require; the design step takes its true length at run time.  Weights
are written once per machine into the temporary directory, as a program
keeps one weights directory, and are the same for every seed; inputs are
drawn on the GPU from the seed.
"""
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from bindcraft2_amd import ops, params as bparams, weights as bweights

TRIATTN = {False: "triangle_attention_starting_node", True: "triangle_attention_ending_node"}
TRIMUL = {True: "triangle_multiplication_outgoing", False: "triangle_multiplication_incoming"}
DEPTHS = (2, 4, 48, 8)  # template, extra, main, fold iterations: AF2 multimer's
STACK_BLOCKS = 4        # blocks in the evoformer cases' weights directory


# ------------------------------------------------------------------- the cases
def listed():
    return [
        # a short peptide binder on a small domain: launches and latency count
        {"name": "triattn_64", "kind": "triattn", "n": 64, "flip": False, "drop": True,
         "masked": 0.1},
        # the README's headline length, ending node
        {"name": "triattn_224", "kind": "triattn", "n": 224, "flip": True, "drop": True,
         "masked": 0.1},
        # the large complex
        {"name": "triattn_512", "kind": "triattn", "n": 512, "flip": False, "drop": True,
         "masked": 0.1},
        # a mini-binder alone on a small target, incoming
        {"name": "trimul_96", "kind": "trimul", "n": 96, "flip": False, "drop": True,
         "masked": 0.0},
        # the headline length, outgoing
        {"name": "trimul_224", "kind": "trimul", "n": 224, "flip": True, "drop": True,
         "masked": 0.1},
        # between the headline and the large complex, in a prediction without dropout
        {"name": "trimul_416", "kind": "trimul", "n": 416, "flip": False, "drop": False,
         "masked": 0.1},
        # the pair transition at a row count that fills no tile evenly
        {"name": "transition_203", "kind": "transition", "rows": 203, "n": 203},
        # a slice of the main stack as a design step runs it: one MSA row, dropout
        {"name": "evoformer_128", "kind": "evoformer", "n": 128, "s": 1, "depth": 4,
         "drop": True, "masked": 0.1, "grad": True},
        # with the template's MSA row beside the query's, no dropout
        {"name": "evoformer_320", "kind": "evoformer", "n": 320, "s": 2, "depth": 2,
         "drop": False, "masked": 0.1, "grad": True},
        # a recycle pass or a prediction: forward only, nothing saved
        {"name": "evoformer_448_fwd", "kind": "evoformer", "n": 448, "s": 1, "depth": 2,
         "drop": False, "masked": 0.05, "grad": False},
        # the template pair stack
        {"name": "template_192", "kind": "template", "n": 192, "drop": False, "masked": 0.1},
        # a whole design step, 151 residues in a bucket of 160
        {"name": "design_160", "kind": "design", "n": 160, "length": 151, "drop": True},
    ]


def _spread(rng, lo, hi, step=32):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + step)))
    return min(hi, max(lo, int(v) // step * step))


def draw(rng):
    kind = rng.choice(("triattn", "triattn", "trimul", "trimul", "transition", "evoformer",
                       "evoformer", "template", "design"))
    masked = round(rng.choice((0.0, rng.uniform(0.02, 0.3))), 3)
    drop = rng.random() < 0.5
    if kind in ("triattn", "trimul"):
        return {"kind": kind, "n": _spread(rng, 32, 512), "flip": rng.random() < 0.5,
                "drop": drop, "masked": masked}
    if kind == "transition":
        return {"kind": kind, "rows": _spread(rng, 30, 500, 1), "n": _spread(rng, 30, 500, 1)}
    if kind == "evoformer":
        return {"kind": kind, "n": _spread(rng, 64, 448), "s": rng.choice((1, 1, 2)),
                "depth": rng.randint(1, 3), "drop": drop, "masked": masked,
                "grad": rng.random() < 0.7}
    if kind == "template":
        return {"kind": kind, "n": _spread(rng, 64, 416), "drop": drop, "masked": masked}
    n = _spread(rng, 96, 160)
    return {"kind": kind, "n": n, "length": n - rng.randint(0, 31), "drop": drop}


# --------------------------------------------------------------------- weights
_made = {}


def _weights(tag, make):
    """The weights directory `tag`, written by make(directory) on first use."""
    if tag not in _made:
        uid = os.getuid() if hasattr(os, "getuid") else 0
        path = os.path.join(tempfile.gettempdir(), f"bc2n_cases_{uid}_{tag}")
        if not os.path.isdir(path):
            tmp = tempfile.mkdtemp(prefix="bc2n_cases_")
            make(tmp)
            try:
                os.rename(tmp, path)
            except OSError:  # another process was first
                shutil.rmtree(tmp, ignore_errors=True)
        _made[tag] = path
    return _made[tag]


def _block_dir():
    """Evoformer blocks with live gates and LayerNorm parameters."""
    def make(d):
        rng = np.random.default_rng(1)
        prm = {}
        for b in range(STACK_BLOCKS):
            prm.update(bparams.init_block_params(b, rng, gates="random", ln="random"))
        bparams.write_manifest(d, prm)
    return _weights("blocks", make)


def _template_dir():
    def make(d):
        rng = np.random.default_rng(2)
        prm = {}
        for b in range(DEPTHS[0]):
            prm.update(bparams.init_template_block_params(b, rng, gates="random", ln="random"))
        bparams.write_manifest(d, prm)
    return _weights("template", make)


def _design_dirs():
    def make(d):
        rng = np.random.default_rng(3)
        tree = bweights.init_af2_params(rng, num_blocks=DEPTHS[2], extra_blocks=DEPTHS[1],
                                        template_blocks=DEPTHS[0])
        bweights.embed_weights_from_params(tree, os.path.join(d, "emb"))
        bweights.tplembed_weights_from_params(tree, os.path.join(d, "tpl"))
        bweights.stack_weights_from_params(tree, os.path.join(d, "extra"), prefix=bweights.EXTRA)
        bweights.stack_weights_from_params(tree, os.path.join(d, "main"), prefix=bweights.MAIN)
        bweights.post_weights_from_params(tree, os.path.join(d, "post"),
                                          tables=bparams.init_residue_tables(rng))
    root = _weights("design", make)
    return [os.path.join(root, k) for k in ("emb", "tpl", "extra", "main", "post")]


# ---------------------------------------------------------------------- inputs
def _inputs(case, seed):
    """The case's operands on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed * 2654435761 % (1 << 31))
    randn = lambda *sh: torch.randn(*sh, generator=g, device="cuda")  # noqa: E731
    rand = lambda *sh: torch.rand(*sh, generator=g, device="cuda")    # noqa: E731
    kind, n = case["kind"], case["n"]
    x = {}
    if kind == "transition":
        return {"act": randn(case["rows"], n, 128), "dout": randn(case["rows"], n, 128)}
    if kind == "design":
        return _design_inputs(case, randn, rand)
    live = torch.ones(n, device="cuda")
    live[rand(n).argsort()[:round(case["masked"] * n)]] = 0.0  # residues left out
    x["mask"] = torch.outer(live, live)
    c = 64 if kind == "template" else 128
    x["pair"] = randn(n, n, c)
    x["dpair"] = randn(n, n, c)
    if kind in ("triattn", "trimul"):
        x["tbl"] = (rand(n, c) < 0.75).float() / 0.75 if case["drop"] else None
    if kind in ("evoformer", "template"):
        x["seed"] = ops.seed_tensor((seed & 0xFFFF, 7), case["drop"])
    if kind == "evoformer":
        x["msa"] = randn(case["s"], n, 256)
        x["dmsa"] = randn(case["s"], n, 256)
        x["msa_mask"] = live[None].expand(case["s"], n).contiguous()
    return x


def _design_inputs(case, randn, rand):
    """The last 48 residues are designed; the rest is the target, which is
    also the template, so its MSA row joins the main stack."""
    n, dev = case["n"], "cuda"
    nt = case["length"] - 48
    pos = torch.arange(n, device=dev)
    chain = (pos >= nt).float()
    logits = 0.5 * randn(n, 20)
    logits[:nt] = torch.nn.functional.one_hot((20 * rand(nt)).long().clamp(max=19), 20).float()
    flags = torch.where(pos < nt, 2, 1).to(torch.uint8)
    seqm = (pos < case["length"]).float()
    shapes = ((n, 14, 3), (n, n, 64), (n, n, 64), (n, 50), (n, 37))
    conf = ((n,), (n, n), (1,), (1,), (n,), (n,))
    keys = torch.tensor([[0, 11 + i, 1] for i in range(4)], dtype=torch.int64)
    return {"logits": logits, "flags": flags, "seqm": seqm,
            "scalars": torch.tensor([1.0, 0.0, 1.0, 1.0], device=dev),
            "ids": [pos.float(), chain + 1, chain + 1, torch.ones(n, device=dev)],
            "iasym": chain.int(), "act_const": 0.1 * randn(n, n, 64),
            "tpl37": 8.0 * randn(n, 37, 3), "tplm37": torch.ones(n, 37, device=dev),
            "length": torch.tensor([case["length"]], dtype=torch.int32, device=dev),
            "seeds": keys.to(torch.uint32).to(dev) if case["drop"] else None,
            "cts": [randn(*sh) for sh in shapes], "conf_cts": [randn(*sh) for sh in conf],
            "ct37": randn(n, 37, 3)}


def _module(case):
    kind = case["kind"]
    if kind == "triattn":
        return ops.TriangleAttention(_block_dir(), f"param/block0/{TRIATTN[case['flip']]}/",
                                     case["flip"])
    if kind == "trimul":
        return ops.TriangleMultiplication(_block_dir(), f"param/block0/{TRIMUL[case['flip']]}/",
                                          case["flip"])
    if kind == "transition":
        return ops.Transition(_block_dir(), "param/block0/pair_transition/", 128)
    if kind == "evoformer":
        mod = ops.EvoformerStack(_block_dir(), case["depth"])
        mod.prealloc(case["n"], case["s"], case["drop"])
        return mod
    if kind == "template":
        return ops.TemplatePairStack(_template_dir(), DEPTHS[0])
    return ops.DesignStepSeq(*_design_dirs(), depths=DEPTHS)


def prepare(case, seed):
    x = _inputs(case, seed)
    x["case"], x["mod"] = case, _module(case)
    if case["kind"] == "design":  # the design loop keeps one save buffer
        x["save"] = torch.empty(x["mod"].save_bytes(case["n"]), dtype=torch.uint8, device="cuda")
    return x


# ----------------------------------------------------------------------- a pass
def run(x):
    case, mod = x["case"], x["mod"]
    kind = case["kind"]
    if kind in ("triattn", "trimul"):
        out, save = mod.forward(x["pair"], x["mask"], x["tbl"])
        return out, mod.backward(x["pair"], x["mask"], x["tbl"], save, x["dpair"])
    if kind == "transition":
        out, save = mod.forward(x["act"])
        return out, mod.backward(x["act"], None, save, x["dout"])
    if kind == "evoformer":
        pair, msa, save = mod.forward(x["pair"], x["msa"], x["mask"], x["msa_mask"], x["seed"],
                                      dropout=case["drop"], detached=not case["grad"])
        if not case["grad"]:
            return pair, msa
        return (pair, msa, *mod.backward(x["dpair"], x["dmsa"], x["mask"], x["msa_mask"], save,
                                         x["seed"], dropout=case["drop"]))
    if kind == "template":
        out, save = mod.forward(x["pair"], x["mask"], x["seed"], dropout=case["drop"])
        return out, mod.backward(x["dpair"], x["mask"], save, x["seed"], dropout=case["drop"])
    outs, save, conf, (atoms, _) = mod.forward(
        x["logits"], x["flags"], x["scalars"], x["ids"], x["seqm"], act_const=x["act_const"],
        seeds=x["seeds"], dropout=case["drop"], save=x["save"], interface_asym=x["iasym"],
        atom37=True, tpl_atoms37=x["tpl37"], tpl_mask37=x["tplm37"], length=x["length"])
    grad = mod.backward(x["cts"], x["logits"], x["flags"], x["scalars"], x["seqm"], save,
                        dropout=case["drop"], interface_asym=x["iasym"], conf_cts=x["conf_cts"],
                        d_atom37=x["ct37"], length=x["length"])
    return list(outs), list(conf), atoms, grad


# --------------------------------------------------------------- work, tolerance
def _triattn_flops(n, c):
    m = n * n  # projections, scores and values, output; the backward twice that
    return 3 * (2 * m * c * 5 * c + 2 * m * c * 4 + 4 * n * m * c)


def _trimul_flops(n, c):
    m = n * n
    return 3 * (2 * m * c * 6 * c + 2 * n * m * c)


def _block_flops(n, s, c, factor):
    """A block's pair track forward and backward, and its MSA rows' products."""
    m = n * n
    pair = 2 * _triattn_flops(n, c) + 2 * _trimul_flops(n, c) + 3 * 4 * m * c * factor * c
    if s == 0:
        return pair
    cm = 256
    msa = 3 * s * n * (2 * cm * 10 * cm + 16 * cm * cm) + 3 * 4 * s * m * cm
    opm = 3 * (2 * s * m * 32 * 32 + 2 * m * 32 * 32 * c)
    return pair + msa + opm + 3 * 2 * m * c * 8


def work(case):
    kind, n = case["kind"], case["n"]
    m = n * n
    if kind in ("triattn", "trimul"):  # pair, mask, cotangent read; output, gradient written
        f = _triattn_flops(n, 128) if kind == "triattn" else _trimul_flops(n, 128)
        return {"bytes": 4 * m * (4 * 128 + 1), "flops": f}
    if kind == "transition":
        m = case["rows"] * n
        return {"bytes": 4 * m * 4 * 128, "flops": 3 * 4 * m * 128 * 512}
    if kind == "template":
        return {"bytes": 4 * m * (4 * 64 + 1), "flops": 2 * _block_flops(n, 0, 64, 2)}
    block_weights = 4 * 1.8e6
    if kind == "evoformer":
        passes = 1 if case["grad"] else 1 / 3
        carries = (4 if case["grad"] else 2) * (m * 128 + case["s"] * n * 256)
        return {"bytes": 4 * (carries + m) + case["depth"] * block_weights,
                "flops": passes * case["depth"] * _block_flops(n, case["s"], 128, 4)}
    stacks = (DEPTHS[2] * _block_flops(n, 2, 128, 4) + DEPTHS[1] * _block_flops(n, 0, 128, 4)
              + DEPTHS[0] * _block_flops(n, 0, 64, 2))
    return {"bytes": 4 * m * (64 + 4 * 64 + 2) + sum(DEPTHS[1:3]) * block_weights,
            "flops": stacks}


def tolerance(case):
    """About four times how far the outputs move when the input does by one
    binary16 rounding (2^-11.7): binary16 operands, 32-bit sums, a 32-bit
    residual.  Where a transition is differentiated, ReLUs near zero flip with
    a rounding, so a few tokens' gradients move by much more."""
    kind = case["kind"]
    if kind == "triattn":
        return {"rel": 1.4e-3, "max": 0.02}
    if kind == "trimul":
        return {"rel": 2.2e-3, "max": 0.02}
    if kind == "evoformer" and not case["grad"]:
        return {"rel": 1.6e-3, "max": 0.01}
    return {"rel": 0.03, "max": 0.9}


# ------------------------------------------------------ the layers in 64 bits
def _layer_norm(x, p, name):
    mean = x.mean(-1, keepdim=True)
    var = ((x - mean) ** 2).mean(-1, keepdim=True)
    return (x - mean) * torch.rsqrt(var + 1e-5) * p[name + "/scale"] + p[name + "/offset"]


def _linear(x, p, name):
    return x @ p[name + "/weights"] + p[name + "/bias"]


def _attention(x, live, bias, p):
    """Gated attention over the rows of x [B, T, C]; keys with live [B, T] = 0
    all take one score far below any other."""
    h, d = p["attention/query_w"].shape[1:]
    heads = lambda w: (x @ p[f"attention/{w}_w"].flatten(1)).unflatten(-1, (h, d)).transpose(1, 2)  # noqa: E731
    s = heads("query") @ heads("key").transpose(-1, -2) * d ** -0.5
    if bias is not None:
        s = s + bias
    s = torch.where(live[:, None, None, :] > 0, s, torch.full_like(s, -1e8))
    o = (torch.softmax(s, -1) @ heads("value")).transpose(1, 2)
    gate = torch.sigmoid(heads("gating").transpose(1, 2) + p["attention/gating_b"])
    return (o * gate).flatten(2) @ p["attention/output_w"].flatten(0, 1) + p["attention/output_b"]


def _ref_triattn(z, mask, p, ending):
    if ending:
        z, mask = z.transpose(0, 1), mask.transpose(0, 1)
    x = _layer_norm(z, p, "query_norm")
    out = _attention(x, mask, (x @ p["feat_2d_weights"]).permute(2, 0, 1), p)
    return out.transpose(0, 1) if ending else out


def _ref_trimul(z, mask, p, outgoing):
    x = _layer_norm(z, p, "left_norm_input")
    ab = mask[..., None] * _linear(x, p, "projection") * torch.sigmoid(_linear(x, p, "gate"))
    a, b = (t.permute(2, 0, 1) for t in ab.chunk(2, -1))  # [channel, row, column]
    # outgoing: sum_k left[i, k] right[j, k]; incoming: sum_k left[k, j] right[k, i]
    t = a @ b.transpose(1, 2) if outgoing else b.transpose(1, 2) @ a
    t = _linear(_layer_norm(t.permute(1, 2, 0), p, "center_norm"), p, "output_projection")
    return t * torch.sigmoid(_linear(x, p, "gating_linear"))


def _ref_transition(x, p):
    h = torch.relu(_linear(_layer_norm(x, p, "input_layer_norm"), p, "transition1"))
    return _linear(h, p, "transition2")


def _ref_opm(msa, mask, p):
    x = _layer_norm(msa, p, "layer_norm_input")
    a, b = (mask[..., None] * _linear(x, p, f"{s}_projection") for s in ("left", "right"))
    o = torch.einsum("sic,sje->ijce", a, b).flatten(2) @ p["output_w"].flatten(0, 1)
    return (o + p["output_b"]) / (1e-3 + mask.T @ mask)[..., None]


def _ref_block(msa, z, msa_mask, mask, p):
    """One Evoformer block (msa None: a template block) without dropout."""
    if msa is not None:
        z = z + _ref_opm(msa, msa_mask, p("outer_product_mean"))
        q = p("msa_row_attention_with_pair_bias")
        bias = (_layer_norm(z, q, "feat_2d_norm") @ q["feat_2d_weights"]).permute(2, 0, 1)
        msa = msa + _attention(_layer_norm(msa, q, "query_norm"), msa_mask, bias, q)
        q = p("msa_column_attention")
        x = _layer_norm(msa.transpose(0, 1), q, "query_norm")
        msa = msa + _attention(x, msa_mask.T, None, q).transpose(0, 1)
        msa = msa + _ref_transition(msa, p("msa_transition"))
    for flip in (True, False):
        z = z + _ref_trimul(z, mask, p(TRIMUL[flip]), flip)
    for flip in (False, True):
        z = z + _ref_triattn(z, mask, p(TRIATTN[flip]), flip)
    return msa, z + _ref_transition(z, p("pair_transition"))


def _read(directory, block):
    """p(module) -> {parameter: float64 tensor} of one block's weights."""
    found = {}
    with open(os.path.join(directory, "manifest.txt")) as fh:
        for line in fh:
            name, file, _, *shape = line.split()
            if name.startswith(f"param/block{block}/"):
                a = np.fromfile(os.path.join(directory, file), dtype="<f4")
                found[name] = torch.tensor(a.reshape([int(v) for v in shape]),
                                           dtype=torch.float64, device="cuda")
    def p(module):
        head = f"param/block{block}/{module}/"
        return {k[len(head):]: v for k, v in found.items() if k.startswith(head)}
    return p


def exact(case, seed):
    kind = case["kind"]
    if kind == "design" or (kind in ("evoformer", "template") and case["drop"]):
        return None  # minutes of work; the stacks' masks are drawn inside the library
    x = {k: v.double() if torch.is_tensor(v) and v.is_floating_point() else v
         for k, v in _inputs(case, seed).items()}
    if kind == "transition":
        act = x["act"].requires_grad_(True)
        out = act + _ref_transition(act, _read(_block_dir(), 0)("pair_transition"))
        return out.detach(), torch.autograd.grad(out, act, x["dout"])[0]
    z = x["pair"].requires_grad_(True)
    if kind in ("triattn", "trimul"):
        p = _read(_block_dir(), 0)((TRIATTN if kind == "triattn" else TRIMUL)[case["flip"]])
        upd = (_ref_triattn if kind == "triattn" else _ref_trimul)(z, x["mask"], p, case["flip"])
        if x["tbl"] is not None:  # the mask is shared over rows, or columns at the ending node
            upd = upd * (x["tbl"][:, None] if kind == "triattn" and case["flip"] else x["tbl"])
        out = z + upd
        return out.detach(), torch.autograd.grad(out, z, x["dpair"])[0]
    if kind == "template":
        out = z
        for b in range(DEPTHS[0]):
            out = _ref_block(None, out, None, x["mask"], _read(_template_dir(), b))[1]
        return out.detach(), torch.autograd.grad(out, z, x["dpair"])[0]
    msa = x["msa"].requires_grad_(True)
    m, out = msa, z
    with torch.set_grad_enabled(case["grad"]):
        for b in range(case["depth"]):
            m, out = _ref_block(m, out, x["msa_mask"], x["mask"], _read(_block_dir(), b))
    if not case["grad"]:
        return out, m
    grads = torch.autograd.grad((out, m), (z, msa), (x["dpair"], x["dmsa"]))
    return (out.detach(), m.detach(), *grads)
