"""Performance cases of turboadam_amd.

Three entry points carry the work a training program gives this package:

* ``TurboAdam.step()`` over a parameter list (kind "step"): the whole point of
  the package, at every size, parameter dtype and compression mode, eagerly
  and replayed from a captured graph;
* ``CoStateManager.update`` (kind "costate") and ``quantize.fused_v_update``
  (kind "fused_v"): the same moments one tensor at a time, for programs that
  build their own optimizer around the codecs;
* ``oneq.compress_v_logscale`` / ``oneq.decompress_v`` (kind "codec"): encode
  and decode of a second moment, as checkpoint conversion and inspection do.

A step case starts in the middle of training: the optimizer is loaded with a
state dict at step 100 whose packed moments are drawn from the seed, and two
gradient sets alternate from pass to pass.  Parameters live in flat buffers
(one per layer or one for the model), as sharded and bucketed training keeps
them, so all of them come back as a few outputs; the optimizer's own state
comes back for as many parameters as the number of outputs allows, the largest
and the smallest ones first.
"""

import math
import random

import torch

BLOCK = 128
START_STEP = 100
MAX_OUTPUTS = 62
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
BETAS = (0.9, 0.999)
EPS = 1e-8


# ------------------------------------------------------------------ shapes
def _gpt2_block():
    return [(768,), (768,), (768, 2304), (2304,), (768, 768), (768,), (768,), (768,), (768, 3072), (3072,),
            (3072, 768), (768,)]


def _gpt2():
    return [[(50257, 768), (1024, 768)]] + [_gpt2_block() for _ in range(12)] + [[(768,), (768,)]]


def _llama_layer():
    h, kv, inter = 4096, 1024, 14336
    return [(h, h), (kv, h), (kv, h), (h, h), (inter, h), (inter, h), (h, inter), (h,), (h,)]


def _llama_8b():
    return [[(128256, 4096)]] + [_llama_layer() for _ in range(32)] + [[(4096,), (128256, 4096)]]


def _ragged(count, log2_max, seed):
    """Sizes log-uniform from 1 to 2**log2_max, most of them no multiple of anything."""
    r = random.Random(seed)
    return [(max(1, round(2.0 ** (log2_max * r.random()))),) for _ in range(count)]


def _spread(count, total, seed):
    """count sizes around total / count, within a factor of eight either way."""
    r = random.Random(seed)
    w = [8.0 ** r.uniform(-1, 1) for _ in range(count)]
    return [(max(1, round(total * x / sum(w))),) for x in w]


def _groups(case):
    """The parameters' shapes, as a list of flat buffers' lists."""
    s = case["shapes"]
    if s == "gpt2-block":
        return [_gpt2_block()]
    if s == "gpt2-block-vectors":  # its norms and biases alone
        return [[x for x in _gpt2_block() if len(x) == 1]]
    if s == "gpt2":
        return _gpt2()
    if s == "llama-layer":
        return [_llama_layer()]
    if s == "llama-8b":
        return _llama_8b()
    if s == "ragged":
        return [_ragged(case["count"], case["log2_max"], case["sizes_seed"])]
    return [_spread(case["count"], case["total"], case["sizes_seed"])]


def _step(name, shapes, dtype, **kw):
    c = dict(name=name, kind="step", shapes=shapes, dtype=dtype, v_bits=4, compress_m=True, compress_v=True,
             error_feedback=False, null_pct=0.10, amp_pct=0.90, weight_decay=0.01, graph=False, packed=False,
             log_sigma=math.log(1e-3))
    c.update(kw)
    return c


def listed():
    return [
        # fine-tuning the norms and biases of one block only: nothing but latency and launches
        _step("vectors_f32", "gpt2-block-vectors", "f32"),
        # one GPT-2 block, the reference's own speed benchmark
        _step("block_f32", "gpt2-block", "f32", weight_decay=0.0),
        # the same block trained in fp16 with the whole step in a captured graph
        _step("block_f16_graph", "gpt2-block", "f16", graph=True, v_bits=6),
        # a small model trained whole in fp32
        _step("gpt2_f32", "gpt2", "f32"),
        # many odd-sized tensors (adapters, convolutions, embeddings of every size), few bits, tight thresholds
        _step("ragged_f32", "ragged", "f32", count=1000, log2_max=20.0, sizes_seed=0, v_bits=3, null_pct=0.05,
              amp_pct=0.95, weight_decay=0.0),
        # one large tensor with only v compressed (m kept in fp32)
        _step("v_only_f32", "flat", "f32", count=1, total=1 << 28, sizes_seed=0, compress_m=False),
        # one 8B-model layer with only m compressed (v kept in fp32)
        _step("layer_bf16_m_only", "llama-layer", "bf16", compress_v=False, weight_decay=0.1),
        # one 8B-model layer with error feedback on m
        _step("layer_bf16_ef", "llama-layer", "bf16", error_feedback=True, weight_decay=0.1),
        # the headline: every parameter of an 8B model in bf16, both moments compressed
        _step("llama8b_bf16", "llama-8b", "bf16", weight_decay=0.1, log_sigma=math.log(1e-4)),
        # the moments one tensor at a time: an MLP matrix's m, an attention matrix's v
        dict(name="costate_update", kind="costate", n=3072 * 768, dtype="f32", error_feedback=False),
        dict(name="fused_v_update", kind="fused_v", n=4096 * 4096, dtype="bf16", v_bits=4),
        # encode and decode of an embedding's second moment (checkpoint conversion)
        dict(name="v_codec", kind="codec", n=50257 * 768, v_bits=4, stochastic=False),
    ]


def draw(rng):
    kind = rng.choices(["step", "costate", "fused_v", "codec"], [0.7, 0.1, 0.1, 0.1])[0]
    if kind != "step":
        n = round(2.0 ** rng.uniform(13, 26))
        if kind == "costate":
            return dict(kind=kind, n=n, dtype=rng.choice(list(DTYPES)), error_feedback=rng.random() < 0.25)
        if kind == "fused_v":
            return dict(kind=kind, n=n, dtype=rng.choice(list(DTYPES)), v_bits=rng.choice([2, 3, 4, 6, 8]))
        return dict(kind=kind, n=n, v_bits=rng.choice([2, 3, 4, 6, 8]), stochastic=rng.random() < 0.5)
    mode = rng.choices(["m+v", "v", "m", "ef"], [0.55, 0.15, 0.15, 0.15])[0]
    null_pct, amp_pct = rng.choice([(0.10, 0.90), (0.05, 0.95)])
    c = _step("", "", rng.choice(list(DTYPES)), v_bits=rng.choice([2, 3, 4, 4, 4, 6, 8]), compress_m=mode != "v",
              compress_v=mode != "m", error_feedback=mode == "ef", null_pct=null_pct, amp_pct=amp_pct,
              weight_decay=rng.choice([0.0, 0.01, 0.1]), graph=rng.random() < 0.15, packed=rng.random() < 0.15,
              sizes_seed=rng.randrange(1 << 20))
    del c["name"]
    if rng.random() < 0.3:
        c.update(shapes="ragged", count=round(2.0 ** rng.uniform(3, 9.5)), log2_max=round(rng.uniform(14, 21), 2))
    else:
        total = round(2.0 ** rng.uniform(14, 28.5))
        c.update(shapes="spread", total=total, count=min(round(2.0 ** rng.uniform(0, 8.3)), max(1, total // 2048)))
    return c


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(n, g):
    return torch.randn(n, generator=g, device="cuda", dtype=torch.float32)


def _rand(n, g):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float32)


def _nb(n):
    return (n + BLOCK - 1) // BLOCK


def _packed_v(n, sigma, bits, g):
    """1Q state of a second moment around sigma**2: indices clustered in each
    block's log range, ranges of two to nine nats."""
    nb, levels = _nb(n), 1 << bits
    idx = (_randn(nb * BLOCK, g) * (levels / 5.0) + levels * 0.55).clamp_(0, levels - 1).to(torch.uint8)
    lo = 2 * math.log(sigma) - 1.0 - 5.0 * _rand(nb, g)
    return idx, torch.stack([lo, lo + 2.0 + 7.0 * _rand(nb, g)], 1).to(torch.float16)


def _packed_m(n, sigma, g):
    """CoState encoding of a first moment: alpha, labels, signs, norms, amplitudes."""
    nb = _nb(n)
    u = _rand(nb, g)
    signs = torch.randint(0, 256, ((n + 7) // 8,), generator=g, device="cuda", dtype=torch.uint8)
    if n % 8:
        signs[-1] &= (0xFF00 >> (n % 8)) & 0xFF
    norms = sigma * math.sqrt(BLOCK) * (0.1 + 0.3 * _rand(nb, g))
    return {"alpha": (0.2 + 0.2 * _rand(1, g)).reshape(()),
            "labels": (u >= 0.1).to(torch.uint8) + (u >= 0.9).to(torch.uint8), "sign_packed": signs,
            "block_norms": norms, "scales": (norms / math.sqrt(BLOCK)).to(torch.float16)}


def _step_inputs(case, seed):
    """Flat parameter buffers, their parameters' views, two gradient sets and
    each parameter's optimizer state, from the seed alone."""
    g, r = _gen(seed), random.Random(int(seed))
    dtype = DTYPES[case["dtype"]]
    slot = 1 if case["packed"] else 64
    flats, views, grads, states = [], [], ([], []), []
    for shapes in _groups(case):
        sizes = [math.prod(s) for s in shapes]
        offs = [0]
        for n in sizes:
            offs.append(offs[-1] + (n + slot - 1) // slot * slot)
        flat = torch.zeros(offs[-1], dtype=dtype, device="cuda")
        gflat = [torch.zeros_like(flat) for _ in range(2)]
        for shape, n, o in zip(shapes, sizes, offs):
            sigma = math.exp(case["log_sigma"] + r.gauss(0, 1))
            flat[o:o + n] = _randn(n, g).mul_(0.02)
            common = _randn(n, g).mul_(0.3)
            for k in range(2):
                z = _randn(n, g).add_(common).mul_(sigma)
                gflat[k][o:o + n] = z
                grads[k].append(gflat[k][o:o + n].view(shape))
            views.append(flat[o:o + n].view(shape))
            st = {"sigma": sigma}
            if case["compress_v"]:
                st["v"] = _packed_v(n, sigma, case["v_bits"], g)
            else:
                st["exp_avg_sq"] = _randn(n, g).square_().mul_(sigma * sigma).view(shape)
            if case["compress_m"] and n >= 4096:
                st["m"] = _packed_m(n, sigma, g)
                if case["error_feedback"]:
                    st["residual"] = _randn(n, g).mul_(0.1 * sigma).view(shape)
            else:
                st["exp_avg"] = _randn(n, g).mul_(0.3 * sigma).view(shape)
            states.append(st)
        flats.append(flat)
    return flats, views, grads, states


def _hyper(case):
    return dict(lr=3e-4, betas=BETAS, eps=EPS, weight_decay=case["weight_decay"], v_bits=case["v_bits"],
                compress_m=case["compress_m"], compress_v=case["compress_v"], null_pct=case["null_pct"],
                amp_pct=case["amp_pct"], error_feedback=case["error_feedback"], capturable=case["graph"])


def _state_dict(case, opt, views, states):
    """The optimizer state dict a checkpoint at START_STEP holds."""
    from turboadam_amd.costate import CoStateManager

    out = {}
    for i, (p, st) in enumerate(zip(views, states)):
        d = {"step": START_STEP, "_compress_m": "m" in st}
        if "v" in st:
            d["compressed_v"] = {"indices": st["v"][0], "scales": st["v"][1], "n_bits": case["v_bits"],
                                 "original_shape": p.shape, "original_length": p.numel(), "block_size": BLOCK}
        else:
            d["exp_avg_sq"] = st["exp_avg_sq"]
        if "m" in st:
            mgr = CoStateManager(error_feedback=case["error_feedback"], null_pct=case["null_pct"],
                                 amp_pct=case["amp_pct"])
            mgr._has_state, mgr._original_numel, mgr._alpha = True, p.numel(), st["m"]["alpha"]
            mgr._encoded = {k: st["m"][k] for k in ("labels", "sign_packed", "block_norms", "scales")}
            mgr._ef_residual = st.get("residual")
            d["m_mgr"] = mgr
        else:
            d["exp_avg"] = st["exp_avg"]
        out[i] = d
    return {"state": out, "param_groups": opt.state_dict()["param_groups"]}


def _state_tensors(opt, p):
    """The state arrays of one parameter."""
    st = opt.state[p]
    out = {}
    if "compressed_v" in st:
        out["v_indices"], out["v_scales"] = st["compressed_v"]["indices"], st["compressed_v"]["scales"]
    else:
        out["exp_avg_sq"] = st["exp_avg_sq"]
    if st["_compress_m"]:
        mgr = st["m_mgr"]
        out.update(alpha=mgr._alpha, labels=mgr._encoded["labels"], signs=mgr._encoded["sign_packed"],
                   norms=mgr._encoded["block_norms"], amps=mgr._encoded["scales"])
        if mgr._ef_residual is not None:
            out["residual"] = mgr._ef_residual
    else:
        out["exp_avg"] = st["exp_avg"]
    return out


def _reported(case):
    """Positions of the parameters whose state comes back: the largest, the
    smallest, the second largest, ... while the outputs last."""
    groups = _groups(case)
    sizes = [math.prod(s) for shapes in groups for s in shapes]
    order = sorted(range(len(sizes)), key=lambda i: (-sizes[i], i))
    mixed = [order[k // 2] if k % 2 == 0 else order[-1 - k // 2] for k in range(len(order))]
    left, out = MAX_OUTPUTS - len(groups), []
    for i in mixed:
        left -= 8 if case["compress_m"] and sizes[i] >= 4096 else 3
        if left < 0:
            break
        out.append(i)
    return out


def prepare(case, seed):
    if case["kind"] == "step":
        return _prepare_step(case, seed)
    g = _gen(seed)
    n = case["n"]
    if case["kind"] == "costate":
        from turboadam_amd.costate import CoStateManager

        mgr = CoStateManager(error_feedback=case["error_feedback"])
        m = _packed_m(n, 1e-3, g)
        mgr.allocate(n, torch.device("cuda", torch.cuda.current_device()))
        mgr._alpha.copy_(m["alpha"])
        for k, t in mgr._encoded.items():
            t.copy_(m[k])
        mgr._has_state, mgr._original_numel = True, n
        grad = _randn(n, g).mul_(1e-3).to(DTYPES[case["dtype"]])
        if case["error_feedback"]:
            mgr._ef_residual = _randn(n, g).mul_(1e-4)
        return {"kind": "costate", "mgr": mgr, "grad": grad}
    if case["kind"] == "fused_v":
        idx, scales = _packed_v(n, 1e-3, case["v_bits"], g)
        grad = _randn(n, g).mul_(1e-3).to(DTYPES[case["dtype"]])
        return {"kind": "fused_v", "idx": idx, "scales": scales, "grad": grad, "bits": case["v_bits"]}
    v = _randn(n, g).mul_(1e-3).square_()
    idx, scales = _packed_v(n, 1e-3, case["v_bits"], g)
    packed = {"indices": idx, "scales": scales, "n_bits": case["v_bits"], "original_shape": torch.Size([n]),
              "original_length": n, "block_size": BLOCK}
    return {"kind": "codec", "v": v, "packed": packed, "bits": case["v_bits"], "stochastic": case["stochastic"]}


def _prepare_step(case, seed):
    from turboadam_amd import TurboAdam

    flats, views, grads, states = _step_inputs(case, seed)
    params = [torch.nn.Parameter(v) for v in views]
    opt = TurboAdam(params, **_hyper(case))
    sd = _state_dict(case, opt, views, states)
    opt.load_state_dict(sd)
    out = {"params": flats, "state": {}}
    s = {"kind": "step", "opt": opt, "params": params, "grads": grads, "pass": 0, "out": out, "graph": None}
    if case["graph"]:
        # one eager step to warm up, the capture, then the values as they were before it
        kept = [f.clone() for f in flats]
        held = [{k: t.clone() for k, t in _state_tensors(opt, p).items()} for p in params]
        for p, g in zip(params, grads[0]):
            p.grad = g
        opt.step()
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            opt.step()
        for f, k in zip(flats, kept):
            f.copy_(k)
        for p, h in zip(params, held):
            for k, t in _state_tensors(opt, p).items():
                t.copy_(h[k])
            opt.state[p]["step"].fill_(START_STEP)
        torch.cuda.synchronize()
    out["state"] = {str(i): _state_tensors(opt, params[i]) for i in _reported(case)}
    return s


# ------------------------------------------------------------------ the pass
def run(s):
    if s["kind"] == "step":
        if s["graph"] is not None:
            s["graph"].replay()
            return s["out"]
        for p, g in zip(s["params"], s["grads"][s["pass"] & 1]):  # this step's gradients
            p.grad = g
        s["pass"] += 1
        s["opt"].step()
        return s["out"]
    if s["kind"] == "costate":
        mgr = s["mgr"]
        m = mgr.update(s["grad"], BETAS[0])
        out = {"m": m, "alpha": mgr._alpha, **mgr._encoded}
        if mgr._ef_residual is not None:
            out["residual"] = mgr._ef_residual
        return out
    if s["kind"] == "fused_v":
        from turboadam_amd.quantize import fused_v_update

        idx, scales, v = fused_v_update(s["idx"], s["scales"], s["grad"], BETAS[1], s["bits"])
        return {"indices": idx, "scales": scales, "v": v}
    from turboadam_amd.oneq import compress_v_logscale, decompress_v

    c = compress_v_logscale(s["v"], s["bits"], stochastic_round=s["stochastic"])
    return {"indices": c["indices"], "scales": c["scales"], "values": decompress_v(s["packed"])}


# ------------------------------------------------------------------ what a pass cannot do without
def _tensor_bytes(case, n):
    """Each input read once and each output written once, for one parameter."""
    e = DTYPES[case["dtype"]].itemsize
    nb = _nb(n)
    b = 3 * e * n  # parameter in and out, gradient in
    b += 2 * (nb * BLOCK + 4 * nb) if case["compress_v"] else 8 * n
    if case["compress_m"] and n >= 4096:
        b += 2 * (n // 8 + 7 * nb) + (8 * n if case["error_feedback"] else 0)
    else:
        b += 8 * n
    return b


def work(case):
    if case["kind"] == "step":
        sizes = [math.prod(s) for shapes in _groups(case) for s in shapes]
        # about 50 operations an element: both moments, their codecs, the update
        return {"bytes": sum(_tensor_bytes(case, n) for n in sizes), "flops": 50 * sum(sizes)}
    n, nb = case["n"], _nb(case["n"])
    if case["kind"] == "costate":
        e = DTYPES[case["dtype"]].itemsize
        ef = 8 if case["error_feedback"] else 0
        return {"bytes": (e + 4 + ef) * n + 2 * (n // 8 + 7 * nb), "flops": 20 * n}
    if case["kind"] == "fused_v":
        return {"bytes": (DTYPES[case["dtype"]].itemsize + 4) * n + 2 * (nb * BLOCK + 4 * nb), "flops": 20 * n}
    return {"bytes": 8 * n + 2 * (nb * BLOCK + 4 * nb), "flops": 20 * n}


def tolerance(case):
    """Every result is defined bit for bit (correctly rounded functions, sums in
    a fixed order, counter-based draws), so another correct implementation of
    the same contract gives the same bits."""
    return "exact"


# ------------------------------------------------------------------ 64 bits
def _blocks(x, fill):
    nb = _nb(x.numel())
    out = torch.full((nb * BLOCK,), fill, dtype=torch.float64, device=x.device)
    out[:x.numel()] = x
    return out.view(nb, BLOCK)


def _decode_m(m, gf):
    """alpha*g + the block's scale with the element's sign."""
    n = gf.numel()
    shift = torch.arange(7, -1, -1, device="cuda", dtype=torch.uint8)
    neg = ((m["sign_packed"].unsqueeze(1) >> shift) & 1).reshape(-1)[:n].double()
    s = torch.where(m["labels"] == 1, m["block_norms"].double() / math.sqrt(BLOCK),
                    torch.where(m["labels"] == 2, m["scales"].double(), 0.0))
    return m["alpha"].double() * gf + s.repeat_interleave(BLOCK)[:n] * (1.0 - 2.0 * neg)


def _encode_m(m, gf):
    """alpha, block norms and amplitudes of the new encoding."""
    alpha = (m * gf).sum() / (gf * gf).sum()
    norms = _blocks(m - alpha * gf, 0.0).square().sum(1).sqrt()
    return alpha, norms, norms / math.sqrt(BLOCK)


def _decode_v(idx, scales, bits):
    sc = scales.double()
    lo, span = sc[:, :1], sc[:, 1:] - sc[:, :1]
    return torch.exp(lo + (idx.view(-1, BLOCK).double() + 0.5) / (1 << bits) * span).reshape(-1)


def _v_scales(v):
    lv = v.clamp(min=1e-38).log()
    return torch.stack([_blocks(lv, math.inf).amin(1), _blocks(lv, -math.inf).amax(1)], 1)


def exact(case, seed):
    if case["kind"] == "step":
        return _exact_step(case, seed)
    g, n = _gen(seed), case["n"]
    if case["kind"] == "costate":
        enc = _packed_m(n, 1e-3, g)
        gf = _randn(n, g).mul_(1e-3).to(DTYPES[case["dtype"]]).double()
        ge = gf + _randn(n, g).mul_(1e-4).double() if case["error_feedback"] else gf
        m = BETAS[0] * _decode_m(enc, gf) + (1 - BETAS[0]) * ge
        alpha, norms, amps = _encode_m(m, gf)
        out = {"m": m, "alpha": alpha, "labels": None, "sign_packed": None, "block_norms": norms, "scales": amps}
        if case["error_feedback"]:
            out["residual"] = None  # follows the labels, which ties decide
        return out
    if case["kind"] == "fused_v":
        idx, scales = _packed_v(n, 1e-3, case["v_bits"], g)
        gf = _randn(n, g).mul_(1e-3).to(DTYPES[case["dtype"]]).double()
        v = BETAS[1] * _decode_v(idx, scales, case["v_bits"])[:n] + (1 - BETAS[1]) * gf * gf
        return {"indices": None, "scales": _v_scales(v), "v": v}
    v = _randn(n, g).mul_(1e-3).square_().double()
    idx, scales = _packed_v(n, 1e-3, case["v_bits"], g)
    lv = _blocks(v.clamp(min=1e-38).log(), v.min().clamp(min=1e-38).log().item())
    return {"indices": None, "scales": torch.stack([lv.amin(1), lv.amax(1)], 1),
            "values": _decode_v(idx, scales, case["v_bits"])[:n]}


def _exact_step(case, seed):
    flats, views, grads, states = _step_inputs(case, seed)
    b1, b2 = BETAS
    lr, wd, t = 3e-4, case["weight_decay"], START_STEP + 1
    bc1, bc2 = 1 - b1 ** t, 1 - b2 ** t
    keep, out = set(_reported(case)), {"params": [], "state": {}}
    slot = 1 if case["packed"] else 64
    i = 0
    for flat, shapes in zip(flats, _groups(case)):
        new = torch.zeros(flat.numel(), dtype=torch.float64, device="cuda")
        o = 0
        for shape in shapes:
            p, gf, st = views[i].reshape(-1).double(), grads[0][i].reshape(-1).double(), states[i]
            n, d = p.numel(), {}
            if "v" in st:
                v = b2 * _decode_v(*st["v"], case["v_bits"])[:n] + (1 - b2) * gf * gf
                d.update(v_indices=None, v_scales=_v_scales(v) if i in keep else None)
            else:
                v = b2 * st["exp_avg_sq"].reshape(-1).double() + (1 - b2) * gf * gf
                d["exp_avg_sq"] = v.view(shape)
            if "m" in st:
                ge = gf + st["residual"].reshape(-1).double() if "residual" in st else gf
                m = b1 * _decode_m(st["m"], gf) + (1 - b1) * ge
                if i in keep:
                    alpha, norms, amps = _encode_m(m, gf)
                    d.update(alpha=alpha, labels=None, signs=None, norms=norms, amps=amps)
                if "residual" in st:
                    d["residual"] = None  # follows the labels, which ties decide
            else:
                m = b1 * st["exp_avg"].reshape(-1).double() + (1 - b1) * gf
                d["exp_avg"] = m.view(shape)
            new[o:o + n] = p * (1 - lr * wd) - lr / bc1 * m / ((v / bc2).sqrt() + EPS)
            if i in keep:
                out["state"][str(i)] = d
            del p, gf, v, m, d
            o += (n + slot - 1) // slot * slot
            i += 1
        out["params"].append(new)
    return out
