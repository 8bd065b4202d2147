"""Workloads of the quantized GEMM engine, as a program that serves a model with it runs them.

Four kinds of pass, each through the public binding (abq-llm_amd/abq_gemm.py) and the C ABI it exposes:

  layer   the quantized linears of decoder layers (QKV, O, gate + up with the fused SiLU gate, down): fp16 activations,
          quantised per token on the device, weights with scales and zero points per group of 128 or 64, fp16 out.
          The record formats and the choice between them per call are those of the weight loader and
          ABQGEMMWrapper::gemm_dynamic (abq-llm_amd/ft).
  static  the drop-in call of the FasterTransformer layers (ABQGEMMWrapper::gemm): fp16 activations packed with one
          static scale, weights prepared once, fp16 out with one scale per tensor.
  int     the integer engine: int32 out on operands that are packed already ("records"), or with the activations
          packed from int32 by the call, on weights in the plane format ("planes") or prepared ones ("prepared").
  load    a loader bringing one layer's weights from integer codes to everything the calls above read.

A pass walks through `copies` sets of weights (the layers of a model), so that a small call does not find its weights
in a cache that the next layers' weights would have displaced.
"""
import importlib.util
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "abq-llm_amd")


def _binding():
    # (the package directory's name is no Python identifier: the binding is loaded by its path)
    if "abq_gemm" not in sys.modules:
        path = os.path.join(os.getcwd(), "abq-llm_amd", "abq_gemm.py")
        if not os.path.exists(path):
            path = os.path.join(_PKG, "abq_gemm.py")
        spec = importlib.util.spec_from_file_location("abq_gemm", path)
        module = importlib.util.module_from_spec(spec)
        sys.modules["abq_gemm"] = module
        spec.loader.exec_module(module)
    return sys.modules["abq_gemm"]


abq = _binding()

# every bit pair of the engine's sweep at 128 rows, (activation bits, weight bits)
SWEEP_PAIRS = [(2, 2), (3, 3), (4, 4), (5, 5), (6, 6), (7, 7), (8, 8), (4, 2), (6, 2), (8, 2), (8, 4)]


# ------------------------------------------------------------------------------------------------- the cases

def listed():
    return [
        # one token through eight layers of the 7B shapes: the decode step of a single user
        {"name": "layer_w2a8_1_token", "kind": "layer", "x_bits": 8, "w_bits": 2, "group": 128, "symmetric": True,
         "rows": 1, "hidden": 4096, "ffn": 11008, "copies": 8},
        # sixteen sequences decoded together
        {"name": "layer_w2a8_16_tokens", "kind": "layer", "x_bits": 8, "w_bits": 2, "group": 128, "symmetric": True,
         "rows": 16, "hidden": 4096, "ffn": 11008, "copies": 8},
        # a small batch of an odd size, 4-bit weights, activations with a zero point
        {"name": "layer_w4a8_asym_43_tokens", "kind": "layer", "x_bits": 8, "w_bits": 4, "group": 128, "symmetric": False,
         "rows": 43, "hidden": 4096, "ffn": 11008, "copies": 4},
        # the prefill of one sequence of 1024 tokens
        {"name": "layer_w2a8_1024_tokens", "kind": "layer", "x_bits": 8, "w_bits": 2, "group": 128, "symmetric": True,
         "rows": 1024, "hidden": 4096, "ffn": 11008, "copies": 2},
        # the prefill of sixteen such sequences, the largest call
        {"name": "layer_w2a8_16384_tokens", "kind": "layer", "x_bits": 8, "w_bits": 2, "group": 128, "symmetric": True,
         "rows": 16384, "hidden": 4096, "ffn": 11008, "copies": 1},
        # the 13B shapes on 4-bit operands, a prompt of an odd length
        {"name": "layer_w4a4_777_tokens", "kind": "layer", "x_bits": 4, "w_bits": 4, "group": 128, "symmetric": True,
         "rows": 777, "hidden": 5120, "ffn": 13824, "copies": 1},
        # the engine's headline GEMMs at one row, operands resident as records, int32 out
        {"name": "int_w2a8_1_row", "kind": "int", "form": "records", "x_bits": 8, "w_bits": 2, "signed": True,
         "rows": 1, "hidden": 4096, "ffn": 11008, "copies": 8},
        # the reference engine's own calls: pack the activations, then init's kernel on plane operands, nothing prepared
        {"name": "int_planes_w2a8_4_rows", "kind": "int", "form": "planes", "x_bits": 8, "w_bits": 2, "signed": True,
         "rows": 4, "hidden": 4096, "ffn": 11008, "copies": 8},
        # the sweep of all bit pairs at 128 rows on the 13B shapes, unsigned codes, weights prepared
        {"name": "int_sweep_128_rows", "kind": "int", "form": "sweep", "x_bits": 0, "w_bits": 0, "signed": False,
         "rows": 128, "hidden": 5120, "ffn": 13824, "copies": 1},
        # prefill through the drop-in call, 8-bit operands
        {"name": "static_w8a8_512_rows", "kind": "static", "x_bits": 8, "w_bits": 8, "signed": True,
         "rows": 512, "hidden": 4096, "ffn": 11008, "copies": 2},
        # the same on 4-bit operands and four times the rows
        {"name": "static_w4a4_2048_rows", "kind": "static", "x_bits": 4, "w_bits": 4, "signed": True,
         "rows": 2048, "hidden": 4096, "ffn": 11008, "copies": 2},
        # one layer's weights through the loader
        {"name": "load_w2_layer", "kind": "load", "x_bits": 8, "w_bits": 2, "group": 128, "symmetric": True,
         "rows": 0, "hidden": 4096, "ffn": 11008, "copies": 1},
    ]


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["layer", "layer", "layer", "int", "int", "static", "load"])
        hidden = 128 * int(round(math.exp(rng.uniform(math.log(8), math.log(64)))))
        ffn = 128 * int(round(hidden / 128 * rng.uniform(2.0, 3.5)))
        case = {"kind": kind, "hidden": hidden, "ffn": ffn, "copies": rng.randint(1, 4)}
        if kind == "layer":
            x_bits, w_bits = rng.choice([(8, 2), (8, 2), (8, 3), (8, 4), (8, 8), (4, 4), (4, 2)])
            case.update(x_bits=x_bits, w_bits=w_bits, group=rng.choice([128, 128, 64]), symmetric=rng.random() < 0.6,
                        rows=_rows(rng, 1, 16384))
        elif kind == "int":
            form = rng.choice(["records", "planes", "prepared", "prepared"])
            x_bits, w_bits = rng.choice(SWEEP_PAIRS + [(8, 3)])
            signed = rng.random() < 0.6
            if form == "records":  # (operands of one field, as the quantising kernel writes them)
                x_bits, w_bits = rng.choice([(8, 2), (8, 4), (4, 4), (2, 2), (8, 8), (4, 2)])
                signed = signed or 8 in (x_bits, w_bits)
            # (planes without a workspace: the reference engine has kernels of up to 8 rows)
            case.update(form=form, x_bits=x_bits, w_bits=w_bits, signed=signed,
                        rows=_rows(rng, 1, {"records": 2048, "planes": 64, "prepared": 2048}[form]))
        elif kind == "static":
            x_bits, w_bits = rng.choice([(8, 8), (4, 4), (8, 4), (8, 2)])
            case.update(x_bits=x_bits, w_bits=w_bits, signed=True, rows=_rows(rng, 1, 4096))
        else:
            case.update(x_bits=8, w_bits=rng.choice([2, 3, 4]), group=128, symmetric=True, rows=0, copies=1)
        if _cost(case) <= most:
            return case


def _rows(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _gemms(case):
    """(N, K, columns of the output) of the GEMMs of one copy"""
    h, f = case["hidden"], case["ffn"]
    if case["kind"] in ("layer", "load"):
        return [(3 * h, h, 3 * h), (h, h, h), (2 * f, h, f), (h, f, h)]
    return [(h, h, h), (f, h, f), (h, f, h)]


def work(case):
    m, nbytes, flops = case["rows"], 0.0, 0.0
    for n, k, cols in _gemms(case):
        if case["kind"] == "load":
            p, g = case["w_bits"], case["group"]
            # codes, scales and zero points in; records of the codes' own width, folded records and the rank-one term out
            fold = _plan(case)["folded"]
            nbytes += 4.0 * n * k + 8.0 * n * k / g + n * k * (p + fold) / 8 + 4 * n
            if p == 4:
                nbytes += 0.75 * n * k
            continue
        for q, p in (SWEEP_PAIRS if case.get("form") == "sweep" else [(case["x_bits"], case["w_bits"])]):
            flops += 2.0 * m * n * k
            nbytes += p * n * k / 8.0
            if case["kind"] == "layer":
                nbytes += 8.0 * n * k / case["group"] + 2.0 * m * k + 2.0 * m * cols + 4 * m
            elif case["kind"] == "static":
                nbytes += 2.0 * m * k + 2.0 * m * n
            else:
                nbytes += (q / 8.0 if case["form"] == "records" else 4.0) * m * k + 4.0 * m * n
    return {"bytes": nbytes * case["copies"], "flops": flops * case["copies"]}


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 5e12, w["flops"] / 1.5e15)


def tolerance(case):
    # Integer results, and the reference's per-tensor fp16 epilogue (its roundings are part of its definition), leave no
    # choice.  Dequantised outputs are sums of the same terms in fp32, rounded once to fp16 (half an ulp is 2^-11 of the
    # value).  Against the path in fp64 the listed cases measure 2.1e-4 of the result's norm, 6e-4 where a quotient next to
    # a rounding tie falls on the other side of an 8-bit code (a zero point more so), and 6e-3 where that is a 4-bit
    # code; single values then are off by 0.02 and 0.2 of the result's root mean square.
    if case["kind"] == "layer":
        return {"rel": 2e-3, "max": 0.08} if case["x_bits"] == 8 else {"rel": 2.4e-2, "max": 0.8}
    return "exact"


# ------------------------------------------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _activations(gen, rows, k):
    """fp16 rows as a transformer's linears meet them: every token at its own level, a few channels far above the rest"""
    x = torch.randn((rows, k), generator=gen, device="cuda")
    level = torch.exp(0.5 * torch.randn((rows, 1), generator=gen, device="cuda"))
    channel = torch.ones(k, device="cuda")
    channel[torch.randint(0, k, (max(1, k // 512),), generator=gen, device="cuda")] = 8.0
    return (x * level * channel).half()


def _quantised_weights(gen, n, k, bits, group):
    """random-init weights N(0, 0.02) quantised per group as the converter does: (signed codes, scales, zero points)"""
    w = torch.randn((n, k // group, group), generator=gen, device="cuda").mul_(0.02)
    lo, hi = w.amin(2, keepdim=True), w.amax(2, keepdim=True)
    scale = ((hi - lo) / (2 ** bits - 1)).clamp_(1e-5, 1e4)
    zero = torch.round(-lo / scale)
    codes = torch.round(w / scale).add_(zero).clamp_(0, 2 ** bits - 1)
    half = 2.0 ** (bits - 1)
    return ((codes - half).to(torch.int32).view(n, k), scale.view(n, k // group).contiguous(),
            (zero - half).view(n, k // group).contiguous())


def _codes(gen, rows, k, bits, signed, sigma=None):
    lo, hi = (-(1 << (bits - 1)), (1 << (bits - 1)) - 1) if signed else (0, (1 << bits) - 1)
    if sigma is None:
        return torch.randint(lo, hi + 1, (rows, k), generator=gen, device="cuda", dtype=torch.int32)
    v = torch.randn((rows, k), generator=gen, device="cuda").mul_(sigma)
    return v.round_().clamp_(lo, hi).to(torch.int32)


def prepare(case, seed):
    gen = _gen(seed)
    state = {"case": case, "lib": abq.lib()}
    if case["kind"] == "layer":
        _prepare_layer(case, gen, state)
    elif case["kind"] == "static":
        _prepare_static(case, gen, state)
    elif case["kind"] == "load":
        state["weights"] = [_quantised_weights(gen, n, k, case["w_bits"], case["group"]) for n, k, _ in _gemms(case)]
    else:
        _prepare_int(case, gen, state)
    return state


def run(state):
    return {"layer": _run_layer, "static": _run_static, "load": _run_load, "int": _run_int}[state["case"]["kind"]](state)


# ------------------------------------------------------------------------------------------------- decoder-layer linears

def _plan(case):
    """Which records a loader keeps of a weight matrix (ABQDeviceWeight): `own` = (width, zero points left) of the
    records every size can run on, `folded` = width of those with the zero points folded in (0: none)."""
    q, p = case["x_bits"], case["w_bits"]
    folded, padded = abq.lib().abq_folded_bits(p), abq.padded_bits(p)
    if folded and not len(abq.native_configs(q, folded, True)):
        folded = 0
    if padded != p and folded == padded:  # as wide as the padded records: they serve every call
        return {"own": padded, "zero": False, "folded": folded}
    return {"own": padded, "zero": True, "folded": folded}


def _load_weight(case, codes, scale, zero):
    """What the loader makes of one matrix: dict of records, scales, zero points and the rank-one term"""
    p, group, plan = case["w_bits"], case["group"], _plan(case)
    planes = abq.pack_i32(codes, p)
    w = {"scale": scale, "zero": zero, "term": abq.weight_zero_term(planes, True, scale, zero, group), "own": None, "folded": None, "fp6": None}
    if plan["zero"]:
        w["own"] = abq.relayout_planes(planes) if plan["own"] == p else abq.relayout_planes_padded(planes, True)
    if plan["folded"]:
        w["folded"] = abq.relayout_planes_folded(planes, zero, group, True)
    if group == 128 and p <= 4 and (case["kind"] == "load" and p == 4 or case["kind"] == "layer" and abq.fp6_eligible(case["x_bits"], p, True, codes.shape[1])):
        w["fp6"] = abq.relayout_planes_fp6_folded(planes, zero, 128, True)
    return w


def _prepare_layer(case, gen, state):
    q, p, group, m, sym = case["x_bits"], case["w_bits"], case["group"], case["rows"], case["symmetric"]
    plan = _plan(case)
    h, f = case["hidden"], case["ffn"]
    x_in, x_attn, x_mlp = (_activations(gen, m, h) for _ in range(3))
    k_max = max(h, f)
    # buffers a serving program keeps: the quantised activations of the call under way, with scales, zero points, sums
    packed = torch.empty(m * k_max * (6 if q <= 5 else q) // 32 + 64, dtype=torch.int32, device="cuda")
    x_scale, x_zero = (torch.empty(m, dtype=torch.float32, device="cuda") for _ in range(2))
    sums = torch.empty(m * (k_max // group), dtype=torch.int32, device="cuda")
    calls = []
    for _ in range(case["copies"]):
        gate_out = torch.empty((m, f), dtype=torch.float16, device="cuda")
        for x, (n, k, cols), act in zip((x_in, x_attn, x_mlp, gate_out), _gemms(case), (0, 0, 1, 0)):
            w = _load_weight(case, *_quantised_weights(gen, n, k, p, group))
            out = gate_out if act else torch.empty((m, cols), dtype=torch.float16, device="cuda")
            kw = dict(out=out, out_kind=abq.OUT_F16_SCALED, x_scale=x_scale, w_scale=w["scale"], group_size=group, act=act)
            own = plan["own"]
            decode = abq.prepared_decode_pays(q, own, True, m, n, k, group, act)
            fp6 = (not decode and w["fp6"] is not None
                   and abq.lib().abq_preferred_weight_layout(q, p, 1, m, n, k, 128) == abq.LAYOUT_FP6)
            zero_in = dict(x_zero=None if sym else x_zero, w_zero_term=None if sym else w["term"])
            layout = abq.LAYOUT_TILED
            if fp6:
                g = abq.Gemm(packed[: m * k * 6 // 32].view(k // 128, m, 24), w["fp6"], True, x_fp6=q, w_fp6=p, **zero_in, **kw)
                layout = abq.LAYOUT_FP6
            else:
                xr = packed[: m * k * q // 32].view(k // 128, m, q, 4)
                folded = w["folded"] is not None and (not plan["zero"] or (not decode and m > 16))
                rec = w["folded"] if folded else w["own"]
                in_kernel = decode and q == 8 and m <= 16 and m * k <= 16384 and (m == 1 or n <= 4096)
                if not folded:
                    zero_in.update(w_zero=w["zero"], x_group_sums=sums)
                vb = None if rec.shape[2] == p or folded else (q, p)
                g = None
                if in_kernel:
                    g = abq.Gemm(xr, rec, True, x_tiled=True, w_tiled=True, value_bits=vb, **kw)
                    try:
                        g.set_dynamic_f16_activations(x, sym, w_zero=None if folded else w["zero"], w_zero_term=zero_in["w_zero_term"])
                        layout = None
                    except abq.AbqError:
                        g = None
                if g is None:
                    g = abq.Gemm(xr, rec, True, x_tiled=True, w_tiled=True, value_bits=vb, **zero_in, **kw)
            if g.workspace_bytes:
                raise RuntimeError("operands are packed: no workspace expected")
            calls.append((g, x, k, layout, w))
    state.update(calls=calls, packed=packed, x_scale=x_scale, x_zero=x_zero, sums=sums)


def _run_layer(state):
    case, L = state["case"], state["lib"]
    q, m, group, sym = case["x_bits"], case["rows"], case["group"], case["symmetric"]
    stream = torch.cuda.current_stream().cuda_stream
    packed, x_scale, sums = state["packed"].data_ptr(), state["x_scale"].data_ptr(), state["sums"].data_ptr()
    x_zero = None if sym else state["x_zero"].data_ptr()
    outs = []
    for g, x, k, layout, _ in state["calls"]:
        if layout is not None:
            rc = L.abq_quant_pack_f16(x.data_ptr(), m, k, q, int(sym), layout, packed, x_scale, x_zero, sums, group, stream)
            if rc:
                raise abq.AbqError(rc, "abq_quant_pack_f16")
        outs.append(g.run(stream))
    return outs


# ------------------------------------------------------------------------------------------------- static scale, fp16 out

def _prepare_static(case, gen, state):
    q, p, m = case["x_bits"], case["w_bits"], case["rows"]
    h, f = case["hidden"], case["ffn"]
    # codes small enough for their sums to stay within fp16, as the reference's epilogue needs
    sigma = {2: 1.0, 4: 2.0, 8: 6.0}
    step = torch.full((1,), 4.0, dtype=torch.float32, device="cuda")
    top = 2.0 ** (q - 1)
    xs = {k: torch.randn((m, k), generator=gen, device="cuda").mul_(sigma[q]).clamp_(-top, top - 1).mul_(0.25).half() for k in (h, f)}
    scale_out = torch.full((1,), 0.01, dtype=torch.float32, device="cuda")
    packed = torch.empty(m * max(h, f) * (6 if q <= 5 else q) // 32 + 64, dtype=torch.int32, device="cuda")
    calls = []
    for _ in range(case["copies"]):
        for n, k, _cols in _gemms(case):
            planes = abq.pack_i32(_codes(gen, n, k, p, True, sigma=2.0 * sigma[p]), p)
            out = torch.empty((m, n), dtype=torch.float16, device="cuda")
            kw = dict(out=out, out_kind=abq.OUT_F16_TENSOR_F32SCALE, c_scale=scale_out)
            if m > 16 and abq.lib().abq_preferred_weight_layout(q, p, 1, m, n, k, 0) == abq.LAYOUT_FP6:
                w = abq.relayout_planes_fp6(planes, True)
                g = abq.Gemm(packed[: m * k * 6 // 32].view(k // 128, m, 24), w, True, x_fp6=q, w_fp6=p, **kw)
                layout = abq.LAYOUT_FP6
            else:
                w = abq.relayout_planes(planes)
                g = abq.Gemm(packed[: m * k * q // 32].view(k // 128, m, q, 4), w, True, x_tiled=True, w_tiled=True, **kw)
                layout = abq.LAYOUT_TILED
                if q == 8 and m * k <= 32768 and (n <= 4096 or (m == 1 and n <= 12288)):  # as ABQGEMMWrapper::gemm
                    try:
                        g.set_f16_activations(xs[k], step)
                        layout = None
                    except abq.AbqError:
                        pass
            calls.append((g, xs[k], k, layout))
    state.update(calls=calls, packed=packed, step=step)


def _run_static(state):
    case, L = state["case"], state["lib"]
    q, m = case["x_bits"], case["rows"]
    stream = torch.cuda.current_stream().cuda_stream
    packed, step = state["packed"].data_ptr(), state["step"].data_ptr()
    outs = []
    for g, x, k, layout in state["calls"]:
        rc = 0
        if layout == abq.LAYOUT_FP6:
            rc = L.abq_pack_f16_fp6(x.data_ptr(), step, packed, m, k, q, 1, stream)
        elif layout == abq.LAYOUT_TILED:
            rc = L.abq_pack_f16_tiled(x.data_ptr(), step, packed, m, k, q, stream)
        if rc:
            raise abq.AbqError(rc, "abq_pack_f16")
        outs.append(g.run(stream))
    return outs


# ------------------------------------------------------------------------------------------------- integer engine

def _prepare_int(case, gen, state):
    m, signed, form = case["rows"], case["signed"], case["form"]
    pairs = SWEEP_PAIRS if form == "sweep" else [(case["x_bits"], case["w_bits"])]
    # activations N(0, 32) for signed 8 bits as in a quantised layer, the full range otherwise
    xs, ws, calls = {}, None, []
    for q, p in pairs:
        for k in {case["hidden"], case["ffn"]}:
            if (q, k) not in xs:
                xs[q, k] = _codes(gen, m, k, q, signed, sigma=32.0 if signed and q == 8 else None)
    planes_of = {key: abq.planes_empty(key[0], m, key[1]) for key in xs}
    records = {}
    for _ in range(case["copies"]):
        for q, p in pairs:
            for n, k, _cols in _gemms(case):
                out = torch.empty((m, n), dtype=torch.int32, device="cuda")
                wp = abq.pack_i32(_codes(gen, n, k, p, signed), p)
                if form == "planes":
                    calls.append([(q, k), planes_of[q, k], wp, dict(out=out)])
                elif form == "records":
                    if (q, k) not in records:
                        records[q, k] = abq.relayout_planes(abq.pack_i32(xs[q, k], q))
                    calls.append([None, records[q, k], abq.relayout_planes(wp), dict(out=out, x_tiled=True, w_tiled=True)])
                else:
                    calls.append([(q, k), planes_of[q, k], *_prepared_weight(q, p, signed, m, n, k, wp, out)])
    gemms = [abq.Gemm(x, w, signed, **kw) for _, x, w, kw in calls]
    if form in ("prepared", "sweep"):
        # one workspace for all calls of the stream, sized as the states ask
        ws = torch.empty(max(g.workspace_bytes for g in gemms) + 1024, dtype=torch.uint8, device="cuda")
        gemms = [abq.Gemm(x, w, signed, workspace=ws, **kw) for _, x, w, kw in calls]
    state.update(xs=xs, planes_of=planes_of, calls=[(key, g) for (key, *_), g in zip(calls, gemms)], ws=ws)


def _prepared_weight(q, p, signed, m, n, k, planes, out):
    """(weight operand, arguments of Gemm) in the records that the library prefers for the shape"""
    width = abq.ctypes.c_int(0)
    layout = abq.lib().abq_preferred_weight_records(q, p, int(signed), m, n, k, 0, abq.ctypes.byref(width))
    kw = dict(out=out)
    if layout == abq.LAYOUT_FP6:
        kw.update(w_fp6=p)
        return abq.relayout_planes_fp6(planes, signed), kw
    kw.update(w_tiled=True)
    if width.value != p:
        kw.update(value_bits=(q, p), x_planes_of=abq.padded_bits(q))
        return abq.relayout_planes_padded(planes, signed), kw
    if not signed and 8 in (q, p):
        kw.update(w_row_sums=abq.row_sums(planes))
        if (q, p) == (8, 8) and m > 128:
            kw.update(biased=(False, True))
            return abq.relayout_planes_biased(planes), kw
    return abq.relayout_planes(planes), kw


def _run_int(state):
    L, xs, planes_of = state["lib"], state["xs"], state["planes_of"]
    stream = torch.cuda.current_stream().cuda_stream
    outs, packed = [], None
    for key, g in state["calls"]:
        if key is not None and key != packed:
            q, k = key
            rc = L.abq_pack_i32(xs[key].data_ptr(), planes_of[key].data_ptr(), xs[key].shape[0], k, q, stream)
            if rc:
                raise abq.AbqError(rc, "abq_pack_i32")
            packed = key
        outs.append(g.run(stream))
    return outs


# ------------------------------------------------------------------------------------------------- weight loading

def _run_load(state):
    outs = []
    for codes, scale, zero in state["weights"]:
        w = _load_weight(state["case"], codes, scale, zero)
        outs.append([w["own"], w["folded"], w["fp6"], w["term"]])
    return outs
