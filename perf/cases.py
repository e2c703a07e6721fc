"""What is timed when the speed of the operators is compared between two states of the code.

Every case is work that a program built on this package does through its public entry points: single operator calls,
training steps of one layer, and the missing-data network (a Similarity layer over 2x2 patches, pairs of MEX and 2x2
sum pooling, a MEX head) in inference and in training.  Sizes are those of bench.py and of the tests, or generic odd
ones beside them.  All tensors are fp32, as everything in the operators' interface is.

A case is a dict: `kind` says which program, the other entries its sizes and options.
"""
import importlib
import math

import torch

_pkg = importlib.import_module("simnets-tf_amd")

_DEV = "cuda:0"


def listed():
    return [
        # The smallest program: the first two layers of the missing-data network as drop-in calls on one small batch.
        # Launches and the latency of a call are most of it.
        dict(name="first_pair_64", kind="pair", batch=64, side=28, templates=32, instances=64),
        # The Similarity operator at convolution size, the benchmark's headline workload.
        _similarity("similarity_l2_conv", 256, 64, 32, 32, 128),
        # The same operator where no size is a multiple of anything.
        _similarity("similarity_l2_ragged", 37, 45, 29, 35, 75),
        # L1 templates in the middle of a residual-network-like stack at batch 32.
        _similarity("similarity_l1_28", 32, 128, 28, 28, 128, function="L1"),
        # Gaussian log-likelihoods with a quarter of the input missing: normalization term, NaN inputs ignored.
        _similarity("similarity_gaussian_missing", 64, 64, 32, 32, 128, norm=True, missing=0.25),
        # Training of such layers: forward and all three gradients through autograd, both similarity functions.
        _similarity("similarity_train_l2", 32, 128, 28, 28, 128, kind="similarity_train"),
        _similarity("similarity_train_l1", 32, 64, 32, 32, 128, kind="similarity_train", function="L1"),
        # A MEX layer over a large batch: the throughput end of the range that first_pair_64 opens.
        dict(name="mex_large", kind="mex", batch=1024, channels=32, height=16, width=16, instances=64, block=1, stride=1,
             unshared=2),
        # Convolution-like MEX: overlapping 3x3 blocks over all channels, one offsets region, forward and gradients.
        dict(name="mex_train_blocks", kind="mex_train", batch=32, channels=16, height=20, width=20, instances=32,
             block=3, stride=1, unshared=0),
        # The missing-data network serving batches with its parameters prepared once.
        dict(name="stack_serve_512", kind="stack_serve", batch=512, templates=32, width=64),
        # The same network as layer objects on a handful of images: what one request costs.
        dict(name="stack_layers_8", kind="stack_layers", batch=8, templates=32, width=64),
        # A training step of that network: logits and the gradients of all parameters.
        dict(name="stack_train_512", kind="stack_train", batch=512, templates=32, width=64),
    ]


def _similarity(name, batch, channels, height, width, templates, block=3, stride=1, pad=1, function="L2", norm=False,
                missing=0.0, kind="similarity"):
    return dict(name=name, kind=kind, batch=batch, channels=channels, height=height, width=width, templates=templates,
                block=block, stride=stride, pad=pad, function=function, norm=norm, missing=missing)


# ------------------------------------------------------------------------------------------------------- the ranges

def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["pair", "similarity", "similarity", "similarity", "similarity_train", "similarity_train", "mex",
                       "mex_train", "stack_serve", "stack_layers", "stack_train"])
    most = _cost(listed()[1])
    while True:
        if kind == "pair":
            case = dict(kind=kind, batch=_log_int(rng, 16, 256), side=rng.randint(20, 40),
                        templates=_log_int(rng, 16, 64), instances=_log_int(rng, 16, 128))
        elif kind in ("similarity", "similarity_train"):
            side = _log_int(rng, 7, 64)
            case = _similarity("", _log_int(rng, 8, 256), _log_int(rng, 16, 256), side, max(7, side + rng.randint(-3, 3)),
                               _log_int(rng, 32, 256), block=rng.choice([1, 3, 3, 3, 5]), stride=rng.choice([1, 1, 1, 2]),
                               function=rng.choice(["L2", "L2", "L1"]), kind=kind)
            case["pad"] = case["block"] // 2
            if kind == "similarity" and case["function"] == "L2":
                case["norm"] = rng.random() < 0.4
                case["missing"] = 0.25 if case["norm"] and rng.random() < 0.5 else 0.0
        elif kind in ("mex", "mex_train"):
            block = rng.choice([1, 1, 3]) if kind == "mex" else rng.choice([1, 3])
            case = dict(kind=kind, batch=_log_int(rng, 16, 1024), channels=_log_int(rng, 8, 128),
                        height=_log_int(rng, 4, 32), width=_log_int(rng, 4, 32), instances=_log_int(rng, 10, 128),
                        block=block, stride=1, unshared=2 if block == 1 else 0)
        else:
            batch = {"stack_serve": (64, 2048), "stack_layers": (1, 64), "stack_train": (32, 1024)}[kind]
            case = dict(kind=kind, batch=_log_int(rng, *batch), templates=rng.choice([16, 24, 32, 48, 64]),
                        width=rng.choice([32, 48, 64, 96]))
        case.pop("name", None)
        if most / 3000 <= _cost(case) <= most or (kind.startswith("stack") and _cost(case) <= most) or kind == "pair":
            return case


def _cost(case):
    """Terms of the operators' sums in one pass, each direction's counted: what sizes are compared by."""
    return work(case)["flops"]


# ------------------------------------------------------------------------------------------- the programs' sizes

def _out(size, pad, block, stride):
    return (size + 2 * pad - block) // stride + 1


def _first_layer(side):
    """Options of the missing-data network's Similarity layer; its output's side."""
    return dict(blocks=[2, 2], strides=[2, 2], padding=[2, 2], normalization_term=True, ignore_nan_input=True,
                out_of_bounds_value=float("nan")), _out(side, 2, 2, 2)


def _whole_channel(channels, region=2):
    return dict(softmax_mode=True, blocks=[channels, 1, 1], strides=[channels, 1, 1], unshared_offset_region=[region])


def _stack_layers(case):
    """(channels in, instances, side) of the MEX + pooling pairs, and the channels of the head's input."""
    pairs, channels, side, width = [], case["templates"], 16, case["width"]
    while side > 1:
        pairs.append((channels, width, side))
        channels, width, side = width, 2 * width, side // 2
    return pairs, channels


def _mex_options(case):
    b, c = case["block"], case["channels"]
    kw = dict(softmax_mode=True, blocks=[c, b, b], strides=[c, case["stride"], case["stride"]],
              padding=[0, b // 2, b // 2])
    if case["unshared"]:
        kw["unshared_offset_region"] = [case["unshared"]]
    else:
        kw.update(use_unshared_regions=False, shared_offset_region=[-1])
    return kw


# -------------------------------------------------------------------------------------------------- inputs and state

def _normal(gen, *shape, scale=1.0):
    return torch.randn(*shape, generator=gen, device=_DEV) * scale


def _uniform(gen, lo, hi, *shape):
    return torch.rand(*shape, generator=gen, device=_DEV) * (hi - lo) + lo


def _drop(gen, x, share):
    """The values of x that are missing become NaN."""
    return x.masked_fill_(torch.rand(x.shape, generator=gen, device=_DEV) < share, float("nan"))


def prepare(case, seed):
    gen = torch.Generator(device=_DEV)
    gen.manual_seed(seed)
    kind, batch = case["kind"], case["batch"]
    state = dict(kind=kind)
    if kind in ("similarity", "similarity_train"):
        c, o, b = case["channels"], case["templates"], case["block"]
        kw = dict(similarity_function=case["function"], blocks=[b, b], strides=[case["stride"]] * 2,
                  padding=[case["pad"]] * 2)
        x = _normal(gen, batch, c, case["height"], case["width"])
        if case["norm"]:
            kw["normalization_term"] = True
        if case["missing"]:
            x = _drop(gen, x, case["missing"])
            kw.update(ignore_nan_input=True, out_of_bounds_value=float("nan"))
        t, w = _normal(gen, o, c, b, b), _uniform(gen, 0.1, 2.0, o, c, b, b)
        state.update(kw=kw, x=x, t=t, w=w)
        if kind == "similarity_train":
            oh, ow = (_out(case[k], case["pad"], b, case["stride"]) for k in ("height", "width"))
            state["grad"] = _normal(gen, batch, o, oh, ow)
            for k in ("x", "t", "w"):
                state[k].requires_grad_()
    elif kind in ("mex", "mex_train"):
        kw = _mex_options(case)
        c, h, w, n = case["channels"], case["height"], case["width"], case["instances"]
        x = _normal(gen, batch, c, h, w)
        out, offsets = _pkg.mex_output_shape((batch, c, h, w), n, **kw)
        off = _normal(gen, *offsets, scale=0.1)
        state.update(kw=dict(kw, normalize_offsets=True), x=x, off=off, n=n)
        if kind == "mex_train":
            state["grad"] = _normal(gen, *out)
            state["x"].requires_grad_()
            state["off"].requires_grad_()
    elif kind == "pair":
        o, n = case["templates"], case["instances"]
        kw, side = _first_layer(case["side"])
        state.update(x=_drop(gen, _uniform(gen, -0.5, 0.5, batch, 1, case["side"], case["side"]), 0.25),
                     t=_normal(gen, o, 1, 2, 2, scale=0.1), w=_uniform(gen, 0.5, 1.5, o, 1, 2, 2), kw=kw,
                     off=_normal(gen, 4, n, o, 1, 1, scale=0.1), n=n,
                     mex=dict(_whole_channel(o), normalize_offsets=True))
    else:
        o = case["templates"]
        kw, side = _first_layer(28)
        pairs, head = _stack_layers(case)
        x = _drop(gen, _uniform(gen, -0.5, 0.5, batch, 1, 28, 28), 0.25)
        t, w = _normal(gen, o, 1, 2, 2, scale=0.1), _uniform(gen, 0.5, 1.5, o, 1, 2, 2)
        # offsets of a network in training: a few channels weigh most in every sum (nearly equal offsets average the
        # channels' differences away within three layers, and the gradients behind them cancel to rounding noise)
        offs = [_normal(gen, 4, n, c, 1, 1, scale=2.0) for c, n, _ in pairs]
        offs.append(_normal(gen, 1, 10, head, 1, 1, scale=2.0))
        opts = [dict(_whole_channel(c), normalize_offsets=True) for c, _, _ in pairs]
        opts.append(dict(softmax_mode=True, blocks=[head, 1, 1], strides=[head, 1, 1], shared_offset_region=[1],
                         normalize_offsets=True))
        state["x"] = x
        if kind == "stack_serve":
            calls = [_pkg.similarity_mex_sum_pool_prepare(x.shape, t, w, offs[0], pairs[0][1], (2, 2), similarity=kw,
                                                          mex=opts[0])]
            for i, (c, n, s) in list(enumerate(pairs))[1:]:
                calls.append(_pkg.mex_sum_pool_prepare((batch, c, s, s), offs[i], n, (2, 2), **opts[i]))
            calls.append(_pkg.mex_prepare((batch, head, 1, 1), offs[-1], 10, **opts[-1]))
            state["calls"] = calls
        elif kind == "stack_layers":
            state["layers"] = _layer_objects(kw, o, pairs, head, t, w, offs)
        else:
            state.update(kw=kw, params=[p.requires_grad_() for p in [t, w] + offs], opts=opts,
                         instances=[n for _, n, _ in pairs] + [10], grad=_normal(gen, batch, 10, 1, 1))
    return state


def _layer_objects(kw, o, pairs, head, t, w, offs):
    """The network as the package's layer classes, with the given parameters."""
    def of(value):
        return lambda p: p.copy_(value)

    sim = _pkg.Similarity(num_instances=o, strides=kw["strides"], blocks=kw["blocks"], padding=kw["padding"],
                          normalization_term=True, ignore_nan_input=True, out_of_bounds_value=float("nan"),
                          templates_initializer=of(t), weights_initializer=of(w))
    mexes = [_pkg.Mex(num_instances=n, blocks=[c, 1, 1], strides=[c, 1, 1], softmax_mode=True, normalize_offsets=True,
                      unshared_offset_region=[2], offsets_initializer=of(off))
             for (c, n, _), off in zip(pairs, offs)]
    mexes.append(_pkg.Mex(num_instances=10, blocks=[head, 1, 1], strides=[head, 1, 1], softmax_mode=True,
                          normalize_offsets=True, shared_offset_region=[1], offsets_initializer=of(offs[-1])))
    sim.build((1, 1, 28, 28))
    for m, (c, _, s) in zip(mexes, pairs + [(head, 10, 1)]):
        m.build((1, c, s, s))
    return [m.to(_DEV) for m in [sim] + mexes]


# --------------------------------------------------------------------------------------------------------- one pass

def run(state):
    kind = state["kind"]
    if kind == "similarity":
        return _pkg.similarity(state["x"], state["t"], state["w"], **state["kw"])
    if kind == "similarity_train":
        leaves = (state["x"], state["t"], state["w"])
        out = _pkg.layers.similarity(*leaves, **state["kw"])
        return (out.detach(),) + torch.autograd.grad(out, leaves, state["grad"])
    if kind == "mex":
        return _pkg.mex(state["x"], state["off"], state["n"], **state["kw"])
    if kind == "mex_train":
        leaves = (state["x"], state["off"])
        out = _pkg.layers.mex(*leaves, state["n"], **state["kw"])
        return (out.detach(),) + torch.autograd.grad(out, leaves, state["grad"])
    if kind == "pair":
        sim = _pkg.similarity(state["x"], state["t"], state["w"], **state["kw"])
        return sim, _pkg.mex(sim, state["off"], state["n"], **state["mex"])
    cur = state["x"]
    if kind == "stack_serve":
        for call in state["calls"]:
            cur = call(cur)
        return cur
    if kind == "stack_layers":
        layers = state["layers"]
        with torch.no_grad():
            cur = layers[0](cur)
            for m in layers[1:-1]:
                cur = _pkg.sum_pooling(m(cur), (2, 2))
            return layers[-1](cur)
    params, opts, instances = state["params"], state["opts"], state["instances"]
    cur = _pkg.layers.similarity(cur, params[0], params[1], **state["kw"])
    for off, n, kw in zip(params[2:-1], instances, opts):
        cur = _pkg.layers.mex_sum_pool(cur, off, n, (2, 2), **kw)
    out = _pkg.layers.mex(cur, params[-1], instances[-1], **opts[-1])
    return (out.detach(),) + torch.autograd.grad(out, params, state["grad"])


# ------------------------------------------------------------------------------------------- the results in 64 bits

_FUDGE = 0.001  # the interface's default normalization_term_fudge


def _by_images(fn, x, params, grad, want_x=True, step=1):
    """fn(images, *params) in 64 bits, `step` images at a time; with `grad` (fn's result's) also the gradients, the
    parameters' summed over the batch.  Few images at a time bound the memory of the term-by-term sums."""
    params = [p.detach().double() for p in params]
    outs, gx, gp = [], [], [torch.zeros_like(p) for p in params]
    for i in range(0, x.shape[0], step):
        xi = x[i:i + step].detach().double()
        if grad is None:
            outs.append(fn(xi, *params))
            continue
        leaves = [t.clone().requires_grad_() for t in [xi] * want_x + params]
        out = fn(*leaves) if want_x else fn(xi, *leaves)
        g = list(torch.autograd.grad(out, leaves, grad[i:i + step].double()))
        if want_x:
            gx.append(g.pop(0))
        for a, b in zip(gp, g):
            a += b
        outs.append(out.detach())
    out = torch.cat(outs)
    return out if grad is None else (out,) + ((torch.cat(gx),) if want_x else ()) + tuple(gp)


def _exact_similarity(kw):
    (bh, bw), (sh, sw), (ph, pw) = kw["blocks"], kw["strides"], kw["padding"]
    norm, nan, l1 = kw.get("normalization_term"), kw.get("ignore_nan_input"), kw.get("similarity_function") == "L1"

    def fn(x, t, w):
        oh, ow = _out(x.shape[2], ph, bh, sh), _out(x.shape[3], pw, bw, sw)
        x = torch.nn.functional.pad(x, (pw, pw, ph, ph), value=kw.get("out_of_bounds_value", 0.0))
        keep = (x == x).double() if nan else torch.ones_like(x)
        x = torch.where(x == x, x, torch.zeros_like(x)) if nan else x
        # patch element k = (channel, row, column), output pixel
        cols = [v.unfold(2, bh, sh).unfold(3, bw, sw).permute(0, 1, 4, 5, 2, 3).reshape(v.shape[0], -1, oh * ow)
                for v in (x, keep)]
        t, w = t.reshape(t.shape[0], -1), w.reshape(w.shape[0], -1)
        if l1:
            out = torch.cat([-(w[m:m + 8, :, None] * (t[m:m + 8, :, None] - cols[0][:, None]).abs()).sum(2)
                             for m in range(0, t.shape[0], 8)], 1)
        else:
            # NaN inputs are 0 here and their terms weighted 0: products of three matrices give all the sums
            out = -(w @ (cols[0] * cols[0]) - 2 * (w * t) @ cols[0] + (w * t * t) @ cols[1])
        if norm:
            out = 0.5 * (out + (torch.log(w + _FUDGE) - math.log(2 * math.pi)) @ cols[1])
        return out.reshape(x.shape[0], -1, oh, ow)
    return fn


def _exact_mex(kw, instances):
    b, s = kw["blocks"][1], kw["strides"][1]
    p = kw.get("padding", [0, 0, 0])[1]

    def fn(x, off):
        x = torch.nn.functional.pad(x, (p, p, p, p))  # blocks_out_of_bounds_value is 0
        cols = x.unfold(2, b, s).unfold(3, b, s)
        n, c, oh, ow = cols.shape[:4]
        cols = cols.permute(0, 2, 3, 1, 4, 5).reshape(n, oh, ow, -1)
        off = torch.log_softmax(off.reshape(off.shape[0], instances, -1), 2)
        side = math.isqrt(off.shape[0])  # regions interleave: a pixel's is (row, column) modulo the region's side
        out = x.new_zeros(n, instances, oh, ow)
        for r in range(off.shape[0]):
            rh, rw = r // side, r % side
            part = cols[:, rh::side, rw::side]
            top, otop = part.amax(-1, keepdim=True).detach(), off[r].amax(-1, keepdim=True).detach()
            sums = torch.exp(part - top) @ torch.exp(off[r] - otop).T
            out = out.clone()
            out[:, :, rh::side, rw::side] = (torch.log(sums) + top + otop[:, 0]).permute(0, 3, 1, 2)
        return out
    return fn


def exact(case, seed):
    kind, state = case["kind"], prepare(case, seed)
    if kind in ("similarity", "similarity_train"):
        return _by_images(_exact_similarity(state["kw"]), state["x"], (state["t"], state["w"]), state.get("grad"))
    if kind in ("mex", "mex_train"):
        return _by_images(_exact_mex(state["kw"], state["n"]), state["x"], (state["off"],), state.get("grad"))
    if kind == "pair":
        sim = _by_images(_exact_similarity(state["kw"]), state["x"], (state["t"], state["w"]), None, step=16)
        return sim, _by_images(_exact_mex(state["mex"], state["n"]), sim, (state["off"],), None, step=16)
    # the whole network, image by image, from the parameters that the layers and the prepared calls were made of
    pairs, head = _stack_layers(case)
    state = prepare(dict(case, kind="stack_train"), seed)
    kw, opts, instances = state["kw"], state["opts"], state["instances"]

    def network(x, t, w, *offs):
        cur = _exact_similarity(kw)(x, t, w)
        for off, n, opt in zip(offs[:-1], instances, opts):
            cur = 4 * torch.nn.functional.avg_pool2d(_exact_mex(opt, n)(cur, off), 2)
        return _exact_mex(opts[-1], instances[-1])(cur, offs[-1])
    grad = state["grad"] if kind == "stack_train" else None
    return _by_images(network, state["x"], state["params"], grad, want_x=False, step=32)


# ------------------------------------------------------------------------------------------- work and tolerances

# Operations of one term of a sum.  Similarity forward: L2 sub, mul, fused multiply-add; L1 sub, |.|-multiply-add; the
# Gaussian modes one add (and one select) more.  Its gradients: L2 two products each for the input and for the
# parameters; L1 sign and fused multiply-add for the input, sub, sign, fused multiply-add and add for the parameters.  MEX: one fused multiply-add per term in each direction
# (the exponential of a sum is the product of the exponentials).
_SIM_FWD = {"L2": 4, "L1": 3}
_SIM_BWD = {"L2": 4 + 4, "L1": 4 + 5}


def _similarity_work(batch, c, h, w, o, bh, bw, oh, ow, fwd_ops, bwd_ops=0, input_grad=True):
    terms = batch * o * oh * ow * c * bh * bw
    x, p, y = batch * c * h * w, 2 * o * c * bh * bw, batch * o * oh * ow
    words = x + p + y
    if bwd_ops:
        words += y + x + p + (x if input_grad else 0) + p
    return 4 * words, terms * (fwd_ops + bwd_ops)


def _mex_work(batch, c, h, w, n, k, oh, ow, regions, directions, pool=1):
    """directions: 1 forward, 2 with the input gradient or the offsets gradient, 3 with both."""
    terms = batch * n * oh * ow * k
    x, p, y = batch * c * h * w, regions * n * k, batch * n * oh * ow
    words = x + p + y // pool
    if directions > 1:
        words += (directions - 1) * (x + p) + y + y // pool
    return 4 * words, 2 * terms * directions


def work(case):
    kind, batch = case["kind"], case["batch"]
    parts = []
    if kind in ("similarity", "similarity_train"):
        b = case["block"]
        oh, ow = (_out(case[k], case["pad"], b, case["stride"]) for k in ("height", "width"))
        ops = _SIM_FWD[case["function"]] + bool(case["norm"]) + bool(case["missing"])
        parts.append(_similarity_work(batch, case["channels"], case["height"], case["width"], case["templates"], b, b,
                                      oh, ow, ops, _SIM_BWD[case["function"]] if kind == "similarity_train" else 0))
    elif kind in ("mex", "mex_train"):
        h, w, b = case["height"], case["width"], case["block"]
        oh, ow = (_out(s, b // 2, b, case["stride"]) for s in (h, w))
        parts.append(_mex_work(batch, case["channels"], h, w, case["instances"], case["channels"] * b * b, oh, ow,
                               case["unshared"] ** 2 or 1, 3 if kind == "mex_train" else 1))
    elif kind == "pair":
        o, side = case["templates"], case["side"]
        s = _first_layer(side)[1]
        parts.append(_similarity_work(batch, 1, side, side, o, 2, 2, s, s, 6))
        parts.append(_mex_work(batch, o, s, s, case["instances"], o, s, s, 4, 1))
    else:
        o, train = case["templates"], kind == "stack_train"
        pairs, head = _stack_layers(case)
        sim = _similarity_work(batch, 1, 28, 28, o, 2, 2, 16, 16, 6, 5 if train else 0, input_grad=False)
        # inside the network an intermediate tensor is written once and read once; in inference the Similarity
        # layer's output need not exist at all
        parts.append(sim if train else (4 * (batch * 28 * 28 + 8 * o), sim[1]))
        for i, (c, n, s) in enumerate(pairs):
            nbytes, flops = _mex_work(batch, c, s, s, n, c, s, s, 4, 3 if train else 1, pool=4)
            parts.append((nbytes - (0 if train or i else 4 * batch * c * s * s), flops))
        parts.append(_mex_work(batch, head, 1, 1, 10, head, 1, 1, 1, 3 if train else 1))
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


# Four times the largest error of any output against the same path in 64 bits, over the listed cases and some sixty
# drawn ones: (2-norm, largest).  The training step's are those of its hardest output: sum pooling leaves log-likelihoods
# of order a thousand, whose differences decide the head's gradient and carry the last bit of the values themselves.
_TOLERANCE = {
    "pair": (5e-7, 2e-6),
    "similarity": (2.5e-6, 1.2e-5),
    "similarity_train": (3e-6, 3e-5),
    "mex": (3e-6, 1e-5),
    "mex_train": (3e-6, 3e-5),
    "stack_serve": (4e-7, 1e-6),
    "stack_layers": (4e-7, 1e-6),
    "stack_train": (4e-3, 8e-2),
}


def tolerance(case):
    rel, largest = _TOLERANCE[case["kind"]]
    return {"rel": rel, "max": largest}
