"""Performance cases of the LUT layers: the calls a user's program makes, over the sizes it makes
them at.  Every case goes through the public classes (LUTLayer, ProjectionLUTLayer,
LUTTransformer, LUTDataManagerI.forward_step_i8).

  listed()   named cases, each with what it stands for
  draw(rng)  one more case of the same ranges
  prepare / run / work / tolerance / exact   see each function

A case is a dict of plain values.  `kind` selects the path:

  fc           LUTLayer: `train` (forward + backward) or evaluation; `summation` float32 or
               int32; `policy` of the weight gradient, Dense or Sparse (applied to the weights)
  int8         evaluation over int8 tables with a scale a table, int32 sums
  projection   ProjectionLUTLayer (sparse connectivity), forward + backward
  seq          sequence-concat LUTLayer (causal attention), train or evaluation
  product      pair-product LUTLayer, forward + backward
  transformer  LUTTransformer, evaluation, returning the logits
"""
import math

import torch

from spiky_amd import (GradientPolicy, GradientType, LUTDataManagerI, LUTLayer, LUTTransformer,
                       ProjectionLUTLayer)
from spiky_amd.util.synapse_growth import PointSamplingPolicy, PointSamplingType

INT_RESCALER = 0.001   # the layers' default fixed-point scale
DENOM = 1048575.0      # int32 fixed point: one unit is 1 / (DENOM * rescaler)
GROUP = 32             # the layers' default block of tables (forward) and outputs (backward)
TABLE_STD = 0.01
DESCENT = 1e-3         # learning rate of the step that applies a sparse gradient


def listed():
    fc = dict(kind="fc", train=True, summation="float32", policy="Dense")
    return [
        # a small classifier (28 x 28 pixels, 10 classes) in training: launches and latency count
        dict(fc, name="fc_small_train", B=64, I=784, T=256, Nc=6, O=10),
        # a large layer answering one request
        dict(fc, name="fc_single_eval", train=False, B=1, I=4096, T=8192, Nc=8, O=1024),
        # an ordinary layer in training, at sizes that are multiples of nothing
        dict(fc, name="fc_ragged_train", B=100, I=784, T=1000, Nc=7, O=301),
        # the headline layer: 8.6 GB of tables, forward and backward
        dict(fc, name="fc_large_train", B=1024, I=4096, T=8192, Nc=8, O=1024),
        # training with int32 fixed-point sums, for results that do not depend on any order
        dict(fc, name="fc_int32_train", summation="int32", B=256, I=1024, T=1024, Nc=8, O=256),
        # training with sparse weight gradients and a plain descent step: few samples, many rows
        dict(fc, name="fc_sparse_grad_train", policy="Sparse", B=32, I=1024, T=1024, Nc=8, O=256),
        # batch inference of the headline layer with int8 tables
        dict(name="int8_eval", kind="int8", B=4096, I=4096, T=8192, Nc=8, O=1024),
        # the first layer of a convolutional stack on 28 x 28 images, mostly black
        dict(name="projection_train", kind="projection", B=128, side=28, out_side=48, grid=12, stride=2,
             pad=2.0, per_group=32, Nc=5, field=5, patch_h=4, patch_w=4),
        # one attention layer of a byte-level transformer in training
        dict(name="seq_train", kind="seq", train=True, B=32, S=256, I=256, T=64, Nc=6, pd=4, O=256),
        # the same layer over the one sequence of a prompt
        dict(name="seq_single_eval", kind="seq", train=False, B=1, S=256, I=256, T=64, Nc=6, pd=4, O=256),
        # the pair-product form of that attention layer in training
        dict(name="product_train", kind="product", train=True, B=32, S=256, I=256, T=64, Nc=6, pd=4, O=256),
        # a whole transformer evaluating a few prompts
        dict(name="transformer_eval", kind="transformer", B=4, S=256, V=256, E=256, layers=4, heads=4,
             n_det=16, Nc=8, Nc_att=6, pd=4),
    ]


# ---------------------------------------------------------------------- draws
def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _near(rng, values):
    """One of the usual widths, or a little off it (odd sizes among them)."""
    v = rng.choice(values)
    return v if rng.random() < 0.5 else max(3, v - rng.randrange(1, max(2, v // 4)))


def _draw_fc(rng):
    while True:
        c = dict(kind="fc", train=rng.random() < 0.7, summation="float32", policy="Dense",
                 B=_log(rng, 1, 2048), I=_near(rng, [64, 256, 784, 1024, 4096]), T=_log(rng, 16, 8192),
                 Nc=rng.randint(4, 10), O=_near(rng, [10, 32, 64, 256, 512, 1024]))
        option = rng.random()
        if option < 0.2:
            c.update(summation="int32")
        elif option < 0.4:
            c.update(policy="Sparse", train=True, B=min(c["B"], 64))
        numel = (c["T"] << c["Nc"]) * c["O"]
        if numel <= 1 << 29 and c["B"] * c["T"] * c["O"] <= 1 << 31 and 2 * c["Nc"] <= c["I"]:
            return c


def _draw_int8(rng):
    while True:
        c = dict(kind="int8", B=_log(rng, 1, 4096), I=_near(rng, [256, 784, 1024, 4096]),
                 T=_log(rng, 64, 8192), Nc=rng.randint(4, 8), O=4 * _near(rng, [16, 64, 128, 256]))
        if c["B"] * c["T"] * c["O"] <= 1 << 34 and (c["T"] << c["Nc"]) * c["O"] <= 1 << 31:
            return c


def _draw_projection(rng):
    grid = rng.randint(5, 12)
    return dict(kind="projection", B=_log(rng, 8, 256), side=28, out_side=48, grid=grid, stride=2, pad=2.0,
                per_group=rng.choice([4, 8, 12, 16]), Nc=rng.randint(4, 6), field=rng.choice([3, 5]),
                patch_h=rng.randint(2, 5), patch_w=rng.randint(3, 6))


def _draw_pairs(rng, kind):
    while True:
        c = dict(kind=kind, train=kind == "product" or rng.random() < 0.6, B=_log(rng, 1, 32),
                 S=_log(rng, 12, 256), I=_near(rng, [64, 128, 256]), T=_log(rng, 8, 64),
                 Nc=rng.randint(4, 6), pd=rng.choice([0, 2, 3, 4]), O=_near(rng, [32, 64, 128, 256]))
        if kind == "product" or c["T"] * c["O"] << (2 * c["Nc"] + c["pd"]) <= 1 << 30:
            return c


def draw(rng):
    kind = rng.choice(["fc", "fc", "fc", "int8", "projection", "seq", "product", "transformer"])
    if kind == "fc":
        return _draw_fc(rng)
    if kind == "int8":
        return _draw_int8(rng)
    if kind == "projection":
        return _draw_projection(rng)
    if kind == "transformer":
        return dict(kind=kind, B=rng.randint(1, 4), S=_log(rng, 32, 256), V=_near(rng, [64, 256]),
                    E=_near(rng, [64, 128, 256]), layers=rng.randint(1, 4), heads=rng.choice([2, 4]),
                    n_det=_log(rng, 8, 16), Nc=rng.randint(6, 8), Nc_att=rng.randint(4, 6),
                    pd=rng.choice([2, 4]))
    return _draw_pairs(rng, kind)


# ---------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _anchors(gen, T, n, Nc):
    """Nc pairs of 2 * Nc distinct inputs for each of T tables, as int32 [T * Nc * 2]."""
    picks = [torch.rand(min(1024, T - t), n, device="cuda", generator=gen).topk(2 * Nc, dim=1).indices
             for t in range(0, T, 1024)]
    return torch.cat(picks).to(torch.int32).reshape(-1).contiguous()


def _fill_tables(layers, gen):
    with torch.no_grad():
        for layer in layers:
            layer._weights.normal_(0.0, TABLE_STD, generator=gen)


def _images(gen, B, side):
    """Uniform pixels, about 80 % of them black."""
    x = torch.rand(B, 1, side, side, device="cuda", generator=gen)
    return x * (torch.rand(B, 1, side, side, device="cuda", generator=gen) > 0.8)


def _projection_layer(case):
    policy = PointSamplingPolicy(PointSamplingType.Grid, pad_h=case["pad"], pad_w=case["pad"],
                                 grid_h=case["grid"], grid_w=case["grid"], stride_h=case["stride"],
                                 stride_w=case["stride"])
    return ProjectionLUTLayer((case["side"],) * 2, (case["out_side"],) * 2, case["Nc"], case["grid"] ** 2,
                              case["per_group"], (case["field"],) * 2, (case["patch_h"], case["patch_w"]),
                              detectors_sampling_policy=policy, random_seed=1,
                              device=torch.device("cuda"))


def _sequence_layer(case, gen):
    product = case["kind"] == "product"
    n = 2 * case["I"] + case["pd"] if product else case["I"]
    return LUTLayer(case["I"], case["Nc"], case["T"], case["O"], sequence_length=case["S"],
                    concatenation_product=not product, positional_dim=case["pd"],
                    _explicit_anchors=_anchors(gen, case["T"], n, case["Nc"]), random_seed=1,
                    device=torch.device("cuda"))


def prepare(case, seed):
    """The layer (or tables) with its anchors and weights, the inputs and the upstream gradient."""
    gen = _generator(seed)
    kind = case["kind"]
    state = dict(kind=kind, train=case.get("train", kind in ("projection", "product")))
    if kind == "int8":
        B, I, T, Nc, O = (case[k] for k in ("B", "I", "T", "Nc", "O"))
        dm = LUTDataManagerI(I, O, T, Nc, 1, 0, 0, GROUP, GROUP, INT_RESCALER)
        dm.register_synapse_meta(1.0, -1.0, 1.0, 0.0, 0.0)
        dm.initialize_neurons(True)
        dm.to_device(torch.cuda.current_device())
        state.update(dm=dm, B=B, anchors=_anchors(gen, T, I, Nc),
                     q=torch.randint(-127, 128, ((T << Nc) * O,), device="cuda", generator=gen,
                                     dtype=torch.int8),
                     scales=torch.rand(T, device="cuda", generator=gen) * 0.009 + 0.001,
                     x=torch.randn(B * I, device="cuda", generator=gen),
                     out=torch.empty(B * O, device="cuda"),
                     idx=torch.empty(B * T, dtype=torch.int32, device="cuda"))
        return state
    if kind == "transformer":
        model = LUTTransformer(vocab_size=case["V"], embedding_dim=case["E"], context_size=case["S"],
                               positional_dim=case["pd"], num_layers=case["layers"],
                               num_heads=case["heads"], n_detectors=case["n_det"],
                               n_anchors_per_detector=case["Nc"],
                               n_anchors_per_detector_attention=case["Nc_att"], seed=int(seed) + 1,
                               device=torch.device("cuda"))
        _fill_tables(model._lut_layers(), gen)
        model.eval()
        state.update(model=model, x=torch.randint(0, case["V"], (case["B"], case["S"]), device="cuda",
                                                  generator=gen))
        return state
    if kind == "fc":
        layer = LUTLayer(case["I"], case["Nc"], case["T"], case["O"],
                         weights_gradient_policy=GradientPolicy(GradientType[case["policy"]]),
                         summation_dtype=getattr(torch, case["summation"]), _int_rescaler=INT_RESCALER,
                         _explicit_anchors=_anchors(gen, case["T"], case["I"], case["Nc"]),
                         random_seed=1, device=torch.device("cuda"))
        x = torch.randn(case["B"], 1, case["I"], device="cuda", generator=gen)
        g_shape = (case["B"], 1, case["O"])
    elif kind == "projection":
        layer = _projection_layer(case)
        x = _images(gen, case["B"], case["side"])
        g_shape = (case["B"], 1, case["out_side"], case["out_side"])
    else:
        layer = _sequence_layer(case, gen)
        x = torch.randn(case["B"], case["S"], case["I"], device="cuda", generator=gen)
        g_shape = (case["B"], case["S"], case["O"])
    _fill_tables([layer], gen)
    layer.train(state["train"])
    state.update(layer=layer, x=x)
    if state["train"]:
        x.requires_grad_(True)
        state["g"] = torch.randn(g_shape, device="cuda", generator=gen)
    return state


def run(state):
    """Training: the output and every gradient of one forward and backward, and in the place of a
    sparse weight gradient, whose length varies, the weights it was applied to.  Evaluation: the
    output (with the lookup indices over int8 tables)."""
    if state["kind"] == "int8":
        state["out"].zero_()
        state["dm"].forward_step_i8(state["q"], state["scales"], state["B"], state["x"], state["anchors"],
                                    state["out"], state["idx"])
        return {"y": state["out"], "idx": state["idx"]}
    if not state["train"]:
        with torch.no_grad():
            return {"y": state.get("model", state.get("layer"))(state["x"])}
    layer, x = state["layer"], state["x"]
    params = {"w": layer._weights, "pe": layer._positional_embeddings}
    x.grad = None
    for p in params.values():
        if p is not None:
            p.grad = None
    y = layer(x)
    y.backward(state["g"])
    result = {"y": y.detach(), "x_grad": x.grad}
    for name, p in params.items():
        if p is None:
            continue
        if p.grad.is_sparse:
            with torch.no_grad():
                p.add_(p.grad, alpha=-DESCENT)
            result[name] = p.detach()
        else:
            result[name + "_grad"] = p.grad
    return result


# ---------------------------------------------------------------------- what a pass cannot do without
def _fc_work(B, I, T, Nc, O, train, entry=4, sparse=False):
    """The table rows that the samples select (all of them at large batches), read in the forward
    and, with the flipped rows, again in the backward, whose upstream gradient comes in between;
    inputs, outputs and gradients once.  A dense weight gradient is written whole; a sparse one is
    an index and a value for each selected entry, written, read and applied."""
    E = 1 << Nc
    rows = T * min(E, B)
    size = rows * O * entry + B * I * 4 + B * O * 4 + T * Nc * 8
    flops = B * T * (O + Nc)
    if train:
        size += T * min(E, 2 * B) * O * 4 + B * O * 4 + B * I * 4
        size += rows * O * 32 if sparse else T * E * O * 4
        flops += B * T * O * 5
    return size, flops


def work(case):
    kind = case["kind"]
    if kind in ("fc", "int8"):
        size, flops = _fc_work(case["B"], case["I"], case["T"], case["Nc"], case["O"],
                               case.get("train", False), 1 if kind == "int8" else 4,
                               case.get("policy") == "Sparse")
    elif kind == "projection":
        # a group's rows project on a patch of the output: every synapse weight is read forward and
        # backward, and its gradient written
        T = case["grid"] ** 2 * case["per_group"]
        row = case["patch_h"] * case["patch_w"]
        pixels = case["B"] * (case["side"] ** 2 + case["out_side"] ** 2) * 4
        size = 3 * (T << case["Nc"]) * row * 4 + 2 * pixels + T * case["Nc"] * 8
        flops = 6 * case["B"] * T * row
    elif kind == "transformer":
        rows, T = case["B"] * case["S"], case["n_det"] * case["heads"]
        att_bytes, att_flops = _pairs_work(case["B"], case["S"], case["E"], T, case["Nc_att"], case["pd"],
                                           case["E"], False, True)
        ffn_bytes, ffn_flops = _fc_work(rows, case["E"], case["n_det"], case["Nc"], case["E"], False)
        out_bytes, out_flops = _fc_work(rows, case["E"], case["n_det"], case["Nc"], case["V"], False)
        size = case["layers"] * (att_bytes + ffn_bytes) + out_bytes
        flops = case["layers"] * (att_flops + ffn_flops) + out_flops
    else:
        size, flops = _pairs_work(case["B"], case["S"], case["I"], case["T"], case["Nc"], case["pd"],
                                  case["O"], case["train"], kind == "seq")
    return {"bytes": size, "flops": flops}


def _pairs_work(B, S, I, T, Nc, pd, O, train, concat):
    """Every causal pair (i < j) of a sequence selects one row of each table."""
    E = 1 << (2 * Nc + pd if concat else Nc)
    pairs = B * S * (S - 1) // 2
    rows = T * min(E, pairs)
    activations = B * S * (I + O) * 4 + (S - 1) * T * pd * 4
    size = rows * O * 4 + activations
    flops = pairs * T * O
    if train:
        size += T * min(E, 2 * pairs) * O * 4 + T * E * O * 4 + activations
        flops += 5 * pairs * T * O
    return size, flops


# ---------------------------------------------------------------------- how far right answers lie apart
def tolerance(case):
    """int8 tables: the int32 sums are fixed by the format.  Elsewhere sums are of 32-bit values in
    any order: measured against 64 bits they are off by 1e-8 to 3e-7.  With int32 sums a block's
    64-bit sum that lies on the edge of a fixed-point unit (1e-3) may be truncated to either side.
    In a whole transformer a rounding can flip a comparison, which replaces a row in what follows."""
    kind = case["kind"]
    if kind == "int8":
        return "exact"
    if kind == "transformer":
        return {"rel": 1e-3, "max": 0.99}
    if case.get("summation") == "int32":
        return {"rel": 2e-6, "max": 1e-2}
    return {"rel": 2e-6, "max": 1e-4}


# ---------------------------------------------------------------------- the same results in 64 bits
def _lookup(d):
    """(row bits, margin of the anchor closest to flipping, its slot) from the fp32 anchor
    differences d [..., Nc]; the first of equal margins counts."""
    Nc = d.shape[-1]
    bits = (d > 0).long() << torch.arange(Nc, device=d.device)
    slot = d.abs().argmin(dim=-1, keepdim=True)
    return bits.sum(-1), d.gather(-1, slot).squeeze(-1), slot.squeeze(-1)


def _du(margin):
    """Derivative of the surrogate step at a margin: sign(u) * 0.5 / (1 + |u|)^2, sign(0) = -1."""
    m = margin.double()
    return torch.where(m > 0, 0.5, -0.5).double() / (1.0 + m.abs()) ** 2


def _payload(v):
    """Fixed-point value of a 64-bit sum, truncated as an int32 accumulator takes it."""
    return (v * DENOM * INT_RESCALER).trunc()


def _from_payload(v):
    return v / DENOM / INT_RESCALER


def _push(x_grad, du, pair):
    """x_grad[i, a] += du, x_grad[i, b] -= du for each row i of du [n, T] and its pairs [n, T, 2]."""
    x_grad.scatter_add_(1, pair[..., 0], du)
    x_grad.scatter_add_(1, pair[..., 1], -du)


def _exact_fc(x, g, anchors, tables, T, Nc, O, ints):
    """tables(t0, t1) gives rows [t1 - t0, E, O] in 64 bits."""
    B, E = x.shape[0], 1 << Nc
    a = anchors.long().view(T, Nc, 2)
    y = torch.zeros(B, O, dtype=torch.float64, device=x.device)
    result = {"y": y}
    if g is not None:
        g = g.double()
        x_grad = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
        w_grad = torch.zeros(T * E, O, dtype=torch.float64, device=x.device)
        pad = -O % GROUP
    # whole blocks of tables at a time, about 2 GB of rows
    step = max(GROUP, (1 << 27) // (B * O) // GROUP * GROUP)
    indices = []
    for t0 in range(0, T, step):
        t1 = min(T, t0 + step)
        w = tables(t0, t1)
        k, margin, slot = _lookup(x[:, a[t0:t1, :, 0]] - x[:, a[t0:t1, :, 1]])
        indices.append(k)
        t = torch.arange(t1 - t0, device=x.device)
        main = w[t[None], k]                                  # [B, n, O]
        if ints:
            blocks = [_payload(main[:, j:j + GROUP].sum(1)) for j in range(0, t1 - t0, GROUP)]
            y += torch.stack(blocks).sum(0)
        else:
            y += main.sum(1)
        if g is None:
            continue
        terms = (main - w[t[None], k ^ (1 << slot)]) * g[:, None]
        pair = a[t0:t1][t[None], slot]
        if ints:
            blocks = torch.nn.functional.pad(terms, (0, pad)).view(B, t1 - t0, -1, GROUP).sum(-1)
            _push(x_grad, _payload(_du(margin)[..., None] * blocks).sum(-1), pair)
        else:
            _push(x_grad, _du(margin) * terms.sum(-1), pair)
        del main, terms
        values = _payload(g) if ints else g
        for i in range(t1 - t0):
            w_grad.index_add_(0, (t0 + i) * E + k[:, i], values)
    if ints:
        result["y"] = _from_payload(y)
    if g is not None:
        result["x_grad"] = _from_payload(x_grad) if ints else x_grad
        result["w_grad"] = (_from_payload(w_grad) if ints else w_grad).view(-1)
    else:
        result["idx"] = torch.cat(indices, dim=1).to(torch.int32).view(-1)
    return result


def _exact_projection(layer, x, g):
    offsets, targets = (torch.as_tensor(v, device="cuda").long() for v in layer._lut_dm.lookup_connectivity())
    B, T, Nc = x.shape[0], layer._n_detectors, layer._n_anchors_per_detector
    w, xs = layer._weights.detach().double(), x.detach().view(B, -1)
    gs = g.double().view(B, -1)
    a = layer._detector_anchors.long().view(T, Nc, 2)
    k, margin, slot = _lookup(xs[:, a[..., 0]] - xs[:, a[..., 1]])
    first = torch.arange(T, device="cuda") * (1 << Nc)

    def synapses(row):
        """(synapse, sample, (sample, table) item) of every synapse of the items' rows."""
        row = (first + row).view(-1)
        length = offsets[row + 1] - offsets[row]
        item = torch.repeat_interleave(torch.arange(B * T, device="cuda"), length)
        start = length.cumsum(0) - length
        return offsets[row][item] + torch.arange(item.numel(), device="cuda") - start[item], item // T, item

    def dot(row):
        s, b, item = synapses(row)
        return torch.zeros(B * T, dtype=torch.float64, device="cuda").index_add_(0, item,
                                                                                   w[s] * gs[b, targets[s]])
    s, b, _ = synapses(k)
    y = torch.zeros(gs.numel(), dtype=torch.float64, device="cuda")
    y.index_add_(0, b * gs.shape[1] + targets[s], w[s])
    w_grad = torch.zeros_like(w).index_add_(0, s, gs[b, targets[s]])
    x_grad = torch.zeros(xs.shape, dtype=torch.float64, device="cuda")
    du = _du(margin) * (dot(k) - dot(k ^ (1 << slot))).view(B, T)
    _push(x_grad, du, a[torch.arange(T, device="cuda")[None], slot])
    return {"y": y.view(g.shape), "x_grad": x_grad.view(x.shape), "w_grad": w_grad}


def _exact_seq(x, g, anchors, w, pe, T, Nc, pd, O):
    """Causal pairs (i < j): row Q_j | K_i | P_(j - i - 1).  The backward flips the closer of the
    query and key margins, and the positional bit where it is closer than both."""
    B, S, I = x.shape
    a = anchors.long().view(T, Nc, 2)
    k, margin, slot = _lookup(x[..., a[..., 0]] - x[..., a[..., 1]])      # [B, S, T]
    w = w.view(T, -1, O)
    i, j = torch.triu_indices(S, S, 1, device=x.device)
    far = j - i - 1
    if pd:
        p, p_margin, p_slot = _lookup(pe.view(S - 1, T, pd))              # [S - 1, T]
    y = torch.zeros(B, S, O, dtype=torch.float64, device=x.device)
    result = {"y": y}
    if g is not None:
        g = g.double()
        x_grad = torch.zeros(B * S, I, dtype=torch.float64, device=x.device)
        w_grad = torch.zeros(w.shape, dtype=torch.float64, device=x.device)
        pe_grad = torch.zeros(S - 1, T, pd, dtype=torch.float64, device=x.device)
    at_b = torch.arange(B, device=x.device)[:, None] * S
    for t in range(T):
        q, key = k[:, j, t], k[:, i, t]                                   # [B, pairs]
        row = (q << (Nc + pd)) | (key << pd)
        if pd:
            row = row | p[far, t]
        table = w[t].double()
        # pairs of one sample at a time: [pairs, O] rows in 64 bits
        for b in range(B):
            main = table[row[b]]
            y[b].index_add_(0, j, main)
            if g is None:
                continue
            gj = g[b, j]
            w_grad[t].index_add_(0, row[b], gj)
            qm, km = margin[b, j, t], margin[b, i, t]
            flip_q = qm.abs() < km.abs()
            at_q, at_k = slot[b, j, t], slot[b, i, t]
            flipped = row[b] ^ torch.where(flip_q, 1 << (Nc + pd + at_q), 1 << (pd + at_k))
            du = _du(torch.where(flip_q, qm, km)) * ((main - table[flipped]) * gj).sum(-1)
            position = b * S + torch.where(flip_q, j, i)
            pair = a[t, torch.where(flip_q, at_q, at_k)]
            x_grad.view(-1).index_add_(0, position * I + pair[:, 0], du)
            x_grad.view(-1).index_add_(0, position * I + pair[:, 1], -du)
            if pd:
                m = p_margin[far, t]
                near = ((m.abs() < qm.abs()) & (m.abs() < km.abs())).nonzero().view(-1)
                bit = p_slot[far[near], t]
                moved = table[row[b, near] ^ (1 << bit)]
                dpe = _du(m[near]) * ((main[near] - moved) * gj[near]).sum(-1)
                pe_grad.view(-1).index_add_(0, (far[near] * T + t) * pd + bit, dpe)
    if g is not None:
        result.update(x_grad=x_grad.view(x.shape), w_grad=w_grad.view(-1))
        if pd:
            result["pe_grad"] = pe_grad.view(-1)
    return result


def _exact_product(x, g, anchors, w, pe, T, Nc, pd, O):
    """Every causal pair looks up the virtual row [x_i | x_j | pe_(j - i - 1)] of each table."""
    B, S, I = x.shape
    E = 1 << Nc
    a = anchors.long().view(T, Nc, 2)
    i, j = torch.triu_indices(S, S, 1, device=x.device)
    far = j - i - 1
    n = i.numel()
    flat_w, flat_g = w.view(T, E, O).double(), g.double().view(B * S, O)
    y = torch.zeros(B * S, O, dtype=torch.float64, device=x.device)
    w_grad = torch.zeros(T, E, O, dtype=torch.float64, device=x.device)
    x_grad = torch.zeros(B * S * I, dtype=torch.float64, device=x.device)
    pe_grad = torch.zeros((S - 1) * T * pd, dtype=torch.float64, device=x.device)
    at = (torch.arange(B, device=x.device)[:, None] * S + j).view(-1)     # row of j, per (sample, pair)

    def values(t, ids):
        """The virtual row's entries `ids` (Nc of them) of every pair: [B, pairs, Nc]."""
        cols = []
        for v in ids.tolist():
            if v < 2 * I:
                cols.append(x[:, i if v < I else j, v % I])
            else:
                cols.append(pe.view(S - 1, T, pd)[far, t, v - 2 * I].expand(B, n))
        return torch.stack(cols, dim=-1)

    def push(t, ids, du):
        """du of every (sample, pair) to its virtual-row entry `ids` [B, pairs]."""
        b = torch.arange(B, device=x.device)[:, None] * S
        inside = ids < 2 * I
        place = (b + torch.where(ids < I, i, j)) * I + ids % I
        x_grad.index_add_(0, place[inside], du[inside])
        if pd:
            place = ((far * T + t) * pd).expand(B, n) + ids - 2 * I
            pe_grad.index_add_(0, place[~inside], du[~inside])

    for t in range(T):
        k, margin, slot = _lookup(values(t, a[t, :, 0]) - values(t, a[t, :, 1]))
        counts = torch.zeros(B * S * E, dtype=torch.float64, device=x.device)
        counts.index_add_(0, at * E + k.view(-1), torch.ones(B * n, dtype=torch.float64, device=x.device))
        counts = counts.view(B * S, E)
        y += counts @ flat_w[t]
        w_grad[t] = counts.T @ flat_g
        dots = flat_g @ flat_w[t].T                                        # [B * S, E]
        flipped = (k ^ (1 << slot)).view(-1)
        du = _du(margin) * (dots[at, k.view(-1)] - dots[at, flipped]).view(B, n)
        push(t, a[t, slot, 0], du)
        push(t, a[t, slot, 1], -du)
    result = {"y": y.view(B, S, O), "x_grad": x_grad.view(x.shape), "w_grad": w_grad.view(-1)}
    if pd:
        result["pe_grad"] = pe_grad
    return result


def _exact_model(model, tokens):
    """The transformer's logits with its activations in 64 bits."""
    B, S = tokens.shape
    z = model.token_embedder.weight.detach().double()[tokens]

    def dense(layer, v):
        w = layer._weights.detach().view(layer._n_detectors, -1, layer._n_outputs)
        return _exact_fc(v, None, layer._detector_anchors, lambda t0, t1: w[t0:t1].double(),
                         layer._n_detectors, layer._n_anchors_per_detector, layer._n_outputs,
                         False)["y"]

    for block in model.layers:
        att = block["attention_lut"]
        z = z + _exact_seq(z, None, att._detector_anchors, att._weights.detach(),
                           att._positional_embeddings.detach(), att._n_detectors,
                           att._n_anchors_per_detector, att._positional_dim, att._n_outputs)["y"]
        z = z + dense(block["ffn"], z.reshape(B * S, -1)).view(B, S, -1)
    return dense(model.unembedder, z.reshape(B * S, -1)).view(B, S, -1)


@torch.no_grad()
def exact(case, seed):
    """What run() returns for prepare(case, seed), summed in 64 bits by plain torch.  Lookup bits and
    margins are fp32 differences of the fp32 inputs by definition; int32 sums are defined by their
    truncated block payloads."""
    state = prepare(case, seed)
    kind = case["kind"]
    if kind == "transformer":
        return {"y": _exact_model(state["model"], state["x"])}
    if kind == "int8":
        T, Nc, O = case["T"], case["Nc"], case["O"]
        q, scales = state["q"].view(T, 1 << Nc, O), state["scales"]
        # a table's entry is the fp32 product of its scale and its int8 value
        r = _exact_fc(state["x"].view(case["B"], -1), None, state["anchors"],
                      lambda t0, t1: (q[t0:t1].float() * scales[t0:t1, None, None]).double(), T, Nc, O,
                      True)
        return {"y": r["y"].view(-1), "idx": r["idx"]}
    layer, x, g = state["layer"], state["x"].detach(), state.get("g")
    if kind == "projection":
        return _exact_projection(layer, x, g)
    w = layer._weights.detach()
    if kind == "fc":
        T, Nc, O = case["T"], case["Nc"], case["O"]
        tables = w.view(T, 1 << Nc, O)
        r = _exact_fc(x.view(case["B"], -1), None if g is None else g.view(case["B"], -1),
                      layer._detector_anchors, lambda t0, t1: tables[t0:t1].double(), T, Nc, O,
                      case["summation"] == "int32")
        r["y"] = r["y"].view(case["B"], 1, O)
        if g is None:
            return {"y": r["y"]}
        r["x_grad"] = r["x_grad"].view(x.shape)
        if case["policy"] == "Sparse":
            r["w"] = w.double() - DESCENT * r.pop("w_grad")
        return r
    pe = layer._positional_embeddings
    pe = pe.detach() if pe is not None else None
    evaluate = _exact_seq if kind == "seq" else _exact_product
    return evaluate(x, g, layer._detector_anchors, w, pe, case["T"], case["Nc"], case["pd"], case["O"])
