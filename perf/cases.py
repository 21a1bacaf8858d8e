"""The framework's measured work: one pass each through its public entry
points, over the sizes, densities, data types and options it is used with.

A case is a dict of plain values; "kind" says which entry points a pass
goes through:

  step    FusedStep: the whole event path (extract, gather, scan, restore,
          forward and backward) with the workspace a training loop keeps
  api     the same path through the drop-in functions and autograd
  infer   the drop-in forward alone, without gradients
  scan    the flat selective scan with autograd, on event streams in hand
  conv    the depthwise causal convolution, forward and backward
  head    the block's spike head (prob_head, sigmoid, spikes), forward and
          backward
  block   the Mamba block behind its spike sampler, forward and backward,
          or forward alone
  model   a training step's forward and backward of the whole network

All inputs are made on the GPU from the seed alone.
"""
import math

import torch
import torch.nn.functional as F

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
THRESHOLD = 0.5
MOST_STEPS = 64 * 128 * 4000       # dense steps of the largest path case
MOST_UPDATES = 360_000_000         # (event, state) updates of the largest path case
MOST_TOKENS = 50 * 1024            # tokens of the largest block case


def listed():
    return [
        # the smallest training pass (config 0's sizes, 31 % events): launches and host calls are what counts
        dict(name="api_small", kind="api", B=2, D=64, L=1024, N=16, dtype="fp32", events="gauss", p=0.3085),
        # the headline training pass: a batch of medium sequences, i.i.d. events
        dict(name="step_train", kind="step", B=32, D=256, L=2048, N=16, dtype="fp32", events="bernoulli", p=0.15),
        # long byte sequences with 16-bit activations and fp32 state
        dict(name="step_long_bf16", kind="step", B=16, D=256, L=4096, N=16, dtype="bf16", events="bernoulli", p=0.10),
        # two towers of bursty, uneven streams with a large state, as a user of the drop-in functions trains them
        dict(name="api_bursty", kind="api", B=64, D=128, L=4000, N=64, dtype="fp32", events="markov", p=0.17),
        # one long sequence scored at a time: few channels with many events each
        dict(name="infer_one_long", kind="infer", B=1, D=512, L=4096, N=16, dtype="bf16", events="bernoulli", p=0.3),
        # the scan with B and C given per event and a z gate (not depthwise), channels of ragged length
        dict(name="scan_event_bc", kind="scan", mode="event", z=True, B=8, D=96, L=1500, N=16, dtype="fp32",
             events="markov", p=0.25),
        # the dense convolution on 16-bit activations of an odd length
        dict(name="conv_bf16", kind="conv", B=16, D=512, L=1023, K=4, dtype="bf16"),
        # the routing head over a batch of short-model tokens
        dict(name="head_train", kind="head", B=32, L=2000, d_model=128),
        # one small block in a test-sized training loop
        dict(name="block_small", kind="block", train=True, B=2, L=256, d_model=32, d_state=16, expand=2, p=0.3),
        # one layer of the six-layer model at its training batch
        dict(name="block_train", kind="block", train=True, B=50, L=1024, d_model=256, d_state=16, expand=2, p=0.3),
        # a few long sequences through one block in evaluation
        dict(name="block_eval", kind="block", train=False, B=4, L=4000, d_model=128, d_state=16, expand=2, p=0.3),
        # the whole network's training step: six layers, byte tokens
        dict(name="model_train", kind="model", B=50, L=1024, d_model=256, n_layers=6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "api", "api", "infer", "scan", "conv", "head", "block", "block", "model"])
    if kind in ("step", "api", "infer", "scan"):
        N = rng.choice([4, 8, 16, 16, 16, 16, 32, 64])
        D = _log(rng, 16, 512)
        L = _log(rng, 64, 8192)
        p = round(rng.uniform(0.03, 0.35), 3)
        most = min(MOST_STEPS, int(MOST_UPDATES / (p * N)))
        if kind == "scan":  # per-event B and C hold N values for each event
            most = min(most, int(32_000_000 / (p * N)))
        B = _log(rng, 1, max(1, min(64, most // (D * L))))
        while B * D * L > most:
            L = max(1, L // 2)
        case = dict(kind=kind, B=B, D=D, L=L, N=N, dtype=rng.choice(["fp32", "fp32", "bf16", "fp16"]),
                    events=rng.choice(["bernoulli", "bernoulli", "markov"]), p=p)
        if kind == "scan":
            case.update(mode=rng.choice(["event", "depthwise"]), z=rng.random() < 0.5)
        return case
    if kind == "conv":
        D, L = _log(rng, 32, 1024), _log(rng, 64, 8192)
        B = _log(rng, 1, max(1, min(64, (16 * 512 * 2048) // (D * L))))
        return dict(kind=kind, B=B, D=D, L=L, K=rng.choice([2, 3, 4, 4, 4]), dtype=rng.choice(["fp32", "bf16", "fp16"]))
    d_model = rng.choice([32, 48, 64, 96, 128, 128, 160, 192, 256, 256])
    L = _log(rng, 128, 4096)
    B = _log(rng, 1, max(1, min(64, MOST_TOKENS // L)))
    if kind == "head":
        return dict(kind=kind, B=B, L=L, d_model=d_model)
    if kind == "block":
        return dict(kind=kind, train=rng.random() < 0.6, B=B, L=L, d_model=d_model, d_state=rng.choice([8, 16, 16, 16, 32]),
                    expand=rng.choice([1, 2, 2]), p=round(rng.uniform(0.1, 0.35), 3))
    return dict(kind=kind, B=B, L=L, d_model=d_model, n_layers=rng.randint(2, 4))


# ------------------------------------------------------------------- inputs
def _gen(case, seed):
    return torch.Generator(device="cuda").manual_seed(1_000_003 * int(seed) + 17)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda")


def _membrane(case, g):
    """[B, D, L] float32 membrane: values above THRESHOLD are events."""
    B, D, L, p = case["B"], case["D"], case["L"], case["p"]
    if case["events"] == "gauss":
        return _randn(g, B, D, L)
    if case["events"] == "bernoulli":
        return (_rand(g, B, D, L) < p).float()
    # bursts: stay on with 0.9, stay off so that the on share is p; half of the channels are nearly silent
    off = 1.0 - 0.1 * p / (1.0 - p)
    u = _rand(g, L, B * D)
    on = _rand(g, B * D) < p
    ev = torch.empty(L, B * D, dtype=torch.bool, device="cuda")
    stay_on, stay_off = u < 0.9, u < off
    for t in range(L):
        on = torch.where(on, stay_on[t], ~stay_off[t])
        ev[t] = on
    ev = ev.t().contiguous()
    silent = torch.randperm(B * D, generator=g, device="cuda")[:B * D // 2]
    ev[silent] = _rand(g, silent.numel(), L) < 0.015
    return ev.view(B, D, L).float()


def _expected_events(case):
    share = case["p"] if case["events"] != "markov" else 0.5 * (case["p"] + 0.015)
    return max(1, round(case["B"] * case["D"] * case["L"] * share))


def _with_count(membrane, E, g):
    """The membrane with random events added or taken away until it holds E."""
    flat = membrane.view(-1)
    now = flat > THRESHOLD
    over = int(now.sum()) - E
    pool = (now if over > 0 else ~now).nonzero(as_tuple=True)[0]
    pick = pool[torch.randperm(pool.numel(), generator=g, device="cuda")[:abs(over)]]
    flat[pick] = 0.0 if over > 0 else 1.0
    return membrane


def _params(g, D, N):
    """dt_idle, dt_active, A, W_B, W_C and the skip weights of D model channels."""
    return [F.softplus(_randn(g, D) - 2.0), F.softplus(_randn(g, D) - 2.0),
            -torch.exp(_rand(g, D, N) * math.log(16.0)),
            _randn(g, D, N) / math.sqrt(N), _randn(g, D, N) / math.sqrt(N), 1.0 + 0.1 * _randn(g, D)]


def _path_inputs(case, seed):
    g = _gen(case, seed)
    dt = DTYPES[case["dtype"]]
    membrane = _membrane(case, g)
    x = _randn(g, case["B"], case["D"], case["L"]).to(dt)
    params = _params(g, case["D"], case["N"])
    dout = _randn(g, case["B"], case["L"], case["D"]).to(dt)
    return membrane, x, params, dout


def _events(membrane):
    """(channel, step, gap, offsets) of a membrane's events, in plain torch."""
    rows = membrane.reshape(-1, membrane.size(-1)) > THRESHOLD
    ch, t = rows.nonzero(as_tuple=True)
    cu = torch.zeros(rows.size(0) + 1, dtype=torch.int64, device="cuda")
    cu[1:] = torch.cumsum(rows.sum(1), 0)
    k = t + 1
    k[1:] = torch.where(ch[1:] == ch[:-1], t[1:] - t[:-1], k[1:])
    return ch, t, k, cu


def _scan_inputs(case, seed):
    """The event streams of a scan call: u, k, offsets, parameters, B, C, z and the output's gradient."""
    g = _gen(case, seed)
    dt = DTYPES[case["dtype"]]
    ch, _, k, cu = _events(_with_count(_membrane(case, g), _expected_events(case), g))
    E, N = ch.numel(), case["N"]
    params = _params(g, case["D"], N)
    if case["mode"] == "event":
        bc = [_randn(g, N, E), _randn(g, N, E)]
    else:
        bc = params[3:5]
    z = _randn(g, E).to(dt) if case["z"] else None
    return dict(ch=ch, k=k, cu=cu, u=_randn(g, E).to(dt), params=params[:3], bc=bc, skip=params[5], z=z,
                dout=_randn(g, E).to(dt))


def _block_weights(case, g):
    """A block's state dict, as the block initialises itself."""
    d, N, di = case["d_model"], case["d_state"], case["d_model"] * case["expand"]

    def linear(o, i):
        return (2.0 * _rand(g, o, i) - 1.0) / math.sqrt(i)

    def level():
        dt = torch.exp(_rand(g, di) * math.log(100.0) + math.log(0.001))
        return torch.log(torch.expm1(dt))

    return {
        "W_BC": 0.02 * _randn(g, di, 2 * N), "D": torch.ones(di, device="cuda"),
        "A_log": torch.log(torch.arange(1, N + 1, dtype=torch.float32, device="cuda")).repeat(di, 1),
        "in_proj.weight": linear(di, d), "conv1d.weight": _rand(g, di, 1, 4) - 0.5, "conv1d.bias": _rand(g, di) - 0.5,
        "out_proj.weight": linear(d, di), "prob_head.weight": linear(d, d),
        "prob_head.bias": torch.full((d,), math.log(0.3 / 0.7), device="cuda"),
        "delta_gen.a0": level(), "delta_gen.a1": level(),
    }


def _block_inputs(case, seed):
    """Weights, spike probabilities of which a share p reaches the threshold, and the output's gradient."""
    g = _gen(case, seed)
    w = _block_weights(case, g)
    shape = (case["B"], case["L"], case["d_model"])
    shift = math.sqrt(2.0) * torch.erfinv(torch.tensor(2.0 * case["p"] - 1.0)).item()
    return w, torch.sigmoid(_randn(g, *shape) + shift), _randn(g, *shape)


def _head_inputs(case, seed):
    g = _gen(case, seed)
    w = _block_weights(dict(case, d_state=16, expand=1), g)
    shape = (case["B"], case["L"], case["d_model"])
    return w, _randn(g, *shape), _randn(g, *shape)


def _conv_inputs(case, seed):
    g = _gen(case, seed)
    dt = DTYPES[case["dtype"]]
    shape = (case["B"], case["D"], case["L"])
    return (_randn(g, *shape).to(dt), _rand(g, case["D"], case["K"]) - 0.5, _rand(g, case["D"]) - 0.5,
            _randn(g, *shape).to(dt))


def _block(case, w):
    from bc_mamba_amd.e_model import Mamba
    blk = Mamba(d_model=case["d_model"], d_state=case.get("d_state", 16), expand=case.get("expand", 1),
                threshold=THRESHOLD, device="cuda")
    blk.load_state_dict(w)
    return blk


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        from bc_mamba_amd.fused_step import FusedStep
        from bc_mamba_amd.workloads import Workload
        membrane, x, params, dout = _path_inputs(case, seed)
        w = Workload(0, case["B"], case["D"], case["L"], case["N"], x.dtype, THRESHOLD, membrane, x, *params, dout)
        return dict(kind=kind, step=FusedStep(w, torch.device("cuda", torch.cuda.current_device()), keep_du=False))
    if kind in ("api", "infer"):
        membrane, x, params, dout = _path_inputs(case, seed)
        if kind == "api":
            x.requires_grad_(True)
            params = [q.requires_grad_(True) for q in params]
        return dict(kind=kind, D=case["D"], L=case["L"], membrane=membrane, x=x, params=params, dout=dout)
    if kind == "scan":
        s = _scan_inputs(case, seed)
        grads = [s["u"], *s["params"], *s["bc"], s["skip"]] + ([s["z"]] if case["z"] else [])
        for v in grads:
            v.requires_grad_(True)
        ms = int((s["cu"][1:] - s["cu"][:-1]).max())
        return dict(s, kind=kind, k=s["k"].int(), cu=s["cu"].int(), ms=ms, grads=grads, depthwise=case["mode"] == "depthwise")
    if kind == "conv":
        x, w, b, dout = _conv_inputs(case, seed)
        return dict(kind=kind, leaves=[v.requires_grad_(True) for v in (x, w, b)], dout=dout)
    if kind == "head":
        w, v, dout = _head_inputs(case, seed)
        return dict(kind=kind, block=_block(case, w), v=v.requires_grad_(True), dout=dout)
    if kind == "block":
        w, prob, dout = _block_inputs(case, seed)
        return dict(kind=kind, block=_block(case, w), prob=prob.requires_grad_(case["train"]), dout=dout,
                    train=case["train"])
    from bc_mamba_amd.workloads import make_model_workload
    net, tokens, labels = make_model_workload(seed, B=case["B"], L=case["L"], device="cuda", d_model=case["d_model"],
                                              n_layers=case["n_layers"])
    # the data-parallel buckets of such a step: one flat gradient for each layer, and one for the rest
    named = [(n, q) for n, q in net.named_parameters() if q.requires_grad]
    buckets = {}
    for n, _ in named:
        buckets.setdefault(n.split(".")[1] if n.startswith("blocks.") else "rest", []).append(n)
    return dict(kind=kind, net=net, tokens=tokens, labels=labels, named=named, buckets=buckets)


# -------------------------------------------------------------------- passes
def _api_forward(s):
    from bc_mamba_amd import extract_events_cuda, selective_scan_interface
    from bc_mamba_amd.e_model import GatherEventsFn, restore_dense_fn
    ch, t, k, cu, _, ms = extract_events_cuda.extract_base_events(s["membrane"], THRESHOLD)
    u = GatherEventsFn.apply(s["x"], ch, t)
    dt_idle, dt_active, A, W_B, W_C, skip = s["params"]
    y, _ = selective_scan_interface.selective_scan_flat_ch_fn(u, k, cu, int(ms), dt_idle, dt_active, A, W_B, W_C,
                                                              D=skip, is_depthwise_bc=True)
    return restore_dense_fn(y, t, cu, s["D"], s["L"]), cu


def run(state):
    kind = state["kind"]
    if kind == "step":
        st = state["step"]
        st.step()
        return dict(out=st.dense, dx=st.dx, grads=st.grads, offsets=st.cu)
    if kind == "api":
        out, cu = _api_forward(state)
        grads = torch.autograd.grad(out, [state["x"], *state["params"]], state["dout"])
        return dict(out=out.detach(), dx=grads[0], grads=list(grads[1:]), offsets=cu)
    if kind == "infer":
        with torch.no_grad():
            out, cu = _api_forward(state)
        return dict(out=out, offsets=cu)
    if kind == "scan":
        from bc_mamba_amd.selective_scan_interface import selective_scan_flat_ch_fn
        out, x = selective_scan_flat_ch_fn(state["u"], state["k"], state["cu"], state["ms"], *state["params"],
                                           *state["bc"], D=state["skip"], z=state["z"],
                                           is_depthwise_bc=state["depthwise"])
        return dict(out=out.detach(), grads=list(torch.autograd.grad(out, state["grads"], state["dout"])))
    if kind == "conv":
        from bc_mamba_amd.causal_conv1d import causal_conv1d_fn
        x, w, b = state["leaves"]
        out = causal_conv1d_fn(x, w, b, activation="silu")
        return dict(out=out.detach(), grads=list(torch.autograd.grad(out, [x, w, b], state["dout"])))
    if kind == "head":
        blk = state["block"]
        s = blk.to_spike(state["v"])
        grads = torch.autograd.grad(s, [state["v"], blk.prob_head.weight, blk.prob_head.bias], state["dout"])
        return dict(events=s.detach() > THRESHOLD, grads=list(grads))
    if kind == "block":
        blk = state["block"]
        if not state["train"]:
            with torch.no_grad():
                return dict(out=blk(blk.spike_sampler(state["prob"])))
        out = blk(blk.spike_sampler(state["prob"]))
        named = [(n, q) for n, q in blk.named_parameters() if not n.startswith("prob_head")]
        grads = torch.autograd.grad(out, [state["prob"], *(q for _, q in named)], state["dout"])
        return dict(out=out.detach(), dprob=grads[0], grads={n: v for (n, _), v in zip(named, grads[1:])})
    logits = state["net"](state["tokens"])
    loss = F.cross_entropy(logits, state["labels"])
    names = [n for n, _ in state["named"]]
    grads = dict(zip(names, torch.autograd.grad(loss, [q for _, q in state["named"]])))
    flat = {b: torch.cat([grads[n].reshape(-1) for n in ns]) for b, ns in state["buckets"].items()}
    return dict(logits=logits.detach(), loss=loss.detach(), grads=flat)


# ---------------------------------------------------------- what a pass needs
def work(case):
    kind = case["kind"]
    if kind in ("step", "api", "infer", "scan"):
        size = {"fp32": 4, "bf16": 2, "fp16": 2}[case["dtype"]]
        M = case["B"] * case["D"] * case["L"]
        E, N = _expected_events(case), case["N"]
        if kind == "scan":
            per_event = 4 + size * (5 + (2 if case["z"] else 0)) + (16 * N if case["mode"] == "event" else 0)
            return dict(bytes=E * per_event, flops=E * N * 24)
        if kind == "infer":
            return dict(bytes=M * (4 + 2 * size), flops=E * N * 7)
        return dict(bytes=M * (4 + 4 * size), flops=E * N * 24)
    if kind == "conv":
        M = case["B"] * case["D"] * case["L"]
        return dict(bytes=M * 4 * (4 if case["dtype"] == "fp32" else 2), flops=M * (6 * case["K"] + 20))
    tokens, d = case["B"] * case["L"], case["d_model"]
    head = dict(bytes=tokens * d * 16 + 3 * d * d * 4, flops=6 * tokens * d * d)
    if kind == "head":
        return head
    expand, N = case.get("expand", 2), case.get("d_state", 16)
    di, p = d * expand, case.get("p", 0.3)
    train = case.get("train", True)
    block = dict(bytes=tokens * d * (16 if train else 8) + 2 * d * di * (8 if train else 4),
                 flops=(3 if train else 1) * 4 * tokens * d * di + tokens * di * p * N * (24 if train else 7))
    if kind == "block":
        return block
    n = case["n_layers"]
    return dict(bytes=tokens * 8 + n * (2 * d * di + d * d) * 8,
                flops=n * block["flops"] + (n + 1) * head["flops"])


def tolerance(case):
    """About four times the largest error against exact() (for the whole
    network: against the same network with its sums in another order) seen
    over the listed and drawn cases."""
    kind = case["kind"]
    if kind == "model":
        # a spike whose probability lies within rounding of the threshold may turn, and travels on: 2.8e-3 seen
        return {"rel": 1.2e-2, "max": 0.7}
    if kind == "head":
        return {"rel": 6e-6, "max": 4e-5, "differ": 4e-6}
    if kind == "block":
        return {"rel": 6e-6, "max": 6e-5}
    if case["dtype"] == "fp32":
        return {"rel": 4e-6, "max": 4e-4}
    if case["dtype"] == "fp16":
        return {"rel": 1.2e-3, "max": 1.2e-2}
    return {"rel": 1e-2, "max": 0.1}


# ---------------------------------------------------------------- in 64 bits
def _d(v):
    return v.detach().double().requires_grad_(True)


def _scan64(u, ch, k, cu, dim, dt_idle, dt_active, A, skip, B, C, per_event=False):
    """y of every event: the recurrence event by event over all channels at
    once. B, C: the [dim, N] weights (B_i = u_i W_B, C_i = u_i W_C), or
    [N, E] values per event."""
    NC, E = cu.numel() - 1, u.numel()
    pos = torch.arange(E, device="cuda") - cu[ch]
    steps = int((cu[1:] - cu[:-1]).max())
    order = torch.argsort(cu[1:] - cu[:-1], descending=True, stable=True)  # the channels that still run come first
    rank = torch.empty_like(order)
    rank[order] = torch.arange(NC, device="cuda")
    alive = (pos.bincount(minlength=steps)).tolist()
    at = torch.zeros(steps + 1, dtype=torch.int64, device="cuda")
    at[1:] = torch.cumsum(pos.bincount(minlength=steps), 0)
    slot = at[pos] + rank[ch]  # events by position, within one by rank
    place = torch.empty_like(slot)
    place[slot] = torch.arange(E, device="cuda")
    dch = ch[place] % dim
    us = u[place]
    delta = dt_active[dch] + dt_idle[dch] * (k[place] - 1)
    if per_event:
        Bs, Cs = B.t()[place], C.t()[place]
    h, ys, o = None, [], 0
    for n in alive:
        if n == 0:
            break
        c = slice(o, o + n)
        a = torch.exp2(torch.clamp(delta[c, None] * A[dch[c]] * math.log2(math.e), -126.0, 126.0))
        if per_event:
            b, w = us[c, None] * Bs[c], Cs[c]
        else:
            b, w = us[c, None].square() * B[dch[c]], us[c, None] * C[dch[c]]
        inc = delta[c, None] * b
        h = inc if h is None else a * h[:n] + inc
        ys.append((h * w).sum(1))
        o += n
    y = torch.cat(ys)[slot] if ys else us
    return y + skip[ch % dim] * u


def _path64(membrane, x, params):
    """Extraction, gather, scan and restore in 64 bits: [B, L, D]."""
    B, D, L = membrane.shape
    ch, t, k, cu = _events(membrane)
    if ch.numel() == 0:
        return (x * 0).transpose(1, 2) + sum(q.sum() * 0 for q in params)
    dt_idle, dt_active, A, W_B, W_C, skip = params
    y = _scan64(x.reshape(B * D, L)[ch, t], ch, k, cu, D, dt_idle, dt_active, A, skip, W_B, W_C)
    rows = membrane.reshape(B * D, L) > THRESHOLD
    seen = torch.cumsum(rows, 1)
    held = y.gather(0, (cu[:-1, None] + seen - 1).clamp(min=0).view(-1)).view(B * D, L)
    return torch.where(seen > 0, held, 0.0).view(B, D, L).transpose(1, 2)


def _conv64(x, w, b):
    K, L = w.size(1), x.size(2)
    padded = F.pad(x, (K - 1, 0))
    pre = b[:, None] + sum(w[:, i, None] * padded[..., i:i + L] for i in range(K))
    return pre * torch.sigmoid(pre)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "api", "infer"):
        membrane, x, params, dout = _path_inputs(case, seed)
        if kind == "infer":
            with torch.no_grad():
                return dict(out=_path64(membrane, x.double(), [q.double() for q in params]), offsets=None)
        x, params = _d(x), [_d(q) for q in params]
        out = _path64(membrane, x, params)
        gx, gi, ga, gA, gB, gC, gD = torch.autograd.grad(out, [x, *params], dout.double())
        if kind == "step":  # FusedStep's order
            return dict(out=out.detach(), dx=gx, grads=[gA, gB, gC, gi, ga, gD], offsets=None)
        return dict(out=out.detach(), dx=gx, grads=[gi, ga, gA, gB, gC, gD], offsets=None)
    if kind == "scan":
        s = _scan_inputs(case, seed)
        leaves = [_d(v) for v in [s["u"], *s["params"], *s["bc"], s["skip"]] + ([s["z"]] if case["z"] else [])]
        u, dt_idle, dt_active, A, B, C, skip = leaves[:7]
        out = _scan64(u, s["ch"], s["k"], s["cu"], case["D"], dt_idle, dt_active, A, skip, B, C,
                      per_event=case["mode"] == "event")
        if case["z"]:
            out = out * F.silu(leaves[7])
        return dict(out=out.detach(), grads=list(torch.autograd.grad(out, leaves, s["dout"].double())))
    if kind == "conv":
        x, w, b, dout = _conv_inputs(case, seed)
        x, w, b = _d(x), _d(w), _d(b)
        out = _conv64(x, w, b)
        return dict(out=out.detach(), grads=list(torch.autograd.grad(out, [x, w, b], dout.double())))
    if kind == "head":
        w, v, dout = _head_inputs(case, seed)
        v, W, b = _d(v), _d(w["prob_head.weight"]), _d(w["prob_head.bias"])
        prob = torch.sigmoid(v @ W.t() + b)  # the spikes pass its gradient on
        return dict(events=None, grads=list(torch.autograd.grad(prob, [v, W, b], dout.double())))
    if kind == "block":
        w, prob, dout = _block_inputs(case, seed)
        N = case["d_state"]
        with torch.set_grad_enabled(case["train"]):
            prob = _d(prob)
            q = {n: _d(v) for n, v in w.items()}
            hard = (prob >= THRESHOLD).double()
            s = hard + prob - prob.detach()
            x = torch.matmul(s, q["in_proj.weight"].t()).transpose(1, 2)
            x = _conv64(x, q["conv1d.weight"][:, 0], q["conv1d.bias"])
            params = [F.softplus(q["delta_gen.a0"]) + 1e-6, F.softplus(q["delta_gen.a1"]) + 1e-6,
                      -torch.exp(q["A_log"]), q["W_BC"][:, :N], q["W_BC"][:, N:], q["D"]]
            fired = hard.transpose(1, 2).repeat_interleave(case["expand"], dim=1)
            out = torch.matmul(_path64(fired, x, params), q["out_proj.weight"].t())
        if not case["train"]:
            return dict(out=out)
        names = [n for n in w if not n.startswith("prob_head")]
        grads = torch.autograd.grad(out, [prob, *(q[n] for n in names)], dout.double())
        return dict(out=out.detach(), dprob=grads[0], grads=dict(zip(names, grads[1:])))
    return None  # the whole network: a spike at the threshold within rounding may turn, so no one value is right
