"""The work a program has this framework do, as cases that can be timed and checked.

Three kinds of call, each through the framework's public entry points:

* "step": a token step of a serving loop on `HybridRuntime` -- `forward_batch`
  over `seqs` sequences of about `length` cached positions (rows == 1), or the
  verify forward of one sequence's `rows` speculated rows. `attn` full-attention
  and `gdn` Gated DeltaNet layers, every fourth one attention as in the model
  (64 layers: 16 and 48; fewer here, the layers of a step being alike). With
  `graph` the program replays a captured step, as the benchmark's serving lines
  do, else it calls the runtime eagerly.
* "attention": one layer's gated causal prefill attention of `tokens` queries at
  position `pos` over its KV cache (`attention_prefill` / `attention_prefill_q8`).
* "prompt": a new prompt of `tokens` tokens through `HybridRuntime.forward` in
  sub-chunks of `chunk` tokens (the backend's MAX_CHUNK is 1024), state made and
  caches grown as the backend does.

The projections between the layers lie outside the framework: `Given` hands each
layer its rows and keeps the layers' outputs. A step is taken at the same
position on every pass (its token is dropped again afterwards), so that a pass
costs the same however many came before. The attention prep normalises and
rotates the projected q and k rows in place, so later passes start from rows
already normalised once: their scale, and with it the softmax, stays the same.
"""
import math

import torch

from __graft_entry__ import load_package

HEADS, KV, DIM = 24, 4, 256              # attention: q heads, kv heads, head dim
ROPE, THETA = 64, 1e7
K_HEADS, V_HEADS, GD = 16, 48, 128       # Gated DeltaNet: k heads, v heads, head dim
ROW = 2 * K_HEADS * GD + V_HEADS * GD    # the q|k|v row: 10240
EPS = 1e-6


def listed():
    return [
        # the smallest call: one user's next token in a short chat, nothing batched
        dict(name="decode_1x4k_kv8", kind="step", seqs=1, length=4096, rows=1, attn=4, gdn=12,
             kv8=True, graph=False),
        # the serving loop's ordinary step: the backend's largest batch over the shipped int8 cache
        dict(name="decode_4x8k_kv8_graph", kind="step", seqs=4, length=8192, rows=1, attn=4, gdn=12,
             kv8=True, graph=True),
        # long documents, fp16 cache
        dict(name="decode_4x100k", kind="step", seqs=4, length=100000, rows=1, attn=1, gdn=3,
             kv8=False, graph=False),
        # an odd batch of middling contexts over the int8 cache
        dict(name="decode_3x33k_kv8_graph", kind="step", seqs=3, length=33333, rows=1, attn=2, gdn=6,
             kv8=True, graph=True),
        # the speculative round of one sequence: three rows, checkpoints kept
        dict(name="verify_3rows_32k_kv8_graph", kind="step", seqs=1, length=32768, rows=3, attn=4,
             gdn=12, kv8=True, graph=True),
        # the model's 48 recurrent layers of a batched decode step
        dict(name="gdn_decode_4x48_graph", kind="step", seqs=4, length=512, rows=1, attn=0, gdn=48,
             kv8=False, graph=True),
        # a fresh 8k prompt's attention in one call
        dict(name="attention_8k", kind="attention", tokens=8192, pos=0, kv8=False),
        # the sub-chunk of a long prompt: 1024 tokens, 30k deep, int8 cache
        dict(name="attention_1k_at_30k_kv8", kind="attention", tokens=1024, pos=30720, kv8=True),
        # the same, 98k deep, fp16 cache: the largest
        dict(name="attention_1k_at_98k", kind="attention", tokens=1024, pos=98000, kv8=False),
        # a follow-up message of odd length behind a cached conversation
        dict(name="attention_777_at_3001", kind="attention", tokens=777, pos=3001, kv8=False),
        # a short chat prompt, odd length, int8 cache: one sub-chunk through a block of four layers
        dict(name="prompt_1000_kv8", kind="prompt", tokens=1000, chunk=1024, attn=1, gdn=3, kv8=True),
        # a long prompt in the backend's sub-chunks through a block of four layers
        dict(name="prompt_8k", kind="prompt", tokens=8192, chunk=1024, attn=1, gdn=3, kv8=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "attention", "prompt"])
    kv8 = rng.random() < 0.5
    if kind == "step":
        rows = rng.choice([1, 1, 1, 2, 3])
        seqs = 1 if rows > 1 else rng.randint(1, 6)
        length = _log(rng, 300, 100000)
        attn = rng.randint(1, 4) if seqs * length < 100000 else 1
        return dict(kind=kind, seqs=seqs, length=length, rows=rows, attn=attn,
                    gdn=3 * attn, kv8=kv8, graph=rng.random() < 0.5)
    if kind == "prompt":
        return dict(kind=kind, tokens=_log(rng, 65, 8000), chunk=1024, attn=1, gdn=3, kv8=kv8)
    tokens = _log(rng, 33, 8192)
    # int8 prompts of the benchmark end at 32k; no more query-key pairs than 1024 x 98k
    deepest = min(32768 - tokens if kv8 else 98000, int(1.0e8 / tokens - tokens / 2))
    pos = _log(rng, 1, deepest + 1) - 1 if deepest > 0 else 0
    return dict(kind=kind, tokens=tokens, pos=pos, kv8=kv8)


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 11)


def _randn(g, *shape, scale=1.0, dtype=torch.float32):
    x = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, scale, generator=g)
    return x if dtype == torch.float32 else x.to(dtype)


def _quantise(x):
    """fp16 rows [n, KV, DIM] in the int8 format: bytes [n, KV, DIM] and fp16
    scales [n, KV, DIM / 32] (absmax / 127 of 32 dims, values rint(x / scale))."""
    b = x.float().view(*x.shape[:-1], DIM // 32, 32)
    s = (b.abs().amax(-1) / 127.0).half()
    q = torch.where(s[..., None] > 0, torch.round(b / s.float()[..., None]).clamp(-127, 127),
                    torch.zeros_like(b))
    return q.to(torch.int8).view(x.shape), s


def _rows8(values, scales):
    return (values.double().view(*values.shape[:-1], DIM // 32, 32)
            * scales.double()[..., None]).view(values.shape)


def _types(case):
    n = case["attn"] + case["gdn"]
    if case["attn"] == 0:
        return ("linear_attention",) * n
    return tuple("full_attention" if (i + 1) % 4 == 0 else "linear_attention" for i in range(n))


def _weights(g, types):
    """Per layer: the norm gammas of q and k, or the conv taps, A_log, dt_bias
    and the output norm's gamma."""
    out = []
    for t in types:
        if t == "full_attention":
            out.append((_randn(g, DIM, scale=0.1), _randn(g, DIM, scale=0.1)))
        else:
            out.append((_randn(g, ROW, 4, scale=0.5, dtype=torch.float16),
                        _randn(g, V_HEADS, scale=0.3), _randn(g, V_HEADS, scale=0.3),
                        1 + _randn(g, GD, scale=0.2)))
    return out


def _projected(g, n, attention=True):
    f16 = torch.float16
    p = dict(qkv=_randn(g, n, ROW, dtype=f16), z=_randn(g, n, V_HEADS, GD, dtype=f16),
             a=_randn(g, n, V_HEADS), b=_randn(g, n, V_HEADS))
    if attention:
        p.update(qg=_randn(g, n, HEADS, 2 * DIM, dtype=f16), k=_randn(g, n, KV, DIM, dtype=f16),
                 v=_randn(g, n, KV, DIM, dtype=f16))
    return p


def _lengths(case):
    """The sequences of a batch differ in length."""
    return [max(2, case["length"] - (case["length"] // 29) * b) for b in range(case["seqs"])]


def _cached(g, n, kv8):
    """n cached positions of one layer's K or V."""
    x = _randn(g, n, KV, DIM, dtype=torch.float16)
    return _quantise(x) if kv8 else x


class Given:
    """The projections a step or prompt hands to the layers; keeps what the layers return."""

    def __init__(self, rows):
        self.rows, self.at, self.out = rows, 0, []

    def full_attn_in(self, layer, T):
        r, s = self.rows, slice(self.at, self.at + T)
        return r["qg"][s], r["k"][s], r["v"][s]

    def gdn_in(self, layer, T):
        r, s = self.rows, slice(self.at, self.at + T)
        return r["qkv"][s], r["z"][s], r["a"][s], r["b"][s]

    def layer_out(self, layer, out):
        self.out.append(out)


def _runtime(case, weights):
    fl = load_package()
    types = _types(case)
    own = {i: fl.runtime.FullWeights(*w) if t == "full_attention" else fl.runtime.GdnWeights(*w)
           for i, (t, w) in enumerate(zip(types, weights))}
    return fl.runtime.HybridRuntime(own, layer_types=types, kv8=case["kv8"])


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------

def _step_inputs(case, seed):
    """(weights, projected rows, recurrent states, conv rings, caches): the
    caches as [sequence][layer] -> (K, V) of the sequence's cached positions."""
    g = _gen(seed)
    types = _types(case)
    n = case["seqs"] * case["rows"]
    weights = _weights(g, types)
    rows = _projected(g, n, case["attn"] > 0)
    S = [_randn(g, case["gdn"], V_HEADS, GD, GD, scale=0.02) for _ in range(case["seqs"])]
    rings = [_randn(g, case["gdn"], ROW, 3, dtype=torch.float16) for _ in range(case["seqs"])]
    caches = [[(_cached(g, n_pos, case["kv8"]), _cached(g, n_pos, case["kv8"]))
               for _ in range(case["attn"])] for n_pos in _lengths(case)]
    return weights, rows, S, rings, caches


def _put(buf, cap, rows, kv8):
    """Cached positions into a layer's buffer."""
    if not kv8:
        buf[:rows.shape[0]].copy_(rows)
        return
    values, scales = rows
    n = values.numel()
    buf[:n].copy_(values.view(-1))
    at = cap * KV * DIM
    buf[at:at + 2 * scales.numel()].copy_(scales.contiguous().view(-1).view(torch.int8))


def _prepare_step(case, seed):
    weights, rows, S, rings, caches = _step_inputs(case, seed)
    rt = _runtime(case, weights)
    states = []
    for b, n_pos in enumerate(_lengths(case)):
        st = rt.new_state()
        rt.grow(st, n_pos + 16)
        st.tokens = list(range(n_pos))
        st.fed = n_pos
        for layer, (k, v) in enumerate(caches[b]):
            _put(st.kk[layer], st.lcap[layer], k, case["kv8"])
            _put(st.kv[layer], st.lcap[layer], v, case["kv8"])
        states.append(st)
    state = dict(rt=rt, states=states, given=Given(rows), case=case, graph=None)
    if case["graph"]:
        kept = {k: v.clone() for k, v in rows.items()}
        _step(state)                       # once as it is, then captured
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        for st in states:
            st.phase = 0
        with torch.cuda.graph(graph):
            state["outputs"] = _step(state)
        state["graph"] = graph
        for k, v in kept.items():
            rows[k].copy_(v)
    for st, s, ring in zip(states, S, rings):
        st.phase = 0
        st.s.copy_(s)
        st.conv.zero_()
        st.conv[0].copy_(ring)
    return state


def _step(state):
    """One step eagerly, its token dropped again (a verify keeps none by itself)."""
    case, rt, states, given = state["case"], state["rt"], state["states"], state["given"]
    given.out = []
    if case["rows"] > 1:
        rt.forward(states[0], given, range(case["rows"]), verify=True)
        more = [rt.snap_s[:case["rows"] - 1]] + ([rt.snap_c] if case["rows"] == 3 else [])
    else:
        rt.forward_batch(states, given, [1] * len(states))
        for st in states:
            st.tokens.pop()
        more = []
    kv = [b for st in states for b in (st.kk or [])[:2] + (st.kv or [])[:2]]
    if len(given.out) + len(more) + len(kv) + 2 * len(states) > 64:
        kv = []
    return dict(layers=given.out, s=[st.s for st in states], conv=[st.conv for st in states],
                checkpoints=more, kv=kv)


def _attention_inputs(case, seed):
    g = _gen(seed)
    T, n = case["tokens"], case["pos"] + case["tokens"]
    qg = _randn(g, T, HEADS, 2 * DIM, dtype=torch.float16)
    return qg, _cached(g, n, case["kv8"]), _cached(g, n, case["kv8"])


def _prepare_attention(case, seed):
    qg, k, v = _attention_inputs(case, seed)
    fl = load_package()
    n = case["pos"] + case["tokens"]
    if case["kv8"]:
        kc, vc = fl.ops.kv8_cache(n), fl.ops.kv8_cache(n)
        _put(kc, n, k, True)
        _put(vc, n, v, True)
    else:
        kc, vc = k, v
    return dict(ops=fl.ops, qg=qg, kc=kc, vc=vc, case=case, n=n)


def _prompt_inputs(case, seed):
    g = _gen(seed)
    weights = _weights(g, _types(case))
    return weights, _projected(g, case["tokens"])


def prepare(case, seed):
    if case["kind"] == "step":
        return _prepare_step(case, seed)
    if case["kind"] == "attention":
        return _prepare_attention(case, seed)
    weights, rows = _prompt_inputs(case, seed)
    return dict(rt=_runtime(case, weights), given=Given(rows), case=case)


def run(state):
    case = state["case"]
    if case["kind"] == "step":
        if state["graph"] is not None:
            state["graph"].replay()
            return state["outputs"]
        return _step(state)
    if case["kind"] == "attention":
        ops = state["ops"]
        if case["kv8"]:
            return ops.attention_prefill_q8(state["qg"], state["kc"], state["vc"], pos0=case["pos"],
                                            max_pos=state["n"], gated=True)
        return ops.attention_prefill(state["qg"], state["kc"], state["vc"], pos0=case["pos"],
                                     gated=True)
    rt, given = state["rt"], state["given"]
    given.out = []
    st = rt.new_state()
    for p in range(0, case["tokens"], case["chunk"]):
        given.at = p
        rt.forward(st, given, range(p, min(p + case["chunk"], case["tokens"])))
    return dict(layers=given.out, s=st.s, conv=st.conv[st.phase], kv=[st.kk[0], st.kv[0]])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _attention_work(tokens, pos, kv8):
    row = KV * (DIM + 16 if kv8 else 2 * DIM)
    nbytes = 2 * (pos + tokens) * row + tokens * HEADS * DIM * 2 * 3     # K, V; q, gate, z
    return nbytes, 4 * HEADS * DIM * (tokens * pos + tokens * (tokens + 1) / 2)


def _prep_bytes(tokens, kv8):
    """q and k rows read and rewritten, v read, the cache rows written."""
    return tokens * (2 * HEADS * DIM * 2 + 2 * KV * DIM * 2 + KV * DIM * 2
                     + 2 * KV * (DIM + 16 if kv8 else 2 * DIM))


def _gdn_row_bytes():
    return ROW * 2 + 2 * V_HEADS * GD * 2 + 2 * V_HEADS * 4              # q|k|v, gate, result, a, b


def work(case):
    if case["kind"] == "attention":
        nbytes, flops = _attention_work(case["tokens"], case["pos"], case["kv8"])
        return {"bytes": nbytes, "flops": flops}
    state = V_HEADS * GD * GD * 4
    nbytes = flops = 0
    if case["kind"] == "step":
        rows = case["rows"]
        for n in _lengths(case):
            b, f = _attention_work(rows, n, case["kv8"])
            nbytes += case["attn"] * (b + _prep_bytes(rows, case["kv8"]))
            flops += case["attn"] * f
        ring = ROW * 3 * 2
        moved = (2 + rows - 1) * (state + ring) + rows * _gdn_row_bytes()
        nbytes += case["gdn"] * (case["seqs"] * moved + ROW * 8)
        flops += case["gdn"] * case["seqs"] * rows * V_HEADS * GD * GD * 7
        return {"bytes": nbytes, "flops": flops}
    T = case["tokens"]
    for p in range(0, T, case["chunk"]):
        n = min(case["chunk"], T - p)
        b, f = _attention_work(n, p, case["kv8"])
        nbytes += case["attn"] * (b + _prep_bytes(n, case["kv8"]))
        flops += case["attn"] * f
        nbytes += case["gdn"] * (2 * state + n * _gdn_row_bytes() + ROW * 8)
    flops += case["gdn"] * T * V_HEADS * GD * GD * 7
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """fp16 results of fp32 sums over fp16 operands, four times what a pass differs
    from the same in 64 bits: attention by 3.4e-4 .. 4.7e-4 in the 2-norm (at most
    0.007 of a value), the other layers by up to 9e-4; the gated norm divides rows
    whose terms nearly cancelled by their own size, single values there by 0.05."""
    if case["kind"] == "attention":
        return {"rel": 2e-3, "max": 0.03}
    return {"rel": 4e-3, "max": 0.2}


# ---------------------------------------------------------------------------
# the same in 64 bits, plain torch
# ---------------------------------------------------------------------------

def _prep64(x, w, pos):
    """x [n, heads, DIM] normalised by its root mean square and 1 + w, the first
    ROPE dims rotated by the positions pos [n]."""
    x = x.double()
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * (1 + w.double())
    j = torch.arange(ROPE // 2, device=x.device, dtype=torch.float64)
    ang = pos.double()[:, None] * THETA ** (-2 * j / ROPE)
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    lo, hi = x[..., :ROPE // 2], x[..., ROPE // 2:ROPE]
    return torch.cat([lo * c - hi * s, hi * c + lo * s, x[..., ROPE:]], -1)


def _attend64(q, gate, k, v, pos):
    """q, gate [n, HEADS, DIM] at positions pos [n] over k, v [m, KV, DIM], causal, gated."""
    out = torch.empty_like(q)
    m = k.shape[0]
    step = max(1, (1 << 26) // m)                  # 512 MiB of scores at a time
    at = torch.arange(m, device=q.device)
    for h in range(HEADS):
        kh, vh = k[:, h * KV // HEADS], v[:, h * KV // HEADS]
        for i in range(0, q.shape[0], step):
            s = (q[i:i + step, h] @ kh.T) / math.sqrt(DIM)
            s.masked_fill_(at[None, :] > pos[i:i + step, None], -math.inf)
            out[i:i + step, h] = torch.softmax(s, -1) @ vh
    return out * torch.sigmoid(gate.double())


def _stored64(x, kv8):
    """New K or V rows as the cache holds them."""
    x = x.half()
    return _rows8(*_quantise(x)) if kv8 else x.double()


def _silu64(x):
    return x * torch.sigmoid(x)


def _gdn64(rows, ring, S, w):
    """The recurrent layer over rows [n, ...] from ring [ROW, 3] (oldest first)
    and S [V_HEADS, GD, GD]: (outputs [n, V_HEADS, GD], states after each row)."""
    conv_w, A_log, dt_bias, norm_w = (t.double() for t in w)
    n = rows["qkv"].shape[0]
    x = torch.cat([ring.double().T, rows["qkv"].double()])
    c = _silu64(sum(conv_w[:, j] * x[j:j + n] for j in range(4)))
    qk = c[:, :2 * K_HEADS * GD].view(n, 2 * K_HEADS, GD)
    qk = qk / torch.sqrt((qk * qk).sum(-1, keepdim=True) + EPS)
    rep = V_HEADS // K_HEADS
    q = qk[:, :K_HEADS].repeat_interleave(rep, 1)
    k = qk[:, K_HEADS:].repeat_interleave(rep, 1)
    v = c[:, 2 * K_HEADS * GD:].view(n, V_HEADS, GD)
    beta = torch.sigmoid(rows["b"].double())
    decay = torch.exp(-torch.exp(A_log) * torch.nn.functional.softplus(rows["a"].double() + dt_bias))
    S = S.double().clone()
    y = torch.empty_like(v)
    kept = []
    for t in range(n):
        S.mul_(decay[t, :, None, None])
        d = beta[t, :, None] * (v[t] - (S * k[t, :, None, :]).sum(-1))
        S.addcmul_(d[:, :, None], k[t, :, None, :])
        y[t] = (S * q[t, :, None, :]).sum(-1)
        if n <= 3:
            kept.append(S.clone())
    y *= GD ** -0.5
    y = y / torch.sqrt((y * y).mean(-1, keepdim=True) + EPS) * norm_w
    return y * _silu64(rows["z"].double()), kept or [S]


def _rows_of(rows, s):
    return {k: v[s] for k, v in rows.items()}


def _exact_step(case, seed):
    weights, rows, S, rings, caches = _step_inputs(case, seed)
    types, n = _types(case), case["rows"]
    lens = _lengths(case)
    layers, after = [], [[None] * case["gdn"] for _ in lens]
    attn = gdn = 0
    for t, w in zip(types, weights):
        outs = []
        for b, n_pos in enumerate(lens):
            own = _rows_of(rows, slice(b * n, (b + 1) * n))
            if t == "full_attention":
                pos = torch.arange(n_pos, n_pos + n, device="cuda")
                # the runtime norms its rows in place: each later layer norms them again
                q = own["qg"][..., :DIM]
                k = own["k"]
                for j in [i for i, x in enumerate(types) if x == "full_attention"][:attn + 1]:
                    q, k = (_prep64(q, weights[j][0], pos).half(), _prep64(k, weights[j][1], pos).half())
                old = [_rows8(*c) if case["kv8"] else c.double() for c in caches[b][attn]]
                kk = torch.cat([old[0], _stored64(k, case["kv8"])])
                vv = torch.cat([old[1], _stored64(own["v"], case["kv8"])])
                outs.append(_attend64(q.double(), own["qg"][..., DIM:], kk, vv, pos))
            else:
                y, kept = _gdn64(own, rings[b][gdn], S[b][gdn], w)
                after[b][gdn] = kept
                outs.append(y)
        layers.append(torch.cat(outs))
        attn, gdn = attn + (t == "full_attention"), gdn + (t != "full_attention")
    out = dict(layers=layers, s=[torch.stack([x[-1] for x in a]) for a in after],
               conv=[None] * len(lens), checkpoints=[], kv=[])
    if n > 1:
        out["checkpoints"] = [torch.stack([torch.stack([x[r] for x in after[0]])
                                           for r in range(n - 1)])]
    return out


def _exact_prompt(case, seed):
    weights, rows = _prompt_inputs(case, seed)
    T = case["tokens"]
    pos = torch.arange(T, device="cuda")
    whole, S = [], []
    for t, w in zip(_types(case), weights):
        if t == "full_attention":
            q = _prep64(rows["qg"][..., :DIM], w[0], pos)
            k = _stored64(_prep64(rows["k"], w[1], pos), case["kv8"])
            whole.append(_attend64(q, rows["qg"][..., DIM:], k, _stored64(rows["v"], case["kv8"]),
                                   pos))
        else:
            ring = torch.zeros((ROW, 3), device="cuda")
            y, kept = _gdn64(rows, ring, torch.zeros((V_HEADS, GD, GD), device="cuda"), w)
            whole.append(y)
            S.append(kept[-1])
    layers = [y[p:p + case["chunk"]] for p in range(0, T, case["chunk"]) for y in whole]
    return dict(layers=layers, s=torch.stack(S), conv=None, kv=[None, None])


def exact(case, seed):
    if case["kind"] == "step":
        return _exact_step(case, seed)
    if case["kind"] == "prompt":
        return _exact_prompt(case, seed)
    qg, k, v = _attention_inputs(case, seed)
    if case["kv8"]:
        k, v = _rows8(*k), _rows8(*v)
    pos = torch.arange(case["pos"], case["pos"] + case["tokens"], device="cuda")
    return _attend64(qg[..., :DIM].double(), qg[..., DIM:], k.double(), v.double(), pos)
