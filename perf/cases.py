"""The work that a user of this framework has it do, as cases that can be timed and compared.

Four kinds of call, each through its public entry point:

* ``forward``: ``smat_attention`` over features (prefill), one mask per length;
* ``qkv``:     ``smat_attention_fused`` from q, k, v (the feature map inside);
* ``train``:   one training step of the layer, forward and backward, with positional or
               content-hashed assignment;
* ``decode``:  ``SmatDecoder`` steps after a context, replayed from one graph (serving) or
               launched one by one.

``listed()`` names the cases, ``draw()`` gives more of the same ranges, ``exact()`` computes a
case in 64 bits with plain torch.  Only the mask's integer tables (which point lies on which
line) are taken from the package there: they are inputs of the path.
"""
import functools
import math

import torch

from smat_attention_amd import attention as A
from smat_attention_amd.assign import ContentAssign
from smat_attention_amd.mask import build_mask

CHUNK = 128
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _forward(name, nb, T, d, hd, dtype="bf16", gate=False, n_P=0):
    return {"name": name, "kind": "forward", "nb": nb, "T": T, "d": d, "hd": hd, "dtype": dtype,
            "gate": gate, "n_P": n_P}


def _qkv(name, nb, T, d, hd=128, dtype="bf16", gate=False, key_gate=False):
    return {"name": name, "kind": "qkv", "nb": nb, "T": T, "d": d, "hd": hd, "dtype": dtype,
            "gate": gate, "key_gate": key_gate, "n_P": 0}


def _train(name, B, H, T, d, hd=64, assign="positional"):
    return {"name": name, "kind": "train", "B": B, "H": H, "nb": B * H, "T": T, "d": d, "hd": hd,
            "dtype": "bf16", "assign": assign, "n_P": 0}


def _decode(name, nb, context, room, d, hd, steps, graph):
    return {"name": name, "kind": "decode", "nb": nb, "context": context, "T": context + room,
            "d": d, "hd": hd, "dtype": "bf16", "steps": steps, "graph": graph, "n_P": 0}


def listed():
    return [
        # a short fp32 prompt, 4 heads of 64: launches and host latency
        _forward("prompt_fp32_T1024", 4, 1024, 2, 64, dtype="fp32"),
        # an ordinary batch of prompts at head size 64 (B = 4, H = 8)
        _forward("batch_T8192_hd64", 32, 8192, 2, 64),
        # ragged length, odd head size, fp16, output gate and global channel
        _forward("ragged_T10007_hd96", 12, 10007, 3, 96, dtype="fp16", gate=True, n_P=128),
        # long prefills at head size 128 (B = 1, H = 8), and the plain causal control
        _forward("prefill_T32768", 8, 32768, 3, 128),
        _forward("prefill_T131072", 8, 131072, 3, 128),
        _forward("prefill_T131072_d1", 8, 131072, 1, 128),
        _forward("prefill_T524288", 8, 524288, 3, 128),
        # the same prefill from q, k, v, with the key gate
        _qkv("qkv_T131072", 8, 131072, 3, key_gate=True),
        # training steps of a small model's layer (B = 8, H = 12)
        _train("train_T4096_d3", 8, 12, 4096, 3),
        _train("train_hashed_T4096_d2", 8, 12, 4096, 2, assign="hashed"),
        # cached decode: a served batch replayed from a graph, and one prompt stepped eagerly
        _decode("decode_nb128", 128, 65536, 4096, 3, 128, steps=64, graph=True),
        _decode("decode_eager_nb8", 8, 8192, 1024, 3, 128, steps=16, graph=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward"] * 4 + ["qkv", "train", "train", "decode"])
    ragged = rng.random() < 0.4
    d = rng.choice([1, 2, 3, 3])
    if kind in ("forward", "qkv"):
        if kind == "qkv":
            hd, dtype = 128, rng.choice(["bf16", "bf16", "fp16"])
        else:
            hd = rng.choice([64, 64, 64, 128, 128, 128, 32, 80, 96])
            dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        # tokens x head size: long prefills at the wide 16-bit shape, batches of prompts elsewhere
        cap = 8 * 131072 * 128 if hd == 128 and dtype != "fp32" and not ragged else 32 * 8192 * 64
        T = _log(rng, 1024, min(262144, cap // (4 * hd)))
        T = T if ragged else -(-T // 128) * 128
        nb = _log(rng, 4, max(4, min(64, cap // (T * hd))))
        if kind == "qkv":
            return {k: v for k, v in _qkv("", nb, T, d, hd, dtype, gate=rng.random() < 0.3,
                                          key_gate=rng.random() < 0.5).items() if k != "name"}
        return {k: v for k, v in _forward("", nb, T, d, hd, dtype, gate=rng.random() < 0.3,
                                          n_P=rng.choice([0, 0, 0, 128]) if T >= 4096 and d > 1
                                          else 0).items() if k != "name"}
    if kind == "train":
        T = _log(rng, 1024, 4096)
        T = T if ragged and rng.random() < 0.5 else -(-T // 128) * 128
        c = _train("", rng.randint(2, 8), rng.choice([4, 8, 12]), T, rng.choice([2, 3]),
                   assign=rng.choice(["positional", "hashed"]))
        return {k: v for k, v in c.items() if k != "name"}
    nb = _log(rng, 8, 128)
    c = _decode("", nb, 128 * _log(rng, 32, 512 if nb <= 64 else 256), 1024, d,
                rng.choice([64, 128, 128]), 2 * rng.randint(4, 32), rng.random() < 0.5)
    return {k: v for k, v in c.items() if k != "name"}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

@functools.lru_cache(maxsize=64)
def _mask(T, d, n_P):
    """The mask of one length, staged once as a program keeps it."""
    return A.to_device(build_mask(T, d, chunk=CHUNK, n_P=n_P), "cuda:0")


def _gen(seed):
    return torch.Generator(device="cuda:0").manual_seed(seed)


def _normal(g, *shape, scale=1.0, dtype=torch.float32):
    return torch.randn(*shape, device="cuda:0", generator=g).mul_(scale).to(dtype)


def _feature_weight(hd, dtype):
    """The feature map's weight: make_phi's draw for its default seed."""
    g = torch.Generator().manual_seed(0)
    W = torch.randn(hd, hd, generator=g, dtype=torch.float64) / math.sqrt(hd)
    return W.to(device="cuda:0", dtype=dtype)


def _features(g, nb, T, hd, dtype, scale=1.0):
    """elu(x W^T) + 1 of x ~ N(0, scale^2), one sequence at a time, rounded to the input type."""
    W = _feature_weight(hd, torch.float32)
    out = torch.empty(nb, T, hd, device="cuda:0", dtype=dtype)
    for s in range(nb):
        out[s] = torch.nn.functional.elu(_normal(g, T, hd, scale=scale) @ W.T).add_(1.0)
    return out


def _values(g, nb, T, hd, dtype):
    """[V, 1] as featurise returns it: rows padded to 8 elements."""
    p = hd + 1
    buf = torch.zeros(nb, T, -(-p // 8) * 8, device="cuda:0", dtype=dtype)
    for s in range(nb):
        buf[s, :, :hd] = _normal(g, T, hd)
    buf[..., hd] = 1.0
    return buf[..., :p]


def _forward_inputs(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    nb, T, hd = c["nb"], c["T"], c["hd"]
    Phi = _features(g, nb, T, hd, dt)
    Psi = _features(g, nb, T, hd, dt, scale=hd ** -0.5)
    Vb = _values(g, nb, T, hd, dt)
    gate = (torch.rand(nb, T, device="cuda:0", generator=g) + 0.5).to(dt) if c["gate"] else None
    return Phi, Psi, Vb, gate


def _qkv_inputs(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    nb, T, hd = c["nb"], c["T"], c["hd"]
    q = _normal(g, nb, T, hd, dtype=dt)
    k = _normal(g, nb, T, hd, scale=hd ** -0.5, dtype=dt)
    v = _normal(g, nb, T, hd, dtype=dt)
    h = (torch.rand(nb, T, device="cuda:0", generator=g) + 0.5).to(dt) if c["key_gate"] else None
    gate = (torch.rand(nb, T, device="cuda:0", generator=g) + 0.5).to(dt) if c["gate"] else None
    return q, k, v, h, gate


def _train_inputs(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    nb, T, hd = c["nb"], c["T"], c["hd"]
    q = _normal(g, nb, T, hd, dtype=dt)
    k = _normal(g, nb, T, hd, scale=hd ** -0.5, dtype=dt)
    v = _normal(g, nb, T, hd, dtype=dt)
    dO = _normal(g, nb, T, hd, dtype=dt)
    x = w = None
    if c["assign"] == "hashed":
        x = _normal(g, c["B"], T, c["H"] * hd)
        w = _normal(g, c["H"], _mask(T, c["d"], 0).dim, c["H"] * hd)
    return q, k, v, dO, x, w


def _decode_inputs(c, seed):
    """Landmark and context keys and values, and the steps' features and values."""
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    nb, hd, ctx, steps = c["nb"], c["hd"], c["context"], c["steps"]
    Psi = _features(g, nb, ctx, hd, dt, scale=hd ** -0.5)
    Vb = _values(g, nb, ctx, hd, dt)
    phi_t = _features(g, nb, steps, hd, dt)
    psi_t = _features(g, nb, steps, hd, dt, scale=hd ** -0.5)
    vb_t = _values(g, nb, steps, hd, dt)
    return Psi, Vb, phi_t, psi_t, vb_t


def prepare(case, seed):
    c, kind = case, case["kind"]
    spec = _mask(c["T"], c["d"], c["n_P"])
    if kind == "forward":
        Phi, Psi, Vb, gate = _forward_inputs(c, seed)
        return {"kind": kind, "spec": spec, "x": (Phi, Psi, Vb), "g": gate}
    if kind == "qkv":
        q, k, v, h, gate = _qkv_inputs(c, seed)
        phi = A.make_phi(c["hd"], c["hd"], device="cuda:0", dtype=q.dtype)
        return {"kind": kind, "spec": spec, "x": (q, k, v), "phi": phi, "h": h, "g": gate}
    if kind == "train":
        q, k, v, dO, x, w = _train_inputs(c, seed)
        phi = A.make_phi(c["hd"], c["hd"], device="cuda:0", dtype=q.dtype)
        m = None
        if x is not None:
            m = ContentAssign(c["H"], c["H"] * c["hd"], spec, mode="point").to("cuda:0")
            with torch.no_grad():
                m.W.copy_(w)
            x.requires_grad_(True)
        for t in (q, k, v):
            t.requires_grad_(True)
        return {"kind": kind, "spec": spec, "x": (q, k, v), "phi": phi, "dO": dO, "u": x, "m": m}
    Psi, Vb, phi_t, psi_t, vb_t = _decode_inputs(c, seed)
    n = spec.n
    dec = A.SmatDecoder(Psi[:, :n], Vb[:, :n], spec)
    dec.advance(Psi[:, n:], Vb[:, n:])
    del Psi, Vb
    out = torch.empty(c["steps"], c["nb"], c["hd"], device="cuda:0")
    state = {"kind": kind, "dec": dec, "x": (phi_t, psi_t, vb_t), "out": out, "graph": None}
    if c["graph"]:
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(stream):
            with torch.cuda.graph(graph, stream=stream):
                _steps(state)
        torch.cuda.current_stream().wait_stream(stream)
        state["graph"] = graph
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _steps(s):
    phi_t, psi_t, vb_t = s["x"]
    for i in range(phi_t.shape[1]):
        s["dec"].step(phi_t[:, i], psi_t[:, i], vb_t[:, i], out=s["out"][i])


def run(state):
    s, kind = state, state["kind"]
    if kind == "forward":
        return A.smat_attention(*s["x"], s["spec"], g=s["g"])
    if kind == "qkv":
        return A.smat_attention_fused(*s["x"], s["phi"], s["spec"], g=s["g"], h=s["h"])
    if kind == "decode":
        if s["graph"] is not None:
            s["graph"].replay()              # an even number of steps: the state's first buffer
        else:
            _steps(s)
        return {"out": s["out"], "S": s["dec"].S}
    q, k, v = s["x"]
    u, m, n = s["u"], s["m"], s["spec"].n
    for t in (q, k, v, u):
        if t is not None:
            t.grad = None
    Phi, Psi, Vb = A.featurise(q, k, v, s["phi"])
    if m is None:
        o = A.smat_attention(Phi, Psi, Vb, s["spec"]).to(q.dtype)
    else:
        m.zero_grad(set_to_none=True)
        H = A.segmented_causal_scan(Phi, Psi, Vb, n, CHUNK)
        o = A.combine_normalise(H, m(u, Phi, Psi, Vb, n), n, out_dtype=q.dtype)
    o.backward(s["dO"])
    got = {"o": o.detach(), "dq": q.grad, "dk": k.grad, "dv": v.grad}
    if m is not None:
        got.update(du=u.grad, dW=m.W.grad, dgamma=m.gamma.grad, db=m.b.grad)
    return got


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _useful_flops(spec, nb, T, r, p):
    """Causal products within chunks, chunk summaries and their reads, pool, query (2 a MAC),
    and the incidence's adds."""
    macs = (T * (min(CHUNK, T) + 1) / 2 * (r + p) + 2 * T * r * p
            + (spec.n - spec.n_P) * r * p + spec.T_R * r * p)
    adds = 0 if spec.d < 3 else spec.I_prof * r * p
    return nb * (2.0 * macs + adds)


def work(case):
    c = case
    spec = build_mask(c["T"], c["d"], chunk=CHUNK, n_P=c["n_P"])
    nb, T, hd = c["nb"], c["T"], c["hd"]
    r, p, eb = hd, hd + 1, DTYPES[c["dtype"]].itemsize
    if c["kind"] == "decode":
        step = nb * (3 * r * p * 4 + (2 * r + p) * eb + hd * 4)
        return {"bytes": c["steps"] * step, "flops": c["steps"] * nb * 6.0 * r * p}
    flops = _useful_flops(spec, nb, T, r, p)
    feat = 2.0 * 2 * nb * T * hd * r
    if c["kind"] == "forward":
        return {"bytes": nb * T * ((2 * r + p) * eb + hd * 4), "flops": flops}
    if c["kind"] == "qkv":
        return {"bytes": nb * T * (3 * hd * eb + hd * 4), "flops": flops + feat}
    # q, k, v, dO in; o and three gradients out; the hash input and its gradient
    nbytes = nb * T * hd * eb * 8
    if c["assign"] == "hashed":
        nbytes += 2 * c["B"] * T * c["H"] * hd * 4
    return {"bytes": nbytes, "flops": 3 * (flops + feat)}


def tolerance(case):
    """About four times what a path is off its 64-bit value where the input type's rounding of
    the in-chunk scores (forward: 1.3e-3 in bf16, 1.7e-4 in fp16) decides it; dq of a training
    step, 1.5e-2 off through the feature map's rounded argument, sets that kind's."""
    if case["kind"] == "decode" or case["dtype"] == "fp32":
        return {"rel": 1e-5}
    if case["kind"] == "train":
        return {"rel": 2e-2, "max": 0.5}
    return {"rel": 5e-3 if case["dtype"] == "bf16" else 8e-4}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _causal64(Phi, Psi, Vb):
    """Sum over j <= i of (Phi_i . Psi_j) Vb_j for one sequence (T, r), (T, r), (T, p)."""
    T, r = Phi.shape
    p, C = Vb.shape[1], CHUNK
    pad = (-T) % C
    f = torch.nn.functional.pad
    P, K, V = (f(t, (0, 0, 0, pad)).reshape(-1, C, t.shape[1]) for t in (Phi, Psi, Vb))
    D = K.transpose(1, 2).contiguous() @ V
    S = torch.cat([torch.zeros_like(D[:1]), D.cumsum(0)[:-1]])
    A_ = (P @ K.transpose(1, 2).contiguous()).tril()
    return (P @ S + A_ @ V).reshape(-1, p)[:T]


def _scan64(Phi, Psi, Vb, n):
    parts = [_causal64(*(t[a:b] for t in (Phi, Psi, Vb)))
             for a, b in ((0, n), (n, Phi.shape[0])) if b > a]
    return torch.cat(parts)


def _pool64(Psi, Vb, N0):
    """Sum of Psi_j Vb_j^T over j = x mod N0: (N0, r, p)."""
    n, r = Psi.shape
    f = torch.nn.functional.pad
    pad = (-n) % N0
    K = f(Psi, (0, 0, 0, pad)).reshape(-1, N0, r).permute(1, 2, 0).contiguous()
    V = f(Vb, (0, 0, 0, pad)).reshape(-1, N0, Vb.shape[1]).permute(1, 0, 2).contiguous()
    return K @ V


def _points(spec):
    return torch.as_tensor(spec.C_indices.reshape(spec.B, -1), device="cuda:0").long()


def _schedule64(Phi, Psi, Vb, spec):
    """Numerators and normaliser (T, p) of one sequence under the positional schedule."""
    n, n_P, B = spec.n, spec.n_P, spec.B
    H = _scan64(Phi, Psi, Vb, n)
    F = _pool64(Psi[n_P:n], Vb[n_P:n], spec.N0)
    pts = _points(spec)
    U = F[pts[:, 0]]
    for j in range(1, pts.shape[1]):
        U = U + F[pts[:, j]]
    if n_P:
        U = U + (Psi[:n_P].T.contiguous() @ Vb[:n_P])[None]
    T_R = Phi.shape[0] - n
    P = torch.nn.functional.pad(Phi[n:], (0, 0, 0, (-T_R) % B))
    P = P.reshape(-1, B, P.shape[1]).transpose(0, 1).contiguous()
    Y = (P @ U).transpose(0, 1).reshape(-1, Vb.shape[1])[:T_R]
    return torch.cat([H[:n], H[n:] + Y])


def _map64(x, W):
    return torch.nn.functional.elu(x @ W.T) + 1.0


def _ones64(v):
    return torch.cat([v, torch.ones_like(v[:, :1])], 1)


def _positions64(x, W, gamma, b, q):
    """Hash positions (L, dim) of one head; the bin of a position is its floor, as the 32-bit
    hash takes it, since a position on a bin's edge falls to either side by rounding alone."""
    def s_of(x, W, gamma, b):
        Wn = W / W.norm(dim=-1, keepdim=True).clamp_min(1e-6)
        z = torch.nn.functional.layer_norm(x, (x.shape[-1],)) @ Wn.T * gamma + b
        return (torch.special.ndtr(z) * q).clamp(0.0, q - 1e-4)
    s = s_of(x, W, gamma, b)
    with torch.no_grad():
        lo = s_of(*(t.float() for t in (x, W, gamma, b))).floor().long()
    return s, lo


def _pairs64(s, lo, q):
    """The cells and straight-through weights (L, 2^dim) of every token: forward one on the
    chosen cell (pair 0) and zero elsewhere, backward the two-bin interpolation."""
    f = s - lo
    hi = (lo + 1).clamp(max=q - 1)
    dim = s.shape[1]
    idx = torch.zeros(s.shape[0], 1, dtype=torch.long, device=s.device)
    w = torch.ones(s.shape[0], 1, dtype=s.dtype, device=s.device)
    for k in range(dim):
        place = q ** (dim - 1 - k)
        one = 1.0 + (f.detach() - f)[:, k:k + 1]
        zero = (f - f.detach())[:, k:k + 1]
        idx = torch.cat([idx + lo[:, k:k + 1] * place, idx + hi[:, k:k + 1] * place], 1)
        w = torch.cat([w * one, w * zero], 1)
    return idx, w


def _hashed64(Phi, Psi, Vb, x, W, gamma, b, spec, cols, cells):
    """The content-addressed long-range term (T_R, p) of one sequence and head."""
    n, r, p = spec.n, Phi.shape[1], Vb.shape[1]
    s, lo = _positions64(x, W, gamma, b, int(spec.q))
    idx, w = _pairs64(s, lo, int(spec.q))
    idk, wk = idx[:n].clone(), w[:n].clone()
    if len(cols):                                    # planted keys: one fixed cell
        idk[cols] = cells[:, None]
        wk[cols] = 0.0
        wk[cols, 0] = 1.0
    F = torch.zeros(spec.N0, r * p, dtype=Phi.dtype, device=Phi.device)
    PV = (Psi[:n, :, None] * Vb[:n, None, :]).reshape(n, r * p)
    for m in range(idk.shape[1]):
        F = F.index_add(0, idk[:, m], wk[:, m, None] * PV)
    y = 0.0
    for m in range(idx.shape[1]):
        rows = F[idx[n:, m]].reshape(-1, r, p)
        y = y + w[n:, m, None] * (Phi[n:, None, :] @ rows)[:, 0]
    return y


def _exact_train(c, seed):
    q, k, v, dO, x, w = _train_inputs(c, seed)
    spec, H = _mask(c["T"], c["d"], 0), c["H"]
    W = _feature_weight(c["hd"], q.dtype).double()
    names = ("o", "dq", "dk", "dv")
    got = {m: torch.empty(*q.shape, dtype=torch.float64, device="cuda:0") for m in names}
    params = []
    if x is not None:
        ones = torch.ones(H, spec.dim, dtype=torch.float64, device="cuda:0")
        params = [t.requires_grad_(True) for t in (w.double(), ones, ones * 0.0)]
        cols = torch.as_tensor(spec.planted_cols, device="cuda:0").long()
        cells = torch.tensor([int(spec.q) ** (spec.dim - i) for i in range(1, spec.dim + 1)],
                             device="cuda:0")
        cells = cells[:len(cols)][cols < spec.n]
        cols = cols[cols < spec.n]
        got["du"] = torch.empty(*x.shape, dtype=torch.float64, device="cuda:0")
    for b in range(c["B"]):
        xb = x[b].double().requires_grad_(True) if x is not None else None
        for h in range(H):
            i = b * H + h
            q_, k_, v_ = (t[i].double().requires_grad_(True) for t in (q, k, v))
            Phi, Psi, Vb = _map64(q_, W), _map64(k_, W), _ones64(v_)
            if x is None:
                N = _schedule64(Phi, Psi, Vb, spec)
            else:
                Hs = _scan64(Phi, Psi, Vb, spec.n)
                Y = _hashed64(Phi, Psi, Vb, xb, *(t[h] for t in params), spec, cols, cells)
                N = torch.cat([Hs[:spec.n], Hs[spec.n:] + Y])
            o = N[:, :-1] / N[:, -1:].clamp_min(1e-6)
            o.backward(dO[i].double())
            for m, t in zip(names, (o.detach(), q_.grad, k_.grad, v_.grad)):
                got[m][i] = t
        if x is not None:
            got["du"][b] = xb.grad
    if x is not None:
        got.update(dW=params[0].grad, dgamma=params[1].grad, db=params[2].grad)
    return got


def _exact_decode(c, seed):
    Psi, Vb, phi_t, psi_t, vb_t = _decode_inputs(c, seed)
    spec = _mask(c["T"], c["d"], c["n_P"])
    n, ctx, nb, r, p = spec.n, c["context"], c["nb"], c["hd"], c["hd"] + 1
    S = torch.empty(nb, r, p, dtype=torch.float64, device="cuda:0")
    for s in range(nb):
        S[s] = Psi[s, n:].double().T.contiguous() @ Vb[s, n:].double()
    pts = _points(spec)
    prof = torch.arange(n, device="cuda:0") % spec.N0
    out = torch.empty(c["steps"], nb, c["hd"], dtype=torch.float64, device="cuda:0")
    U = {}
    for i in range(c["steps"]):
        S = S + psi_t[:, i].double()[:, :, None] * vb_t[:, i].double()[:, None, :]
        h = (ctx - n + i) % spec.B
        if h not in U:
            on = torch.isin(prof, pts[h]).nonzero()[:, 0]
            U = {h: torch.stack([Psi[s, on].double().T.contiguous() @ Vb[s, on].double()
                                 for s in range(nb)])}
        o = (phi_t[:, i].double()[:, None, :] @ (S + U[h]))[:, 0]
        out[i] = o[:, :-1] / o[:, -1:]
    return {"out": out, "S": S}


def exact(case, seed):
    c = case
    if c["kind"] == "train":
        return _exact_train(c, seed)
    with torch.no_grad():
        if c["kind"] == "decode":
            return _exact_decode(c, seed)
        spec = _mask(c["T"], c["d"], c["n_P"])
        out = torch.empty(c["nb"], c["T"], c["hd"], dtype=torch.float64, device="cuda:0")
        if c["kind"] == "forward":
            Phi, Psi, Vb, gate = _forward_inputs(c, seed)
            feats = lambda s: (Phi[s].double(), Psi[s].double(), Vb[s].double())
        else:
            q, k, v, h, gate = _qkv_inputs(c, seed)
            W = _feature_weight(c["hd"], q.dtype).double()

            def feats(s):
                Psi = _map64(k[s].double(), W)
                Psi = Psi * h[s].double()[:, None] if h is not None else Psi
                return _map64(q[s].double(), W), Psi, _ones64(v[s].double())
        for s in range(c["nb"]):
            N = _schedule64(*feats(s), spec)
            out[s] = N[:, :-1] / N[:, -1:]
            if gate is not None:
                out[s] *= gate[s].double()[:, None]
        return out
