"""The work that users of this framework have it do, as measurable cases.

Each case is one call of a public entry point: the four kernel modules that
``compile_kernels()`` returns and the layer ``GDNLayerCustom``.  Shapes come
from this repository's configurations, tests and benchmark (hidden 2048,
H = 16, dk = 128, dv = 128 or the reference's 256, conv of 4 taps) with odd
and ragged lengths beside the round ones.  ``listed()`` names the fixed cases,
``draw(rng)`` gives others from the same ranges.
"""

import math

import torch

DEV = "cuda"
DK, CK, D = 128, 4, 2048
LN_HALF = math.log(0.5)


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # One user being answered, token by token: the smallest call there is,
        # where launches and latency are the time.  The reference layer's dims.
        dict(name="decode_one_user", kind="layer_decode", B=1, dv=256),
        # A serving batch in the middle of the range, not a round number.
        dict(name="decode_serving", kind="layer_decode", B=48, dv=128),
        # The recurrence alone over a full batch: 512 MiB of state in place.
        dict(name="decode_full_batch", kind="decode", B=256, H=32, dv=128),
        # A chat-sized prompt through the prefill kernel, ragged, dv = 256.
        dict(name="prefill_prompt", kind="prefill", B=1, H=16, T=333, dv=256, masked=False, state=False),
        # One long document (the headline prefill).
        dict(name="prefill_document", kind="prefill", B=1, H=16, T=8192, dv=128, masked=False, state=False),
        # A right-padded batch that continues from earlier states.
        dict(name="prefill_batch", kind="prefill", B=8, H=16, T=2000, dv=128, masked=True, state=True),
        # Eight packed sequences of unequal length, nonzero initial states.
        dict(name="prefill_packed", kind="varlen", H=16, dv=128,
             lengths="3670,1053,3636,3547,4688,709,2874,4497"),
        # A short question through the whole layer, the state kept for decode.
        dict(name="layer_question", kind="layer", B=1, T=77, dv=256, masked=False, keep=True),
        # A longer prompt through the whole layer, the state kept for decode.
        dict(name="layer_prompt", kind="layer", B=1, T=1500, dv=128, masked=False, keep=True),
        # A full training-sized batch through the layer: the largest call.
        dict(name="layer_batch", kind="layer", B=4, T=4096, dv=128, masked=False, keep=False),
        # What a server's step packs together: short prompts of mixed length.
        dict(name="layer_packed", kind="layer_packed", dv=128,
             lengths="31,410,7,873,128,250,64,520,99,301", keep=True),
        # The fused projection + conv + SiLU on its own.
        dict(name="projection", kind="proj", B=1, T=2048, D_out=2048),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _lengths(rng, most, total):
    n, got = rng.randint(2, 12), []
    for _ in range(n):
        room = total - sum(got)
        if room < 1:
            break
        got.append(min(room, _log_int(rng, 4, most)))
    return ",".join(str(x) for x in got)


def draw(rng):
    kind = rng.choice(["layer_decode", "decode", "prefill", "prefill", "varlen", "layer", "layer", "layer_packed", "proj"])
    dv = rng.choice([128, 128, 256])
    if kind == "layer_decode":
        return dict(kind=kind, B=_log_int(rng, 1, 256), dv=dv)
    if kind == "decode":
        return dict(kind=kind, B=_log_int(rng, 4, 256 * 128 // dv), H=rng.choice([8, 16, 32]), dv=dv)
    if kind == "prefill":
        T = _log_int(rng, 1, 8192)
        return dict(kind=kind, B=_log_int(rng, 1, max(1, min(32, 65536 // T * 128 // dv))), H=rng.choice([4, 16, 16]), T=T,
                    dv=rng.choice([64, 128, 128, 256]), masked=rng.random() < 0.3, state=rng.random() < 0.5)
    if kind == "varlen":
        return dict(kind=kind, H=16, dv=dv, lengths=_lengths(rng, 8192, 24000))
    if kind == "layer":
        T = _log_int(rng, 1, 4096)
        return dict(kind=kind, B=_log_int(rng, 1, max(1, min(16, 12000 // T))), T=T, dv=dv, masked=rng.random() < 0.3,
                    keep=rng.random() < 0.6)
    if kind == "layer_packed":
        return dict(kind=kind, dv=dv, lengths=_lengths(rng, 2048, 8192), keep=rng.random() < 0.6)
    T = _log_int(rng, 1, 4096)
    return dict(kind=kind, B=_log_int(rng, 1, max(1, min(16, 16384 // T))), T=T, D_out=rng.choice([2048, 2048, 4096]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
class _Draws:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device=DEV) * std

    def bf(self, *shape, std=1.0):
        return self.normal(*shape, std=std).to(torch.bfloat16)

    def unit_rows(self, *shape):
        x = self.normal(*shape)
        return (x / x.norm(dim=-1, keepdim=True)).to(torch.bfloat16)

    def uniform(self, *shape):
        return torch.rand(shape, generator=self.g, device=DEV)


def _len_list(case):
    return [int(x) for x in case["lengths"].split(",")]


def _padding_mask(d, B, T):
    """Right padding: each row keeps at least half of its tokens (the first row all)."""
    keep = (T * (0.5 + 0.5 * d.uniform(B))).ceil()
    keep[0] = T
    return (torch.arange(T, device=DEV)[None, :] < keep[:, None]).float().contiguous()


def _weights(d, dv, H=16):
    """Layer weights: the reference's fan-in scaled draws at dv = 256, N(0, 0.02) at dv = 128."""
    std = 0.02 if dv == 128 else None

    def proj(rows, cols, extra=1.0):
        return d.bf(rows, cols, std=std or cols ** -0.5 * extra)

    def conv(rows):
        return d.bf(rows, CK, std=std or CK ** -0.5)

    return dict(norm_gamma=(1 + d.normal(D, std=0.1)).to(torch.bfloat16),
                W_q=proj(H * DK, D, DK ** -0.5), conv_q=conv(H * DK), W_k=proj(H * DK, D, DK ** -0.5), conv_k=conv(H * DK),
                W_v=proj(H * dv, D, DK ** -0.5), conv_v=conv(H * dv), W_a=proj(H, D), W_b=proj(H, D),
                A_log=torch.full((H,), LN_HALF, device=DEV), dt_bias=torch.tensor(0.25, device=DEV), W_o=proj(D, H * dv))


def _inputs(case, seed):
    """The tensors of a case, made from the seed alone."""
    d, kind = _Draws(seed), case["kind"]
    if kind == "decode":
        B, H, dv = case["B"], case["H"], case["dv"]
        return dict(q=d.unit_rows(B, H, DK), k=d.unit_rows(B, H, DK), v=d.bf(B, H, dv), a=d.bf(B, H), b=d.bf(B, H),
                    A_log=torch.full((H,), LN_HALF, device=DEV), dt_bias=torch.zeros(H, device=DEV),
                    S=d.normal(B, H, DK, dv, std=0.02))
    if kind in ("prefill", "varlen"):
        H, dv = case["H"], case["dv"]
        if kind == "prefill":
            B, T, n = case["B"], case["T"], case["B"]
        else:
            B, T, n = 1, sum(_len_list(case)), len(_len_list(case))
        i = dict(q=d.unit_rows(B, H, T, DK), k=d.unit_rows(B, H, T, DK), v=d.bf(B, H, T, dv), a=d.bf(B, H, T),
                 b=d.bf(B, H, T), A_log=torch.full((H,), LN_HALF, device=DEV))
        i["mask"] = _padding_mask(d, B, T) if case.get("masked") else torch.ones(B, T, device=DEV)
        if kind == "varlen" or case["state"]:
            i["S"] = d.normal(n, H, DK, dv, std=0.02)
        return i
    if kind == "proj":
        return dict(x=d.bf(case["B"], case["T"], D), W=d.bf(case["D_out"], D, std=D ** -0.5), conv=d.bf(case["D_out"], CK, std=0.5))
    dv, H = case["dv"], 16
    w = _weights(d, dv)
    if kind == "layer_decode":
        B = case["B"]
        p = 0.9 if dv == 128 else 0.09  # the projections' spread under these weights
        state = dict(recurrent=d.normal(B, H, DK, dv, std=0.02), conv_q=d.bf(B, H * DK, CK - 1, std=p),
                     conv_k=d.bf(B, H * DK, CK - 1, std=p), conv_v=d.bf(B, H * dv, CK - 1, std=p), xn=d.bf(B, CK - 1, D))
        return dict(w=w, x=d.bf(B, 1, D), state=state)
    if kind == "layer_packed":
        return dict(w=w, x=d.bf(1, sum(_len_list(case)), D), mask=None)
    B, T = case["B"], case["T"]
    return dict(w=w, x=d.bf(B, T, D), mask=_padding_mask(d, B, T) if case["masked"] else None)


def prepare(case, seed):
    from gdn_18646_amd import compile_kernels

    i = _inputs(case, seed)
    i["case"] = case
    i["exts"] = compile_kernels()
    if case["kind"] in ("varlen", "layer_packed"):  # host offsets, as a server has them
        cu = [0]
        for n in _len_list(case):
            cu.append(cu[-1] + n)
        i["cu"] = torch.tensor(cu, dtype=torch.int32)
    if case["kind"].startswith("layer"):
        from gdn_18646_amd.gdn_layer import GDNLayerCustom

        i["layer"] = GDNLayerCustom(i["w"], i["exts"])
    if case["kind"] == "decode":
        i["o"] = torch.empty(case["B"], case["H"], case["dv"], device=DEV)
    if case["kind"] == "prefill" and "S" not in i:
        i["S"] = torch.empty(0, device=DEV)
    return i


def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "layer_decode":
        return s["layer"].decode(s["x"], s["state"], inplace=True)
    if kind == "decode":
        s["exts"]["decode"].forward(s["q"], s["k"], s["v"], s["a"], s["b"], s["A_log"], s["dt_bias"], s["S"], DK ** -0.5, s["o"], s["S"])
        return s["o"], s["S"]
    if kind == "prefill":
        return s["exts"]["prefill"].prefill(s["q"], s["k"], s["v"], s["A_log"], s["a"], 0.0, s["b"], s["mask"], s["S"], 0.0)
    if kind == "varlen":
        return s["exts"]["prefill"].prefill_varlen(s["q"], s["k"], s["v"], s["A_log"], s["a"], 0.0, s["b"], s["cu"], s["S"], 0.0)
    if kind == "proj":
        return s["exts"]["proj"].forward(s["x"], s["W"], s["conv"])
    if kind == "layer_packed":
        return s["layer"].forward(s["x"], return_state=case["keep"], cu_seqlens=s["cu"])
    return s["layer"].forward(s["x"], s["mask"], return_state=case["keep"])


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _prefill_work(ntok, H, nseq, dv, state):
    C = 64
    return dict(bytes=ntok * H * (2 * (2 * DK + dv) + 2 * dv + 4) + 4 * nseq * H * DK * dv * (2 if state else 1),
                flops=ntok * H * 2 * (3 * C * DK + 2 * C * dv + 3 * DK * dv))


def work(case):
    kind = case["kind"]
    if kind == "decode":
        n, dv = case["B"] * case["H"], case["dv"]
        return dict(bytes=n * (8 * DK * dv + 2 * (2 * DK + dv) + 4 * dv + 4), flops=n * 7 * DK * dv)
    if kind == "prefill":
        return _prefill_work(case["B"] * case["T"], case["H"], case["B"], case["dv"], case["state"])
    if kind == "varlen":
        return _prefill_work(sum(_len_list(case)), case["H"], len(_len_list(case)), case["dv"], True)
    if kind == "proj":
        n, Do = case["B"] * case["T"], case["D_out"]
        return dict(bytes=2 * (n * D + Do * D + Do * CK + n * Do), flops=2 * n * D * Do)
    H, dv = 16, case["dv"]
    cols = 2 * H * DK + H * dv
    w_bytes = 2 * (D * (cols + 2 * H) + cols * CK + D * H * dv + D)
    if kind == "layer_decode":
        n = case["B"]
        caches = 2 * 2 * (CK - 1) * (cols + D)
        return dict(bytes=w_bytes + n * (8 * H * DK * dv + caches + 4 * D),
                    flops=n * (2 * D * (cols + 2 * H) + 2 * D * H * dv + 7 * H * DK * dv))
    lens = _len_list(case) if kind == "layer_packed" else [case["T"]] * case["B"]
    n = sum(lens)
    kept = len(lens) * (4 * H * DK * dv + 2 * (CK - 1) * (cols + D)) if case["keep"] else 0
    return dict(bytes=w_bytes + 4 * n * D + kept,
                flops=n * (2 * D * (cols + 2 * H) + 2 * D * H * dv) + _prefill_work(n, H, 0, dv, False)["flops"])


def tolerance(case):
    """Two to four times the distance from exact() that each kind showed over
    its range: relative errors 1e-7 (decode), 1.7e-3 (proj), 3.1e-3
    (layer_decode's y), 3.4e-3 (prefill), 5.7e-3 (layer); largest
    differences 1.3e-6, 4e-3, 1.4e-2, 5.6e-2 and 7.2e-2."""
    kind = case["kind"]
    if kind == "decode":  # fp32 throughout
        return {"rel": 1e-6, "max": 1e-5}
    if kind == "proj":  # fp32 sums, one bf16 rounding of the result
        return {"rel": 7e-3, "max": 2e-2}
    if kind == "layer_decode":  # q, k, v and o rounded to bf16 on the way
        return {"rel": 1e-2, "max": 6e-2}
    if kind in ("prefill", "varlen"):  # the state rounded to bf16 as an operand, chunk by chunk
        return {"rel": 1e-2, "max": 0.25}
    return {"rel": 1.5e-2, "max": 0.25}


# ---------------------------------------------------------------------------
# The same in 64 bits, token by token, in plain torch
# ---------------------------------------------------------------------------
def _recurrence(q, k, v, logg, beta, S, scale):
    """q, k [N, T, K], v [N, T, V], logg, beta [N, T], S [N, K, V], all float64.  Returns (o [N, T, V], S)."""
    g, o = logg.exp(), torch.empty_like(v)
    for t in range(q.shape[1]):
        S = S * g[:, t, None, None]
        r = torch.matmul(k[:, t, None, :], S)[:, 0]
        S = S + k[:, t, :, None] * (beta[:, t, None] * (v[:, t] - r))[:, None, :]
        o[:, t] = torch.matmul(q[:, t, None, :], S)[:, 0] * scale
    return o, S


def _gated(q, k, v, a, b, A_log, dt_bias, mask, S, scale):
    """Head-major [B, H, T, .] inputs: float64 (o [B, H, T, V], S [B, H, K, V]).  Masked tokens decay the state, write nothing and give zeros."""
    B, H, T, V = v.shape
    logg = -A_log.double().exp()[None, :, None] * torch.nn.functional.softplus(a.double() + dt_bias, threshold=60.0)
    beta = torch.sigmoid(b.double())
    if mask is not None:
        beta = beta * mask.double()[:, None, :]
    S = torch.zeros(B, H, DK, V, dtype=torch.float64, device=v.device) if S is None else S.double()
    flat = lambda x: x.double().reshape(B * H, *x.shape[2:])  # noqa: E731
    o, S = _recurrence(flat(q), flat(k), flat(v), flat(logg), flat(beta), S.reshape(B * H, DK, V), scale)
    o = o.reshape(B, H, T, V)
    if mask is not None:
        o = o * mask.double()[:, None, :, None]
    return o, S.reshape(B, H, DK, V)


def _normed(x, gamma):
    x = x.double()
    return x * (x.square().mean(-1, keepdim=True) + 1e-6).rsqrt() * gamma.double()


def _conv_silu(P, conv, before=None):
    """P [B, T, N] float64, conv [N, CK]; `before` [B, CK - 1, N] precedes t = 0 (zeros without)."""
    head = P.new_zeros(P.shape[0], CK - 1, P.shape[2]) if before is None else before
    ext, T = torch.cat([head, P], 1), P.shape[1]
    y = sum(ext[:, j:j + T] * conv[:, j].double() for j in range(CK))
    return torch.nn.functional.silu(y), ext[:, T:]


def _layer_tokens(w, x, dv, mask, before=None, S=None):
    """(y, S, conv caches [B, N, CK - 1], x_n) of B equal-length sequences, in float64."""
    B, T, _ = x.shape
    H = w["A_log"].numel()
    xn = _normed(x, w["norm_gamma"])
    heads, caches = [], []
    for n in "qkv":
        P = xn @ w["W_" + n].double().T
        y, last = _conv_silu(P, w["conv_" + n], None if before is None else before["conv_" + n].double().transpose(1, 2))
        heads.append(y.reshape(B, T, H, -1).transpose(1, 2))
        caches.append(last.transpose(1, 2))
    a, b = ((xn @ w["W_" + n].double().T).transpose(1, 2) for n in "ab")
    o, S = _gated(*heads, a, b, w["A_log"], float(w["dt_bias"]), mask, S, DK ** -0.5)
    y = o.transpose(1, 2).reshape(B, T, H * dv) @ w["W_o"].double().T
    return y, S, caches, xn


def exact(case, seed):
    i, kind = _inputs(case, seed), case["kind"]
    if kind == "decode":
        one = lambda x: x.unsqueeze(2)  # noqa: E731
        logg = -i["A_log"].double().exp() * torch.nn.functional.softplus(i["a"].double() + i["dt_bias"].double(), threshold=60.0)
        n = case["B"] * case["H"]
        f = lambda x: one(x).double().reshape(n, 1, *x.shape[2:])  # noqa: E731
        o, S = _recurrence(f(i["q"]), f(i["k"]), f(i["v"]), f(logg), f(torch.sigmoid(i["b"].double())),
                           i["S"].double().reshape(n, DK, case["dv"]), DK ** -0.5)
        return o.reshape(i["v"].shape), S.reshape(i["S"].shape)
    if kind == "prefill":
        return _gated(i["q"], i["k"], i["v"], i["a"], i["b"], i["A_log"], 0.0, i["mask"], i.get("S"), DK ** -0.5)
    if kind == "varlen":
        os_, Ss, t = [], [], 0
        for n, length in enumerate(_len_list(case)):
            cut = {x: i[x][:, :, t:t + length] for x in ("q", "k", "v", "a", "b")}
            o, S = _gated(cut["q"], cut["k"], cut["v"], cut["a"], cut["b"], i["A_log"], 0.0, None, i["S"][n:n + 1], DK ** -0.5)
            os_.append(o)
            Ss.append(S)
            t += length
        return torch.cat(os_, 2), torch.cat(Ss, 0)
    if kind == "proj":
        return _conv_silu(i["x"].double() @ i["W"].double().T, i["conv"])[0]
    dv = case["dv"]
    if kind == "layer_decode":
        st = i["state"]
        y, S, caches, xn = _layer_tokens(i["w"], i["x"], dv, None, before=st, S=st["recurrent"])
        hist = torch.cat([st["xn"].double()[:, 1:], xn], 1)
        return y, dict(recurrent=S, conv_q=caches[0], conv_k=caches[1], conv_v=caches[2], xn=hist)
    if kind == "layer":
        y, S, caches, xn = _layer_tokens(i["w"], i["x"], dv, i["mask"])
        if not case["keep"]:
            return y
        hist = torch.cat([xn.new_zeros(case["B"], CK - 1, D), xn], 1)[:, case["T"]:]
        return y, dict(recurrent=S, conv_q=caches[0], conv_k=caches[1], conv_v=caches[2], xn=hist)
    got, t = [], 0
    for length in _len_list(case):
        y, S, caches, xn = _layer_tokens(i["w"], i["x"][:, t:t + length], dv, None)
        got.append((y, S, *caches, torch.cat([xn.new_zeros(1, CK - 1, D), xn], 1)[:, length:]))
        t += length
    y = torch.cat([g[0] for g in got], 1)
    if not case["keep"]:
        return y
    cat = [torch.cat([g[j] for g in got], 0) for j in range(1, 6)]
    return y, dict(recurrent=cat[0], conv_q=cat[1], conv_k=cat[2], conv_v=cat[3], xn=cat[4])
