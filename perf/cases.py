"""Performance cases: the work that a program using this package has it do.

The listed cases and the ranges that draw() samples cover both ways into the
package: the instruction Y = X . W^T (+ bias) over resident weights
(Context.linear with host arrays, Context.linear_dev with device pointers), and
the resident models (Model.generate, forward and forward_batch) in the three
model shapes of purebee_amd.synth.CONFIGS.  Weights are GGUF blocks of
N(0, 0.02) matrices, activations N(0, 1) (what an RMSNorm hands on), tokens
uniform.  exact() evaluates the same pass in float64 with plain torch.
"""
import math

import numpy as np
import torch

import purebee_amd as pb
from purebee_amd import native, synth

TYPES = {"q4_0": pb.TYPE_Q4_0, "q4_1": pb.TYPE_Q4_1, "q8_0": pb.TYPE_Q8_0, "q6_k": pb.TYPE_Q6_K,
         "f16": pb.TYPE_F16, "f32": pb.TYPE_F32, "q8_ref": pb.TYPE_Q8_REF}
STD = 0.02


def listed():
    return [
        # One synchronous quantizedMatvec call as the streaming runtime makes it,
        # host arrays in and out: the smallest call, the q / o projection of a
        # 2048-wide model.
        {"name": "matvec_host_q4_0", "kind": "linear", "type": "q4_0", "N": 2048, "K": 2048, "M": 1,
         "bias": False, "host": True},
        # A handful of rows through an FFN matrix: batched single-token requests.
        {"name": "linear_q4_0_m16", "kind": "linear", "type": "q4_0", "N": 8192, "K": 2048, "M": 16,
         "bias": False, "host": False},
        # A prompt's rows through the gate (or up) projection.
        {"name": "linear_q4_0_m512", "kind": "linear", "type": "q4_0", "N": 8192, "K": 2048, "M": 512,
         "bias": False, "host": False},
        # A ragged short prompt through a Q8_0 down projection (long K).
        {"name": "linear_q8_0_m100", "kind": "linear", "type": "q8_0", "N": 2048, "K": 8192, "M": 100,
         "bias": False, "host": False},
        # engine.js LINEAR (tensorMulAdd): f32 weights and a bias.
        {"name": "linear_f32_m512", "kind": "linear", "type": "f32", "N": 2048, "K": 2048, "M": 512,
         "bias": True, "host": False},
        # The Q6_K output matrix of a Q4_0 GGUF file over the rows of a
        # speculative verify.
        {"name": "linear_q6_k_head_m5", "kind": "linear", "type": "q6_k", "N": 128256, "K": 2048, "M": 5,
         "bias": False, "host": False},
        # Interactive decoding: greedy tokens after a short prompt.
        {"name": "decode_llama1b", "kind": "decode", "model": "llama32_1b", "start": 128, "n": 32},
        # The same late in a long conversation.
        {"name": "decode_llama1b_long", "kind": "decode", "model": "llama32_1b", "start": 3500, "n": 32},
        # A prompt, and a long one.
        {"name": "prefill_llama1b_512", "kind": "prefill", "model": "llama32_1b", "start": 0, "n": 512},
        {"name": "prefill_llama1b_2000", "kind": "prefill", "model": "llama32_1b", "start": 0, "n": 2000},
        # The verify of a speculative round: four drafts and the bonus position.
        {"name": "verify_llama1b_m5", "kind": "verify", "model": "llama32_1b", "start": 128, "n": 5},
        # Decoding with a small Q8_0 model (a draft model, an edge model).
        {"name": "decode_smollm2", "kind": "decode", "model": "smollm2_135m", "start": 32, "n": 32},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "decode", "prefill", "prefill", "verify"])
    if kind == "linear":
        t = rng.choice(["q4_0", "q4_0", "q8_0", "q4_1", "q6_k", "f16", "f32", "q8_ref"])
        K = 32 * _log_int(rng, 8, 256)
        if t == "q6_k":
            K = (K + 255) // 256 * 256
        # q8_ref is the single-token path of the quantised llama.js models
        M = rng.choice([1, _log_int(rng, 1, 8), _log_int(rng, 4, 64 if t == "q8_ref" else 700)])
        N = _log_int(rng, 48, 16384)
        return {"kind": kind, "type": t, "N": N, "K": K, "M": M, "bias": rng.random() < 0.3,
                "host": M <= 4 and rng.random() < 0.3}
    model = rng.choice(["llama32_1b", "llama32_1b", "smollm2_135m", "stories15m"])
    top = {"llama32_1b": 3600, "smollm2_135m": 480, "stories15m": 220}[model]
    if kind == "decode":
        return {"kind": kind, "model": model, "start": _log_int(rng, 8, top), "n": rng.randint(4, 32)}
    if kind == "verify":
        return {"kind": kind, "model": model, "start": _log_int(rng, 8, top), "n": rng.randint(2, 9)}
    n = _log_int(rng, 6, min(top, 2000))
    start = rng.choice([0, 0, rng.randint(0, min(top, 2000) - n)])  # a fresh prompt, or a later turn's
    return {"kind": kind, "model": model, "start": start, "n": n}


# ---- inputs ------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _u8(t):
    return t.contiguous().view(torch.uint8)


def _weight_bytes(gen, t, N, K):
    """GGUF bytes of an N x K matrix of N(0, STD), on the GPU: [N, bytes of a row]."""
    if t == "q6_k":
        # codes, 16-element scales and d as they come out for such a matrix
        q = (torch.randn(N, K // 256, 2, 4, 32, device="cuda", generator=gen) * 12).round()
        q = (q.clamp(-32, 31) + 32).to(torch.uint8)  # [half][group][l]: element 128 half + 32 group + l
        ql = torch.cat([(q[:, :, :, 0] & 15) | (q[:, :, :, 2] << 4),
                        (q[:, :, :, 1] & 15) | (q[:, :, :, 3] << 4)], -1).flatten(2)
        qh = ((q[:, :, :, 0] >> 4) | (q[:, :, :, 1] >> 4 << 2) | (q[:, :, :, 2] >> 4 << 4)
              | (q[:, :, :, 3] >> 4 << 6)).flatten(2)
        sc = torch.randint(70, 128, (N, K // 256, 16), device="cuda", generator=gen, dtype=torch.int8)
        d = (STD / 1200 * (0.9 + 0.2 * torch.rand(N, K // 256, 1, device="cuda", generator=gen))).half()
        return torch.cat([ql, qh, _u8(sc), _u8(d)], -1).reshape(N, -1)
    w = torch.randn(N, K, device="cuda", generator=gen) * STD
    if t == "f32":
        return _u8(w)
    if t == "f16":
        return _u8(w.half())
    b = w.view(N, K // 32, 32)
    if t == "q8_0":
        d = (b.abs().amax(-1, keepdim=True) / 127).half()
        q = (b / d.float()).round().clamp(-127, 127).to(torch.int8)
        return torch.cat([_u8(d), _u8(q)], -1).reshape(N, -1)
    if t == "q4_0":
        d = (b.abs().amax(-1, keepdim=True) / 8).half()
        q = ((b / d.float()).round().clamp(-8, 7) + 8).to(torch.uint8)
        head = [_u8(d)]
    else:
        lo = b.amin(-1, keepdim=True).half()
        d = ((b.amax(-1, keepdim=True) - lo.float()) / 15).half()
        q = ((b - lo.float()) / d.float()).round().clamp(0, 15).to(torch.uint8)
        head = [_u8(d), _u8(lo)]
    return torch.cat(head + [q[..., :16] | (q[..., 16:] << 4)], -1).reshape(N, -1)


def _weight_f64(raw, t, N, K):
    """The matrix that those bytes stand for, in float64."""
    if t == "f32":
        return raw.view(torch.float32).view(N, K).double()
    if t == "f16":
        return raw.view(torch.float16).view(N, K).double()
    if t == "q6_k":
        r = raw.view(N, K // 256, 210)
        ql, qh = r[..., :128].unflatten(-1, (2, 2, 32)), r[..., 128:192].unflatten(-1, (2, 1, 32))
        low = torch.cat([ql & 15, ql >> 4], -2)  # groups 0, 1 then 2, 3 of a half
        high = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], -2)
        q = (low | (high << 4)).double() - 32
        sc = r[..., 192:208].contiguous().view(torch.int8).double()
        d = r[..., 208:].contiguous().view(torch.float16).double()
        return (q.reshape(N, K // 256, 16, 16) * (sc * d).unsqueeze(-1)).reshape(N, K)
    nb = {"q8_0": 34, "q4_0": 18, "q4_1": 20}[t]
    r = raw.view(N, K // 32, nb)
    d = r[..., :2].contiguous().view(torch.float16).double()
    if t == "q8_0":
        return (r[..., 2:].contiguous().view(torch.int8).double() * d).view(N, K)
    c = r[..., nb - 16:]
    q = torch.cat([c & 15, c >> 4], -1).double()
    if t == "q4_0":
        return ((q - 8) * d).view(N, K)
    return (q * d + r[..., 2:4].contiguous().view(torch.float16).double()).view(N, K)


def _linear_inputs(case, seed):
    """(weight bytes or (codes, scales), X, bias) on the GPU."""
    g = _generator(seed)
    M, N, K = case["M"], case["N"], case["K"]
    if case["type"] == "q8_ref":
        w = torch.randn(K * N, device="cuda", generator=g) * STD
        w = torch.nn.functional.pad(w, (0, -(K * N) % 32)).view(-1, 32)
        s = w.abs().amax(-1) / 127
        raw = ((w / s[:, None]).round().to(torch.int8).view(-1)[:K * N], s)
    else:
        raw = _weight_bytes(g, case["type"], N, K)
    x = torch.randn(M, K, device="cuda", generator=g)
    bias = torch.randn(N, device="cuda", generator=g) if case["bias"] else None
    return raw, x, bias


def _config(case):
    """The model shape of a case, with cache room for its positions."""
    cfg = dict(synth.CONFIGS[case["model"]])
    cfg["max_seq"] = max(cfg["max_seq"], (case["start"] + case["n"] + 1 + 1023) // 1024 * 1024)
    return cfg


NAMES = {v: k for k, v in TYPES.items()}
NORMS = (native.T_OUTPUT_NORM, native.T_ATTN_NORM, native.T_FFN_NORM)


def _model_tensors(case, seed):
    """(tensor id, layer, type, N, K, bytes on the GPU) of every tensor, in load order."""
    g = _generator(seed)
    for tid, layer, N, K, t in synth.tensor_specs(_config(case)):
        if tid in NORMS:  # trained norm weights lie around 1
            yield tid, layer, "f32", N, K, _u8(1 + 0.1 * torch.randn(N, K, device="cuda", generator=g))
        else:
            yield tid, layer, NAMES[t], N, K, _weight_bytes(g, NAMES[t], N, K)


def _tokens(case, seed):
    """(the prompt before the pass, the tokens of the pass)."""
    vocab = synth.CONFIGS[case["model"]]["vocab_size"]
    g = np.random.default_rng(int(seed) + 1)
    return (g.integers(0, vocab, case["start"]).astype(np.int32),
            g.integers(0, vocab, case["n"]).astype(np.int32))


# ---- the cases ---------------------------------------------------------------

_ctx = None


class _State:
    """What a program holds on to; gives its device memory back when dropped."""

    def __init__(self, case):
        global _ctx
        if _ctx is None:
            _ctx = pb.Context(0)
        self.ctx, self.case = _ctx, case
        self.weight = self.model = None

    def __del__(self):
        if self.weight is not None:
            self.weight.free()
        if self.model is not None:
            self.model.free()


def prepare(case, seed):
    s = _State(case)
    if case["kind"] == "linear":
        raw, x, bias = _linear_inputs(case, seed)
        if case["type"] == "q8_ref":
            s.weight = s.ctx.upload_q8ref(case["K"], case["N"], raw[0].cpu().numpy(), raw[1].cpu().numpy())
        else:
            s.weight = s.ctx.upload(TYPES[case["type"]], case["N"], case["K"], raw.cpu().numpy())
        if case["host"]:
            s.x = (x[0] if case["M"] == 1 else x).cpu().numpy()
            s.bias = None if bias is None else bias.cpu().numpy()
        else:
            s.x, s.bias = x, bias
            s.y = torch.empty(case["M"], case["N"], device="cuda")
        torch.cuda.synchronize()  # the context works on a stream of its own
        return s
    cfg = _config(case)
    s.model = pb.Model(s.ctx, cfg["dim"], cfg["hidden_dim"], cfg["n_layers"], cfg["n_heads"],
                       cfg["n_kv_heads"], cfg["vocab_size"], cfg["max_seq"], cfg["weight_type"],
                       cfg["embed_type"], rope_theta=cfg["rope_theta"])
    for tid, layer, t, N, K, raw in _model_tensors(case, seed):
        s.model.set_tensor(tid, layer, raw.cpu().numpy())
    prompt, s.tokens = _tokens(case, seed)
    if len(prompt):
        s.model.forward(prompt, 0, want_logits=False)
    return s


def run(s):
    c = s.case
    if c["kind"] == "linear":
        if c["host"]:
            return s.ctx.linear(s.weight, s.x, s.bias)
        s.ctx.linear_dev(s.weight, s.x.data_ptr(), c["M"], s.y.data_ptr(),
                         None if s.bias is None else s.bias.data_ptr())
        return s.y
    if c["kind"] == "decode":
        return s.model.generate(s.tokens[0], c["start"], c["n"], want_logits=True)
    if c["kind"] == "prefill":
        return s.model.forward(s.tokens, c["start"])
    return s.model.forward_batch(s.tokens, c["start"])


def _row_bytes(t, K):
    return K * 34 // 32 if t == "q8_ref" else native.row_bytes(TYPES[t], K)


def work(case):
    if case["kind"] == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": N * _row_bytes(case["type"], K) + 4 * M * (N + K) + (4 * N if case["bias"] else 0),
                "flops": 2 * M * N * K}
    cfg = _config(case)
    d, h, L, V = cfg["dim"], cfg["hidden_dim"], cfg["n_layers"], cfg["vocab_size"]
    kv = d // cfg["n_heads"] * cfg["n_kv_heads"]
    params = L * (2 * d * d + 2 * kv * d + 3 * h * d)
    layers = params // 32 * native.block_bytes(cfg["weight_type"])
    head = V * native.row_bytes(cfg["embed_type"], d)
    a, n = case["start"], case["n"]
    pairs = sum(range(a + 1, a + n + 1))  # (query, visible key) pairs
    attention = L * 4 * d * pairs
    if case["kind"] == "decode":  # every step reads the weights and the cache up to its position
        return {"bytes": n * (layers + head) + L * 8 * kv * (pairs + n) + 4 * V,
                "flops": 2 * n * (params + V * d) + attention}
    rows = 1 if case["kind"] == "prefill" else n  # rows that take the head
    return {"bytes": layers + head + L * 8 * kv * (a + n) + 4 * V * rows,
            "flops": 2 * (n * params + rows * V * d) + attention}


def tolerance(case):
    """32-bit sums of exact weights and activations of 22 bits and more (up to 5e-7
    off exact() here); over the 16 or 30 layers of a whole model such roundings
    travel on and add up (up to 4.4e-6)."""
    if case["kind"] == "linear":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 3e-5, "max": 3e-4, "differ": 0.01}


def _exact_model(case, seed):
    """The reference's forward pass (RMSNorm, rotation of adjacent pairs, causal
    grouped-query attention, SwiGLU, tied head) in float64."""
    cfg = _config(case)
    d, H, G = cfg["dim"], cfg["n_heads"], cfg["n_kv_heads"]
    hd, total = d // H, case["start"] + case["n"]
    W = {}
    for tid, layer, t, N, K, raw in _model_tensors(case, seed):
        W[tid, layer] = _weight_f64(raw, t, N, K)
    ang = (torch.arange(total, device="cuda").double()[:, None]
           * cfg["rope_theta"] ** (-torch.arange(0, hd, 2, device="cuda").double() / hd))
    cos, sin = ang.cos(), ang.sin()
    cache = [[torch.empty(total, G, hd, device="cuda", dtype=torch.float64) for _ in range(2)]
             for _ in range(cfg["n_layers"])]

    def norm(x, w):
        return x / (x.square().mean(-1, keepdim=True) + 1e-5).sqrt() * w

    def rotate(x, a):
        c, s = cos[a:a + len(x), None], sin[a:a + len(x), None]
        u, v = x[..., 0::2], x[..., 1::2]
        return torch.stack([u * c - v * s, u * s + v * c], -1).flatten(-2)

    def layer(x, l, a):
        n = len(x)
        y = norm(x, W[native.T_ATTN_NORM, l])
        q = rotate((y @ W[native.T_ATTN_Q, l].T).view(n, H, hd), a)
        k, v = cache[l]
        k[a:a + n] = rotate((y @ W[native.T_ATTN_K, l].T).view(n, G, hd), a)
        v[a:a + n] = (y @ W[native.T_ATTN_V, l].T).view(n, G, hd)
        hidden = torch.arange(a + n, device="cuda")[None] > torch.arange(a, a + n, device="cuda")[:, None]
        o = torch.empty(n, H, hd, device="cuda", dtype=torch.float64)
        for h in range(H):
            s = q[:, h] @ k[:a + n, h * G // H].T / math.sqrt(hd)
            o[:, h] = s.masked_fill(hidden, -math.inf).softmax(-1) @ v[:a + n, h * G // H]
        x = x + o.view(n, d) @ W[native.T_ATTN_OUTPUT, l].T
        y = norm(x, W[native.T_FFN_NORM, l])
        u = torch.nn.functional.silu(y @ W[native.T_FFN_GATE, l].T) * (y @ W[native.T_FFN_UP, l].T)
        return x + u @ W[native.T_FFN_DOWN, l].T

    def forward(tokens, a):
        """The rows that enter the head."""
        x = W[native.T_TOKEN_EMBD, -1][torch.as_tensor(tokens, device="cuda").long()]
        for l in range(cfg["n_layers"]):
            x = layer(x, l, a)
        return norm(x, W[native.T_OUTPUT_NORM, -1])

    head = W[native.T_TOKEN_EMBD, -1].T
    prompt, tokens = _tokens(case, seed)
    if len(prompt):
        forward(prompt, 0)
    if case["kind"] == "verify":
        return forward(tokens, case["start"]) @ head, None
    if case["kind"] == "prefill":
        return forward(tokens, case["start"])[-1] @ head, None
    tok = tokens[:1]
    for i in range(case["n"]):
        logits = forward(tok, case["start"] + i)[-1] @ head
        tok = logits.argmax()[None]
    return None, logits


def exact(case, seed):
    if case["kind"] != "linear":
        return _exact_model(case, seed)
    raw, x, bias = _linear_inputs(case, seed)
    N, K = case["N"], case["K"]
    if case["type"] == "q8_ref":
        w = raw[0].double() * raw[1].double().repeat_interleave(32)[:K * N]
        y = x.double() @ w.view(K, N)
    else:
        y = x.double() @ _weight_f64(raw, case["type"], N, K).T
    if bias is not None:
        y += bias.double()
    return y[0] if case["host"] and case["M"] == 1 else y
