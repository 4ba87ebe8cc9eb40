"""The work a program gives this framework, as measurable cases.

A program prefills Qwen2.5 / Qwen3 text models: it launches the decoder
layer's operators on device memory it owns (kernrelay_amd.ops), or hands a
model directory to the prefill runtime (libapi.qwen_run), or a schedule of
producer GEMMs and their consumers to the DAG executor (libapi.plan_run).

* layer: one decoder layer's operator sequence, prompts of 16 to 4096 tokens
  at the three shipped model shapes, on buffers kept from call to call;
* gemm: one projection by itself (any of a layer's, or lm_head over all
  rows), bf16 or fp16, with and without bias;
* attention: causal attention of a whole prompt by itself, up to 8192 tokens;
* consumers: the fp16 producer GEMM and its GELU, softmax and cast consumers
  (the relay workloads' shapes);
* relay_norm: the o / down projection releasing row tiles to its own
  Add+RMSNorm;
* plan: a schedule through the DAG executor, from files to files;
* prefill: a short model through the prefill runtime, from the model
  directory to the last row's logits.

Inputs: activations N(0, 1), weights and biases N(0, 0.02), norm gains
1 + N(0, 0.02), uniform token ids (kernrelay_amd.modeldir writes the same).
"""

import os
import sys
import tempfile
from pathlib import Path

import numpy as np
import torch

from kernrelay_amd import dag_bench, libapi, modeldir, ops, schedule, workloads

MODELS = ("qwen2.5-0.5b", "qwen2.5-7b", "qwen3-8b")
EPS = 1e-6
DT = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # a short chat turn on the small model: every launch is tiny
        dict(name="layer_0.5b_s37", kind="layer", model="qwen2.5-0.5b", S=37),
        # an odd, ordinary prompt on the small model (head size 64, split-K down)
        dict(name="layer_0.5b_s1001", kind="layer", model="qwen2.5-0.5b", S=1001),
        # a question to the 7B model: weights are read for few rows
        dict(name="layer_7b_s200", kind="layer", model="qwen2.5-7b", S=200),
        # the benchmarked prefill's layer
        dict(name="layer_7b_s2048", kind="layer", model="qwen2.5-7b", S=2048),
        # the longest configured prompt, q/k norms, separate q/k/v projections
        dict(name="layer_8b_s4096", kind="layer", model="qwen3-8b", S=4096),
        # logits of every row of a medium prompt
        dict(name="lm_head_0.5b_s515", kind="gemm", model="qwen2.5-0.5b", op="lm_head", S=515, dtype="bf16",
             bias=False),
        # fused q/k/v projection of an fp16 caller
        dict(name="qkv_8b_s1111_fp16", kind="gemm", model="qwen3-8b", op="qkv", S=1111, dtype="fp16", bias=True),
        # a long document's attention
        dict(name="attention_7b_s8192", kind="attention", model="qwen2.5-7b", S=8192, dtype="bf16"),
        # the relay workloads' GEMM and its three consumers, at half their rows
        dict(name="consumers_s16384", kind="consumers", S=16384, K=1024, N=2048),
        # o projection + Add+RMSNorm in one launch, four relay tiles
        dict(name="relay_norm_7b_s1024", kind="relay_norm", model="qwen2.5-7b", op="o", S=1024, k=4),
        # a split schedule through the executor
        dict(name="plan_fanout_1024", kind="plan", M=1024, K=512, N=1024, k=4),
        # a four-layer model from its directory to its logits
        dict(name="prefill_l4_s300", kind="prefill", layers=4, vocab=16384, S=300),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("layer", "layer", "layer", "gemm", "gemm", "attention", "consumers", "relay_norm", "plan",
                       "prefill"))
    model = rng.choice(MODELS)
    if kind == "layer":
        return dict(kind=kind, model=model, S=_log_int(rng, 16, 4096))
    if kind == "gemm":
        op = rng.choice(("qkv", "o", "gate_up", "down", "lm_head"))
        return dict(kind=kind, model=model, op=op, S=_log_int(rng, 16, 1024 if op == "lm_head" else 4096),
                    dtype=rng.choice(("bf16", "fp16")), bias=op == "qkv")
    if kind == "attention":
        return dict(kind=kind, model=model, S=_log_int(rng, 64, 8192), dtype=rng.choice(("bf16", "fp16")))
    if kind == "consumers":
        return dict(kind=kind, S=_log_int(rng, 128, 32768), K=8 * rng.randint(32, 256), N=8 * rng.randint(32, 256))
    if kind == "relay_norm":
        k = rng.choice((1, 2, 4))
        return dict(kind=kind, model=model, op=rng.choice(("o", "down")), S=64 * k * rng.randint(1, 16 // k), k=k)
    if kind == "plan":
        k = rng.choice((1, 2, 4))
        return dict(kind=kind, M=64 * k * rng.randint(2, 12), K=64 * rng.randint(4, 16), N=128 * rng.randint(2, 12),
                    k=k)
    return dict(kind="prefill", layers=rng.randint(2, 4), vocab=16384, S=_log_int(rng, 16, 1024))


# ------------------------------------------------------------------- helpers
class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
        return torch.empty(*shape, device="cuda").normal_(mean, std, generator=self.g).to(dtype)


def _cfg(model):
    c = modeldir.PRESETS[model]
    return dict(H=c["hidden_size"], I=c["intermediate_size"], HQ=c["num_attention_heads"],
                HKV=c["num_key_value_heads"], D=c["head_dim"], V=c["vocab_size"], qk_norm=c["qk_norm"],
                theta=c["rope_theta"])


def _gemm_dims(case):
    c = _cfg(case["model"])
    return {"qkv": ((c["HQ"] + 2 * c["HKV"]) * c["D"], c["H"]), "o": (c["H"], c["HQ"] * c["D"]),
            "gate_up": (2 * c["I"], c["H"]), "down": (c["H"], c["I"]), "lm_head": (c["V"], c["H"])}[case["op"]]


class _Linear:
    """A projection as the prefill runtime keeps it: weight [N, K], output
    buffer, and the split-K workspace the library asks for (if any)."""

    def __init__(self, gen, M, N, K, bias=False, dtype=torch.bfloat16):
        self.w = gen.normal(N, K, std=0.02, dtype=dtype)
        self.b = gen.normal(N, std=0.02, dtype=dtype) if bias else None
        self.y = torch.empty(M, N, dtype=dtype, device="cuda")
        nbytes, ncnt = ops.gemm_streamk_workspace(M, N, K)
        self.ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda") if nbytes else None
        self.cnt = torch.zeros(ncnt, dtype=torch.int32, device="cuda") if nbytes else None

    def __call__(self, x):
        if self.ws is not None:
            ops.gemm_streamk(x, self.w, self.y, self.ws, self.cnt, bias=self.b)
        else:
            ops.gemm(x, self.w, self.y, bias=self.b)
        return self.y


class _Attention:
    def __init__(self, S, HQ, HKV, D, dtype=torch.bfloat16):
        self.dims = (S, HQ, HKV, D)
        self.y = torch.empty(S, HQ * D, dtype=dtype, device="cuda")
        nbytes, ncnt = ops.attention_workspace(S, HQ, D)
        self.ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda") if nbytes else None
        self.cnt = torch.zeros(ncnt, dtype=torch.int32, device="cuda") if nbytes else None

    def __call__(self, q, k, v):
        ld = dict(ldq=q.stride(0), ldk=k.stride(0), ldv=v.stride(0))
        if self.ws is not None:
            ops.attention_split(q, k, v, self.y, *self.dims, self.ws, self.cnt, **ld)
        else:
            ops.attention(q, k, v, self.y, *self.dims, **ld)
        return self.y


def _rope(S, D, theta):
    cos, sin = modeldir.rope_table(S, D, theta)
    return cos.reshape(S, D).cuda(), sin.reshape(S, D).cuda()


# --------------------------------------------------------------------- layer
class _Layer:
    def __init__(self, gen, model, S):
        c = self.c = _cfg(model)
        H, I, HQ, HKV, D = c["H"], c["I"], c["HQ"], c["HKV"], c["D"]
        self.S = S
        self.h = gen.normal(S, H)
        self.g1, self.g2, self.g3 = (gen.normal(H, std=0.02, mean=1.0) for _ in range(3))
        if c["qk_norm"]:
            self.q, self.k, self.v = (_Linear(gen, S, n * D, H) for n in (HQ, HKV, HKV))
            self.gq, self.gk = (gen.normal(D, std=0.02, mean=1.0) for _ in range(2))
            self.qn = torch.empty(S, HQ * D, dtype=torch.bfloat16, device="cuda")
            self.kn = torch.empty(S, HKV * D, dtype=torch.bfloat16, device="cuda")
        else:
            self.qkv = _Linear(gen, S, (HQ + 2 * HKV) * D, H, bias=True)
        self.attn = _Attention(S, HQ, HKV, D)
        self.o = _Linear(gen, S, H, HQ * D)
        self.gu = gen.normal(2 * I, H, std=0.02)
        self.down = _Linear(gen, S, H, I)
        self.cos, self.sin = _rope(S, D, c["theta"])
        new = lambda n: torch.empty(S, n, dtype=torch.bfloat16, device="cuda")  # noqa: E731
        self.x1, self.x2, self.x3, self.h1, self.h2, self.act = new(H), new(H), new(H), new(H), new(H), new(I)

    def run(self):
        c, S = self.c, self.S
        HQ, HKV, D = c["HQ"], c["HKV"], c["D"]
        ops.rowop("rmsnorm", self.h, self.x1, gamma=self.g1, eps=EPS)
        if c["qk_norm"]:
            ops.rowop("rmsnorm", self.q(self.x1).view(S * HQ, D), self.qn.view(S * HQ, D), gamma=self.gq, eps=EPS)
            ops.rowop("rmsnorm", self.k(self.x1).view(S * HKV, D), self.kn.view(S * HKV, D), gamma=self.gk, eps=EPS)
            q, k, v = self.qn, self.kn, self.v(self.x1)
        else:
            qkv = self.qkv(self.x1)
            q, k, v = qkv[:, :HQ * D], qkv[:, HQ * D:(HQ + HKV) * D], qkv[:, (HQ + HKV) * D:]
        ops.rope(q, S, HQ, D, self.cos, self.sin, ld=q.stride(0))
        ops.rope(k, S, HKV, D, self.cos, self.sin, ld=k.stride(0))
        o = self.o(self.attn(q, k, v))
        ops.rowop("add_rmsnorm", self.h, self.x2, x1=o, gamma=self.g2, sum_out=self.h1, eps=EPS)
        ops.gemm_swiglu_epilogue(self.x2, self.gu, self.act)
        ops.rowop("add_rmsnorm", self.h1, self.x3, x1=self.down(self.act), gamma=self.g3, sum_out=self.h2, eps=EPS)
        return {"hidden": self.h2, "normed": self.x3, "k": k, "v": v}


def _rms64(x, g):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * g


def _rope64(x, cos, sin):  # x [S, heads, D]
    half = x.shape[-1] // 2
    rot = torch.cat([-x[..., half:], x[..., :half]], dim=-1)
    return x * cos[:, None, :] + rot * sin[:, None, :]


def _attention64(q, k, v):  # [S, HQ, D], [S, HKV, D] float64
    S, HQ, D = q.shape
    group = HQ // k.shape[1]
    out = torch.empty_like(q)
    for h in range(HQ):
        kt = k[:, h // group].t().contiguous()
        vh = v[:, h // group].contiguous()
        for lo in range(0, S, 2048):
            hi = min(lo + 2048, S)
            s = (q[lo:hi, h].contiguous() @ kt[:, :hi]) * D ** -0.5
            keys = torch.arange(hi, device=q.device)
            s.masked_fill_(keys[None, :] > torch.arange(lo, hi, device=q.device)[:, None], float("-inf"))
            out[lo:hi, h] = torch.softmax(s, dim=-1) @ vh[:hi]
    return out


def _mm64(x, w):
    """x @ w^T in float64, the weight converted a block of rows at a time."""
    return torch.cat([x @ w[lo:lo + 16384].double().t() for lo in range(0, w.shape[0], 16384)], dim=1)


def _layer64(c, h, q, k, v, gq, gk, cos, sin, wo, g1, g2, wg, wu, wd):
    """One decoder layer in float64 from weights [N, K]; q, k, v are
    (weight, bias) pairs. Returns the residual after it, its k and v."""
    S, D = h.shape[0], c["D"]
    x = _rms64(h, g1.double())
    lin = lambda wb: _mm64(x, wb[0]) + (wb[1].double() if wb[1] is not None else 0.0)  # noqa: E731
    qq, kk, vv = lin(q).view(S, -1, D), lin(k).view(S, -1, D), lin(v).view(S, -1, D)
    if gq is not None:
        qq, kk = _rms64(qq, gq.double()), _rms64(kk, gk.double())
    qq, kk = _rope64(qq, cos.double(), sin.double()), _rope64(kk, cos.double(), sin.double())
    h = h + _mm64(_attention64(qq, kk, vv).reshape(S, -1), wo)
    x = _rms64(h, g2.double())
    return h + _mm64(torch.nn.functional.silu(_mm64(x, wg)) * _mm64(x, wu), wd), kk.reshape(S, -1), vv.reshape(S, -1)


def _exact_layer(L):
    c = L.c
    HQ, HKV, D = c["HQ"], c["HKV"], c["D"]
    if c["qk_norm"]:
        q, k, v = (L.q.w, None), (L.k.w, None), (L.v.w, None)
        gq, gk = L.gq, L.gk
    else:
        cut = [HQ * D, HKV * D, HKV * D]
        q, k, v = zip(L.qkv.w.split(cut), L.qkv.b.split(cut))
        gq = gk = None
    gu = L.gu.view(c["I"] // 8, 2, 8, c["H"])
    h, kk, vv = _layer64(c, L.h.double(), q, k, v, gq, gk, L.cos, L.sin, L.o.w, L.g1, L.g2,
                         gu[:, 0].reshape(c["I"], -1), gu[:, 1].reshape(c["I"], -1), L.down.w)
    return {"hidden": h, "normed": _rms64(h, L.g3.double()), "k": kk, "v": vv}


# ------------------------------------------------------------------- prefill
def _prefill_config(case):
    c = dict(modeldir.PRESETS["qwen2.5-0.5b"])
    c.update(num_hidden_layers=case["layers"], vocab_size=case["vocab"])
    return c


def _prefill_dir(case, seed):
    base = "/dev/shm" if os.path.isdir("/dev/shm") else None
    tmp = tempfile.TemporaryDirectory(prefix="kr_perf_", dir=base)
    modeldir.write_model_dir(tmp.name, _prefill_config(case), seq=case["S"], seed=seed, max_pos=1024, device="cuda")
    return tmp


def _run_prefill(state):
    path = state["dir"].name
    os.environ["KR_DUMP_DIR"] = path
    try:
        r = libapi.qwen_run(path, mode="graph_whole", seq=state["S"], warmup=0, iters=1)
    finally:
        del os.environ["KR_DUMP_DIR"]
    if r["_rc"] != 0:
        raise RuntimeError("kr_qwen_run: %s" % r.get("error"))
    raw = np.fromfile(path + "/last_logits_bf16.bin", dtype=np.uint16)
    return {"logits": (raw.astype(np.uint32) << 16).view(np.float32)}


def _exact_prefill(case, seed):
    import json
    cfg = _prefill_config(case)
    tmp = _prefill_dir(case, seed)
    root = Path(tmp.name)
    tensors = json.loads((root / "manifest.json").read_text())["tensors"]
    data = np.fromfile(root / "weights.bin", dtype=np.int16)

    def get(name):
        t = tensors[name]
        a = torch.from_numpy(data[t["offset"] // 2:(t["offset"] + t["bytes"]) // 2].copy())
        return a.view(torch.bfloat16).reshape(t["shape"]).cuda()

    def proj(name):  # [K, N] in the file
        return get(name + ".weight_t").t().contiguous()

    S, D = case["S"], cfg["head_dim"]
    ids = torch.from_numpy(np.fromfile(root / "ids.bin", dtype=np.int64)).cuda()[:S]
    h = get("embed.weight")[ids].double()
    cos, sin = get("rope.cos").reshape(-1, D)[:S], get("rope.sin").reshape(-1, D)[:S]
    for i in range(cfg["num_hidden_layers"]):
        p = "L%02d." % i
        qkv = [(proj(p + n), get(p + n + ".bias")) for n in ("q_proj", "k_proj", "v_proj")]
        h, _, _ = _layer64(dict(D=D), h, *qkv, None, None, cos, sin, proj(p + "o_proj"),
                           get(p + "input_layernorm.weight"), get(p + "post_attention_layernorm.weight"),
                           proj(p + "gate_proj"), proj(p + "up_proj"), proj(p + "down_proj"))
    x = _rms64(h[-1:], get("final_norm.weight").double())
    return {"logits": _mm64(x, proj("lm_head")).reshape(-1).cpu().numpy()}


# ---------------------------------------------------------------------- plan
_PLAN_CONSUMERS = ("softmax", "gelu", "cast")


def _plan_state(case, seed):
    tmp = tempfile.TemporaryDirectory(prefix="kr_perf_")
    M, K, N = case["M"], case["K"], case["N"]
    inputs = workloads.write_inputs(tmp.name, M, K, N, seed)
    dag = schedule.dag_from_dict(workloads.mm_consumers_dag("fanout", M, K, N, _PLAN_CONSUMERS, inputs=inputs))
    path = schedule.dump_schedule(workloads.variants(dag, case["k"])["split"], Path(tmp.name) / "schedule.json")
    return dict(dir=tmp, path=path, inputs=inputs, M=M, K=K, N=N)


def _run_plan(state):
    root = Path(state["dir"].name)
    os.environ["KR_DUMP_DIR"] = str(root)
    try:
        with dag_bench._stdout_to_stderr():  # the executor prints its result line
            r = libapi.plan_run(state["path"], mode="graph_per_stream", iters=1, warmup=0, out_json=root / "out.json")
    finally:
        del os.environ["KR_DUMP_DIR"]
    if r["_rc"] != 0 or not r["ok"]:
        raise RuntimeError("kr_plan_run: %s" % r)
    out = {}
    for name in _PLAN_CONSUMERS:
        raw = np.fromfile(root / (name + ".bin"), dtype=np.uint16)
        out[name] = raw.view(np.float16) if name == "cast" else (raw.astype(np.uint32) << 16).view(np.float32)
    return out


# ------------------------------------------------------------------ the file
def prepare(case, seed):
    kind = case["kind"]
    if kind == "plan":
        return dict(kind=kind, **_plan_state(case, seed))
    if kind == "prefill":
        return dict(kind=kind, dir=_prefill_dir(case, seed), S=case["S"])
    gen = _Gen(seed)
    if kind == "layer":
        return dict(kind=kind, layer=_Layer(gen, case["model"], case["S"]))
    if kind == "gemm":
        N, K = _gemm_dims(case)
        dt = DT[case["dtype"]]
        return dict(kind=kind, x=gen.normal(case["S"], K, dtype=dt),
                    lin=_Linear(gen, case["S"], N, K, case["bias"], dt))
    if kind == "attention":
        c = _cfg(case["model"])
        S, HQ, HKV, D = case["S"], c["HQ"], c["HKV"], c["D"]
        dt = DT[case["dtype"]]
        qkv = gen.normal(S, (HQ + 2 * HKV) * D, dtype=dt)
        return dict(kind=kind, q=qkv[:, :HQ * D], k=qkv[:, HQ * D:(HQ + HKV) * D], v=qkv[:, (HQ + HKV) * D:],
                    attn=_Attention(S, HQ, HKV, D, dt))
    if kind == "consumers":
        S, K, N = case["S"], case["K"], case["N"]
        f16 = torch.float16
        st = dict(kind=kind, x=gen.normal(S, K, dtype=f16), w=gen.normal(N, K, std=0.02, dtype=f16))
        st.update({n: torch.empty(S, N, dtype=f16, device="cuda") for n in ("mm", "gelu", "softmax")})
        st["cast"] = torch.empty(S, N, dtype=torch.float32, device="cuda")
        return st
    N, K = _gemm_dims(case)  # relay_norm
    S, bf = case["S"], torch.bfloat16
    return dict(kind=kind, x=gen.normal(S, K), lin=_Linear(gen, S, N, K), res=gen.normal(S, N),
                gamma=gen.normal(N, std=0.02, mean=1.0), y=torch.empty(S, N, dtype=bf, device="cuda"),
                sum=torch.empty(S, N, dtype=bf, device="cuda"), rows=S // case["k"],
                ctrl=torch.zeros(case["k"] * ops.CTRL_WORDS, dtype=torch.int32, device="cuda"))


def run(state):
    kind = state["kind"]
    if kind == "layer":
        return state["layer"].run()
    if kind == "gemm":
        return {"y": state["lin"](state["x"])}
    if kind == "attention":
        return {"o": state["attn"](state["q"], state["k"], state["v"])}
    if kind == "consumers":
        ops.gemm(state["x"], state["w"], state["mm"])
        ops.elementwise("gelu", state["mm"], state["gelu"])
        ops.rowop("softmax", state["mm"], state["softmax"])
        ops.elementwise("cast", state["mm"], state["cast"])
        return {n: state[n] for n in ("mm", "gelu", "softmax", "cast")}
    if kind == "relay_norm":
        lin = state["lin"]
        ops.gemm_add_rmsnorm(state["x"], lin.w, lin.y, state["res"], state["gamma"], state["y"],
                             ops.make_pub(state["ctrl"], 0, state["rows"]), sum_out=state["sum"], eps=EPS, ws=lin.ws,
                             counters=lin.cnt)
        return {"c": lin.y, "sum": state["sum"], "normed": state["y"]}
    if kind == "plan":
        return _run_plan(state)
    return _run_prefill(state)


def exact(case, seed):
    kind = case["kind"]
    if kind == "prefill":
        return _exact_prefill(case, seed)
    st = prepare(case, seed)
    if kind == "layer":
        return _exact_layer(st["layer"])
    if kind == "gemm":
        y = _mm64(st["x"].double(), st["lin"].w)
        return {"y": y if st["lin"].b is None else y + st["lin"].b.double()}
    if kind == "attention":
        S, HQ, HKV, D = st["attn"].dims
        q, k, v = (st[n].double().reshape(S, -1, D) for n in "qkv")
        return {"o": _attention64(q, k, v).reshape(S, -1)}
    if kind == "relay_norm":
        y = _mm64(st["x"].double(), st["lin"].w)
        s = y + st["res"].double()
        return {"c": y, "sum": s, "normed": _rms64(s, st["gamma"].double())}
    if kind == "consumers":
        y = _mm64(st["x"].double(), st["w"])
    else:
        x, w = (torch.from_numpy(np.fromfile(st["inputs"][n], dtype=np.int16)).cuda().view(torch.bfloat16).double()
                for n in ("in", "b"))
        y = x.view(st["M"], st["K"]) @ w.view(st["K"], st["N"])
    out = {"mm": y, "gelu": torch.nn.functional.gelu(y, approximate="tanh"), "softmax": torch.softmax(y, dim=-1),
           "cast": y}
    if kind == "consumers":
        return out
    return {n: out[n].reshape(-1).cpu().numpy() for n in _PLAN_CONSUMERS}


def _attn_work(S, HQ, HKV, D):
    return dict(bytes=2 * S * D * 2 * (HQ + HKV), flops=2 * 2 * (S * (S + 1) // 2) * HQ * D)


def work(case):
    kind = case["kind"]
    if kind == "plan":
        M, K, N = case["M"], case["K"], case["N"]
        return dict(bytes=2 * (M * K + K * N + 3 * M * N), flops=2 * M * N * K)
    if kind == "consumers":
        M, K, N = case["S"], case["K"], case["N"]
        return dict(bytes=2 * (M * K + K * N) + (2 + 2 + 2 + 4) * M * N, flops=2 * M * N * K)
    if kind == "prefill":
        c, S, V = _cfg("qwen2.5-0.5b"), case["S"], case["vocab"]
        one = work(dict(kind="layer", model="qwen2.5-0.5b", S=S))
        params = (c["HQ"] + 2 * c["HKV"]) * c["D"] * c["H"] + c["HQ"] * c["D"] * c["H"] + 3 * c["H"] * c["I"]
        # the model directory is read whole; logits of every row are computed
        return dict(bytes=2 * (case["layers"] * params + 2 * V * c["H"]),
                    flops=case["layers"] * one["flops"] + 2 * S * V * c["H"])
    if kind in ("gemm", "relay_norm"):
        N, K = _gemm_dims(case)
        M = case["S"]
        extra = 3 * M * N if kind == "relay_norm" else 0
        return dict(bytes=2 * (M * K + N * K + M * N + extra), flops=2 * M * N * K)
    c, S = _cfg(case["model"]), case["S"]
    attn = _attn_work(S, c["HQ"], c["HKV"], c["D"])
    if kind == "attention":
        return attn
    H, I, NQ = c["H"], c["I"], (c["HQ"] + 2 * c["HKV"]) * c["D"]
    params = NQ * H + c["HQ"] * c["D"] * H + 3 * H * I
    # weights, the residual in and out, the normed rows out, k and v out
    return dict(bytes=2 * (params + 3 * S * H + 2 * S * c["HKV"] * c["D"]), flops=2 * S * params + attn["flops"])


def tolerance(case):
    """About four times the relative error measured against `exact`."""
    kind = case["kind"]
    if kind == "prefill":
        return {"rel": 6e-2}
    if kind == "layer":
        return {"rel": 2e-2}
    if kind in ("consumers",) or case.get("dtype") == "fp16":
        return {"rel": 1e-3}
    return {"rel": 1e-2}


if __name__ == "__main__":
    # relative error of one pass of every case against `exact`
    import random
    cases = listed() + [draw(random.Random(int(a))) for a in sys.argv[1:]]
    for case in cases:
        print(case, flush=True)
        st = prepare(case, 1)
        got, ref = run(st), exact(case, 1)
        for key in ref:
            a, b = (torch.as_tensor(t).double().reshape(-1).cuda() for t in (got[key], ref[key]))
            d = a - b
            print("   %-8s rel %.3g max/rms %.3g" % (key, d.norm() / b.norm(), d.abs().max() / b.square().mean().sqrt()),
                  flush=True)
