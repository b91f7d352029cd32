"""What this framework is timed on: the calls a serving program makes, over the sizes it makes
them at.

Every case goes through the public entry points: the op seam (``mini_vllm.kernels.ops``) for
the attention calls and the MLP, the sampler's distribution, the paged model's forward pass
and the engine's decode graphs. Shapes are the Qwen3-0.6B ones that the repository's
configurations and benchmark use (16 query heads over 8 kv heads or, as a generic wider model,
32 over 8; head dim 128; hidden 1024; MLP 3072; vocabulary 151936; 16-token pages in shuffled
order). K, V and queries are N(0, 1), which is what QK-normed heads hold.
"""

import math
import random
import sys
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "mini-vllm_amd"))

from mini_vllm import torch_path  # noqa: E402
from mini_vllm.block.block_manager import BlockManager  # noqa: E402
from mini_vllm.kernels import ops  # noqa: E402
from mini_vllm.model.qwen3_paged import ModelConfig, Qwen3Paged  # noqa: E402
from mini_vllm.sampler import SamplingParams, sampling_probabilities  # noqa: E402
from mini_vllm.serve.batch import ForwardBatch  # noqa: E402
from mini_vllm.serve.graphs import DecodeGraphs  # noqa: E402
from mini_vllm.serve.sequence import Sequence  # noqa: E402
from mini_vllm.workloads import build_batch  # noqa: E402

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16,
          "fp8": torch.float8_e4m3fn}
BYTES = {"f32": 4, "f16": 2, "bf16": 2, "fp8": 1}
D = 128           # head dim
PAGE = 16         # tokens per page
HIDDEN, MLP, VOCAB = 1024, 3072, 151936
EPS = 1e-6
MAX_POSITIONS = 40960
THETA = 1_000_000.0


# ------------------------------------------------------------------------------- cases


def listed():
    return [
        # The smallest call: four short fp32 requests, one decode step's attention (the
        # repository's parity configuration): launches and latency, nothing to stream.
        dict(name="decode_f32_4", kind="paged", dtype="f32", kv="f32", hq=16, hk=8,
             decodes=4, lo=37, hi=1000, chunks=0, chunk_lo=0, chunk_hi=0, prefix_lo=0,
             prefix_hi=0),
        # A full decode batch at mixed contexts, 16-bit cache: the bandwidth headline.
        dict(name="decode_bf16_64", kind="paged", dtype="bf16", kv="bf16", hq=16, hk=8,
             decodes=64, lo=512, hi=4096, chunks=0, chunk_lo=0, chunk_hi=0, prefix_lo=0,
             prefix_hi=0),
        # A large decode batch of long contexts over an fp8 cache.
        dict(name="decode_fp8_128", kind="paged", dtype="bf16", kv="fp8", hq=16, hk=8,
             decodes=128, lo=2048, hi=8192, chunks=0, chunk_lo=0, chunk_hi=0, prefix_lo=0,
             prefix_hi=0),
        # One user's long conversation: a decode step's attention with its new token's
        # QK-norm, RoPE and cache write, for a single sequence.
        dict(name="step_attention_1", kind="step", dtype="bf16", hq=16, hk=8, decodes=1,
             lo=8192, hi=8192),
        # Chunked prefill as the scheduler makes it: 512-token chunks after ragged prefixes.
        dict(name="prefill_bf16_8x512", kind="paged", dtype="bf16", kv="bf16", hq=16, hk=8,
             decodes=0, lo=0, hi=0, chunks=8, chunk_lo=512, chunk_hi=512, prefix_lo=0,
             prefix_hi=1536),
        # A long document's last chunk, float16, four query heads per kv head.
        dict(name="prefill_f16_long", kind="paged", dtype="f16", kv="f16", hq=32, hk=8,
             decodes=0, lo=0, hi=0, chunks=1, chunk_lo=2048, chunk_hi=2048, prefix_lo=14336,
             prefix_hi=14336),
        # An engine iteration's attention over an fp8 cache: ragged prompt chunks beside
        # running decodes.
        dict(name="mixed_fp8", kind="paged", dtype="bf16", kv="fp8", hq=16, hk=8,
             decodes=28, lo=64, hi=2300, chunks=5, chunk_lo=61, chunk_hi=512, prefix_lo=0,
             prefix_hi=1536),
        # The dense-cache model's decode: 32 sequences in a cache allocated for twice as many
        # positions.
        dict(name="dense_decode_32", kind="dense", dtype="bf16", hq=16, hk=8, batch=32,
             length=1, keys=2048, room=4096),
        # A decode step's MLP: gate/up with SwiGLU, down with the residual add and the norm.
        dict(name="mlp_decode_32", kind="mlp", dtype="bf16", rows=32),
        # The sampling distribution of a batch whose requests use temperature, top-k, top-p
        # and greedy decoding side by side.
        dict(name="sample_32", kind="sample", dtype="bf16", rows=32, vocab=VOCAB,
             profile="mixed"),
        # A prefill iteration through the paged model (two layers of it): projections, norms,
        # RoPE, cache write, attention, MLP and the last rows' logits.
        dict(name="forward_prefill", kind="forward", dtype="bf16", layers=2, decodes=24,
             lo=64, hi=2300, chunks=4, chunk_lo=380, chunk_hi=512, prefix_lo=0, prefix_hi=1536),
        # A decode iteration of the paged model as the engine runs it (replayed graph), four
        # layers deep: a rounding that falls differently grows through the layers (3% of the
        # logits over all 28, 1% over six).
        dict(name="engine_step_32", kind="graph", dtype="bf16", layers=4, decodes=32,
             lo=900, hi=1300),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of these ranges: sizes are spread over their logarithm."""
    kind = rng.choice(["decode", "decode", "step", "prefill", "prefill", "mixed", "dense", "mlp",
                       "sample", "forward", "graph"])
    seed = rng.randrange(1 << 20)  # of the case's lengths
    none = dict(chunks=0, chunk_lo=0, chunk_hi=0, prefix_lo=0, prefix_hi=0)
    if kind == "decode":
        dtype, kv = rng.choice([("bf16", "bf16"), ("f16", "f16"), ("bf16", "fp8"), ("f32", "f32")])
        n = _log_int(rng, 1, 64)
        hi = _log_int(rng, 100, 8192 if dtype != "f32" else 1000)
        return dict(kind="paged", dtype=dtype, kv=kv, hq=rng.choice([16, 16, 32]), hk=8, decodes=n,
                    lo=max(1, hi // rng.choice([1, 2, 8])), hi=hi, seed=seed, **none)
    if kind == "step":
        hi = _log_int(rng, 100, 8192)
        return dict(kind="step", dtype=rng.choice(["bf16", "f16"]), hq=rng.choice([16, 16, 32]), hk=8,
                    decodes=_log_int(rng, 1, 64), lo=max(1, hi // rng.choice([1, 2, 8])), hi=hi,
                    seed=seed)
    if kind in ("prefill", "mixed"):
        dtype, kv = rng.choice([("bf16", "bf16"), ("f16", "f16"), ("bf16", "fp8")])
        chunk = _log_int(rng, 61, 2048)
        chunks = min(_log_int(rng, 1, 8), max(1, 4096 // chunk))
        decodes = _log_int(rng, 4, 64) if kind == "mixed" else 0
        return dict(kind="paged", dtype=dtype, kv=kv, hq=rng.choice([16, 16, 32]), hk=8,
                    decodes=decodes, lo=64 if decodes else 0, hi=2300 if decodes else 0,
                    chunks=chunks, chunk_lo=max(2, chunk // rng.choice([1, 1, 4])), chunk_hi=chunk,
                    prefix_lo=0, prefix_hi=_log_int(rng, 64, 8192), seed=seed)
    if kind == "dense":
        length = rng.choice([1, 1, _log_int(rng, 64, 512)])
        keys = _log_int(rng, max(64, length), 4096)
        return dict(kind="dense", dtype=rng.choice(["bf16", "f16"]), hq=16, hk=8,
                    batch=_log_int(rng, 1, 32 if length == 1 else 8), length=length, keys=keys,
                    room=keys * rng.choice([1, 2]), seed=seed)
    if kind == "mlp":
        return dict(kind="mlp", dtype=rng.choice(["bf16", "f16"]), rows=_log_int(rng, 1, 2048),
                    seed=seed)
    if kind == "sample":
        return dict(kind="sample", dtype=rng.choice(["bf16", "f32"]), rows=_log_int(rng, 1, 32),
                    vocab=rng.choice([VOCAB, 32000, 50257]),
                    profile=rng.choice(["mixed", "top_p", "top_k", "temperature"]), seed=seed)
    if kind == "forward":
        chunk = _log_int(rng, 70, 512)
        return dict(kind="forward", dtype="bf16", layers=2, decodes=rng.choice([0, 8, 24]), lo=64,
                    hi=2300, chunks=rng.choice([1, 2, 4]), chunk_lo=max(2, chunk // 2),
                    chunk_hi=chunk, prefix_lo=0, prefix_hi=1536, seed=seed)
    hi = _log_int(rng, 100, 2300)
    return dict(kind="graph", dtype="bf16", layers=4, decodes=_log_int(rng, 1, 32),
                lo=max(1, hi // rng.choice([1, 2, 8])), hi=hi, seed=seed)


def _lengths(case):
    """(contexts, query lengths) of a case's sequences, prompt chunks among the decodes: the
    case's own, whatever the inputs' seed."""
    rng = random.Random(case.get("seed", 0))
    rows = [(rng.randint(case["lo"], case["hi"]), 1) for _ in range(case["decodes"])]
    for _ in range(case.get("chunks", 0)):
        n = rng.randint(case["chunk_lo"], case["chunk_hi"])
        rows.append((n + rng.randint(case["prefix_lo"], case["prefix_hi"]), n))
    if case.get("chunks", 0):
        rng.shuffle(rows)
    return [c for c, _ in rows], [n for _, n in rows]


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _randn(gen, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=gen, device=DEVICE) * std).to(dtype)


# ----------------------------------------------------------------------------- prepare


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def _prepare_paged(case, seed):
    contexts, lens = _lengths(case)
    b = build_batch(contexts, lens, dtype=DTYPES[case["dtype"]], kv_dtype=DTYPES[case["kv"]],
                    num_q_heads=case["hq"], num_kv_heads=case["hk"], head_dim=D, block_size=PAGE,
                    seed=seed, device=DEVICE, generator_device=DEVICE)
    return {"kind": "paged", "b": b, "args": b.args()}


def _prepare_step(case, seed):
    contexts, lens = _lengths(case)
    dtype = DTYPES[case["dtype"]]
    b = build_batch(contexts, lens, dtype=dtype, num_q_heads=case["hq"], num_kv_heads=case["hk"],
                    head_dim=D, block_size=PAGE, seed=seed, device=DEVICE, generator_device=DEVICE)
    gen = _generator(seed + 1)
    n, hq, hk = len(contexts), case["hq"], case["hk"]
    # the q/k/v projection's output, read through column views as the model passes it
    qkv = _randn(gen, n, (hq + 2 * hk) * D, dtype=dtype)
    q, k, v = qkv.split([hq * D, hk * D, hk * D], dim=1)
    cos, sin = torch_path.rope_tables(D, MAX_POSITIONS, THETA, device=DEVICE)
    return {"kind": "step", "b": b, "q": q.view(n, hq, D), "k": k.view(n, hk, D),
            "v": v.view(n, hk, D), "qw": 1 + _randn(gen, D, std=0.1, dtype=dtype),
            "kw": 1 + _randn(gen, D, std=0.1, dtype=dtype), "cos": cos, "sin": sin}


def _prepare_dense(case, seed):
    gen = _generator(seed)
    dtype = DTYPES[case["dtype"]]
    b, L, keys = case["batch"], case["length"], case["keys"]
    cache = [_randn(gen, b, case["hk"], case["room"], D, dtype=dtype) for _ in range(2)]
    return {"kind": "dense", "q": _randn(gen, b, case["hq"], L, D, dtype=dtype),
            "k": cache[0][:, :, :keys], "v": cache[1][:, :, :keys]}


def _prepare_mlp(case, seed):
    gen = _generator(seed)
    dtype = DTYPES[case["dtype"]]
    gate, up = (_randn(gen, MLP, HIDDEN, std=0.02, dtype=dtype) for _ in range(2))
    down = _randn(gen, HIDDEN, MLP, std=0.02, dtype=dtype)
    return {"kind": "mlp", "x": _randn(gen, case["rows"], HIDDEN, dtype=dtype),
            "h": _randn(gen, case["rows"], HIDDEN, dtype=dtype),
            "norm": 1 + _randn(gen, HIDDEN, std=0.1, dtype=dtype), "gate": gate, "up": up,
            "gate_up": ops.pack_weight(torch_path.interleave_gate_up(gate, up), use_cuda=True),
            "down": ops.pack_weight(down, use_cuda=True)}


# Requests of one batch, in turn: (temperature, top_k, top_p).
_PROFILES = {
    "mixed": [(0.7, 0, 0.9), (1.0, 50, 1.0), (0.6, 20, 0.95), (0.0, 0, 1.0), (1.0, 0, 1.0),
              (0.8, 40, 0.95), (1.2, 0, 0.8)],
    "top_p": [(0.7, 0, 0.9), (1.0, 0, 0.95)],
    "top_k": [(1.0, 50, 1.0), (0.6, 20, 0.95)],
    "temperature": [(1.0, 0, 1.0), (0.7, 0, 1.0)],
}


def _prepare_sample(case, seed):
    gen = _generator(seed)
    # token probabilities that fall off as a power of the rank, as a language model's do
    u = torch.rand(case["rows"], case["vocab"], generator=gen, device=DEVICE)
    logits = (-1.6 * torch.log1p(-u)).to(DTYPES[case["dtype"]])
    profile = _PROFILES[case["profile"]]
    return {"kind": "sample", "logits": logits,
            "params": [SamplingParams(*profile[i % len(profile)]) for i in range(case["rows"])]}


def _model(case, seed):
    """A paged model with random weights, its pool filled as by earlier iterations, and the
    scheduled (sequence, tokens) pairs of one more."""
    gen = _generator(seed)
    dtype = DTYPES[case["dtype"]]
    contexts, lens = _lengths(case)
    config = ModelConfig(num_hidden_layers=case["layers"], dtype=dtype)
    q, kv, e, i = config.q_size, config.kv_size, config.hidden_size, config.intermediate_size
    weights = {"embedding": _randn(gen, config.vocab_size, e, std=0.02, dtype=dtype),
               "final_norm": 1 + _randn(gen, e, std=0.1, dtype=dtype)}
    for layer in range(config.num_hidden_layers):
        for name, shape in (("wq", (q, e)), ("wk", (kv, e)), ("wv", (kv, e)), ("wo", (e, q)),
                            ("gate", (i, e)), ("up", (i, e)), ("down", (e, i))):
            weights[f"layers.{layer}.{name}"] = _randn(gen, *shape, std=0.02, dtype=dtype)
        for name, n in (("q_norm", D), ("k_norm", D), ("attn_norm", e), ("mlp_norm", e)):
            weights[f"layers.{layer}.{name}"] = 1 + _randn(gen, n, std=0.1, dtype=dtype)
    pages = [-(-c // PAGE) for c in contexts]
    manager = BlockManager(sum(pages) + 8, PAGE, config.num_hidden_layers,
                           config.num_key_value_heads, config.head_dim, dtype, DEVICE)
    # pages are handed out a few at a time, to the sequences in turn, as serving does
    rng = random.Random(seed)
    grown = [0] * len(pages)
    while any(g < p for g, p in zip(grown, pages)):
        s = rng.choice([j for j, p in enumerate(pages) if grown[j] < p])
        grown[s] = min(pages[s], grown[s] + rng.randint(1, 8))
        manager.allocate(s, grown[s] * PAGE)
    for layer in range(config.num_hidden_layers):
        for pool in (manager.kv.keys, manager.kv.values):
            pool[layer].copy_(_randn(gen, *pool[layer].shape))
    ids = torch.randint(0, config.vocab_size, (sum(contexts),), generator=gen,
                        device=DEVICE).tolist()
    scheduled = []
    for s, (c, n) in enumerate(zip(contexts, lens)):
        tokens, ids = ids[:c], ids[c:]
        scheduled.append((Sequence(s, tokens, 256, num_computed_tokens=c - n), n))
    return Qwen3Paged(config, weights, manager, use_cuda=True), scheduled


def _prepare_forward(case, seed):
    model, scheduled = _model(case, seed)
    return {"kind": "forward", "model": model, "scheduled": scheduled,
            "batch": ForwardBatch.from_scheduled(scheduled, model.manager, DEVICE)}


def _prepare_graph(case, seed):
    model, scheduled = _model(case, seed)
    return {"kind": "graph", "model": model, "scheduled": scheduled,
            "graphs": DecodeGraphs(model, max_batch=32)}


_PREPARE = {"paged": _prepare_paged, "step": _prepare_step, "dense": _prepare_dense,
            "mlp": _prepare_mlp, "sample": _prepare_sample, "forward": _prepare_forward,
            "graph": _prepare_graph}


# --------------------------------------------------------------------------------- run


def run(state):
    return _RUN[state["kind"]](state)


def _run_paged(s):
    b = s["b"]
    return ops.paged_attention(*s["args"], use_cuda=True, k_scale=b.k_scale, v_scale=b.v_scale)


def _run_step(s):
    b = s["b"]
    out = ops.paged_decode_qk_norm_rope(
        s["q"], s["k"], s["v"], s["qw"], s["kw"], s["cos"], s["sin"], EPS, b.key_pool,
        b.value_pool, b.block_tables, b.cu_seqlens_q, b.context_lens, b.seq_lens,
        b.max_context_len, b.scale, use_cuda=True)
    return out, b.key_pool, b.value_pool


def _run_dense(s):
    return ops.attention(s["q"], s["k"], s["v"], mask="causal", use_cuda=True)


def _run_mlp(s):
    gated = ops.linear_swiglu(s["x"], s["gate_up"], use_cuda=True)
    both = ops.linear_residual_rmsnorm(gated, s["down"], s["h"], s["norm"], EPS, use_cuda=True)
    if both is None:  # a prefill's rows: the product, then the add and the norm in one pass
        both = ops.add_rmsnorm(ops.linear(gated, s["down"], use_cuda=True), s["h"], s["norm"],
                               EPS, use_cuda=True)
    return both


def _run_sample(s):
    return sampling_probabilities(s["logits"], s["params"])


def _run_forward(s):
    kv = s["model"].manager.kv
    return s["model"](s["batch"]), kv.keys, kv.values


def _run_graph(s):
    kv = s["model"].manager.kv
    return s["graphs"].run(s["scheduled"]), kv.keys, kv.values


_RUN = {"paged": _run_paged, "step": _run_step, "dense": _run_dense, "mlp": _run_mlp,
        "sample": _run_sample, "forward": _run_forward, "graph": _run_graph}


# -------------------------------------------------------------------------------- work


def _attention_work(contexts, lens, hq, hk, q_bytes, kv_bytes, fp8=False):
    """Visible (query, key) pairs in flops; every visible K/V row, query and output once."""
    pairs = sum(n * (c - n) + n * (n + 1) // 2 for c, n in zip(contexts, lens))
    nbytes = 2 * sum(contexts) * hk * D * kv_bytes + 2 * sum(lens) * hq * D * q_bytes
    if fp8:
        nbytes += 2 * sum(-(-c // PAGE) for c in contexts) * hk * 4
    return nbytes, 4 * hq * D * pairs


def work(case):
    kind = case["kind"]
    size = BYTES[case["dtype"]]
    if kind == "paged":
        nbytes, flops = _attention_work(*_lengths(case), case["hq"], case["hk"], size,
                                        BYTES[case["kv"]], case["kv"] == "fp8")
    elif kind == "step":
        contexts, lens = _lengths(case)
        nbytes, flops = _attention_work(contexts, lens, case["hq"], case["hk"], size, size)
        # the new rows of k and v come from the projection and go to the pools
        nbytes += 2 * len(lens) * case["hk"] * D * size + len(lens) * 2 * D * 4
    elif kind == "dense":
        b, n, c = case["batch"], case["length"], case["keys"]
        nbytes, flops = _attention_work([c] * b, [n] * b, case["hq"], case["hk"], size, size)
    elif kind == "mlp":
        m = case["rows"]
        nbytes = size * (3 * HIDDEN * MLP + 4 * m * HIDDEN)
        flops = 2 * m * 3 * HIDDEN * MLP
    elif kind == "sample":
        n = case["rows"] * case["vocab"]
        nbytes, flops = n * (size + 4), 5 * n
    else:
        contexts, lens = _lengths(case)
        tokens, rows = sum(lens), len(lens)
        c = ModelConfig(num_hidden_layers=case["layers"])
        e, q, kv, i = c.hidden_size, c.q_size, c.kv_size, c.intermediate_size
        layer = e * (q + 2 * kv) + q * e + 3 * e * i
        abytes, aflops = _attention_work(contexts, lens, c.num_attention_heads,
                                         c.num_key_value_heads, size, size)
        per_token = 2 * q + 2 * kv  # q and the attention's output aside: K and V written
        nbytes = case["layers"] * (size * layer + abytes + size * tokens * per_token)
        nbytes += size * (c.vocab_size * e + rows * c.vocab_size + tokens * e)
        # the last layer's down projection and the logits take each sequence's last row only
        flops = case["layers"] * (2 * tokens * layer + aflops) - 2 * (tokens - rows) * e * i
        flops += 2 * rows * c.vocab_size * e
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what another order of the sums, or the error against 64 bits, shows."""
    kind = case["kind"]
    if kind == "sample":
        # 3e-7 (fp32), except where the token at the edge of a nucleus falls the other way:
        # its own probability then, of a row or a few
        return {"rel": 4e-3, "max": 0.9}
    if kind == "forward":  # 4.6e-3 and 6e-2 with another prefill schedule
        return {"rel": 1.8e-2, "max": 0.24}
    if kind == "graph":  # about 8e-3 and 7e-2 with another BLAS and split
        return {"rel": 3e-2, "max": 0.3}
    if case["dtype"] == "f32":  # 1.9e-7 against 64 bits
        return {"rel": 1e-6, "max": 4e-5}
    if case["dtype"] == "f16":  # 2.9e-4 against 64 bits, 3.6e-4 with another schedule
        return {"rel": 1.4e-3, "max": 1.2e-2}
    return {"rel": 8e-3, "max": 0.1}  # 1.7e-3 to 3.5e-3 against 64 bits, 2.1e-3


# ------------------------------------------------------------------------------- exact


def exact(case, seed):
    s = prepare(case, seed)
    return _EXACT[case["kind"]](s)


def _pool64(pool, scales, ids):
    """The pages ``ids`` of a pool as (tokens, kv heads, D) in 64 bits."""
    x = pool[ids].double()
    if scales is not None:
        x = x * scales[ids].double()[:, None, :, None]
    return x.reshape(-1, pool.shape[2], pool.shape[3])


def _attend64(q, k, v, scale):
    """q (L, hq, D) over k and v (S, hk, D), causal with the queries at the end."""
    L, hq, _ = q.shape
    S, hk, _ = k.shape
    out = torch.empty_like(q)
    hidden = (torch.arange(S, device=q.device)[None, :]
              > torch.arange(L, device=q.device)[:, None] + (S - L))
    group = hq // hk
    for j in range(hq):
        scores = (q[:, j] @ k[:, j // group].t()) * scale
        out[:, j] = scores.masked_fill_(hidden, -math.inf).softmax(dim=-1) @ v[:, j // group]
    return out


def _exact_paged(s):
    b = s["b"]
    outs, at = [], 0
    for i, (c, n) in enumerate(zip(b.contexts, b.query_lens)):
        ids = b.block_tables[i, : -(-c // PAGE)].long()
        k = _pool64(b.key_pool, b.k_scale, ids)[:c]
        v = _pool64(b.value_pool, b.v_scale, ids)[:c]
        outs.append(_attend64(b.q[at:at + n].double(), k, v, b.scale))
        at += n
    return torch.cat(outs)


def _rms64(x, w):
    return x * torch.rsqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * w.double()


def _rope64(x, positions):
    """x (T, H, D) rotated at positions (T,)."""
    freq = THETA ** (-torch.arange(0, D, 2, device=x.device, dtype=torch.float64) / D)
    angle = positions.double()[:, None] * freq[None, :]
    angle = torch.cat((angle, angle), dim=-1)[:, None, :]
    turned = torch.cat((-x[..., D // 2:], x[..., :D // 2]), dim=-1)
    return x * angle.cos() + turned * angle.sin()


def _exact_step(s):
    b = s["b"]
    positions = b.context_lens.long() - 1
    q = _rope64(_rms64(s["q"].double(), s["qw"]), positions)
    k_new = _rope64(_rms64(s["k"].double(), s["kw"]), positions)
    v_new = s["v"].double()
    keys, values = b.key_pool.double(), b.value_pool.double()
    outs = []
    for i, c in enumerate(b.contexts):
        ids = b.block_tables[i, : -(-c // PAGE)].long()
        page, row = ids[(c - 1) // PAGE], (c - 1) % PAGE
        keys[page, row], values[page, row] = k_new[i], v_new[i]
        k, v = (_pool64(t, None, ids)[:c] for t in (keys, values))
        outs.append(_attend64(q[i:i + 1], k, v, b.scale))
    return torch.cat(outs), keys, values


def _exact_dense(s):
    out = [_attend64(q.double().transpose(0, 1), k.double().transpose(0, 1),
                     v.double().transpose(0, 1), 1.0 / math.sqrt(D)).transpose(0, 1)
           for q, k, v in zip(s["q"], s["k"], s["v"])]
    return torch.stack(out)


def _exact_mlp(s):
    x = s["x"].double()
    gate, up = x @ s["gate"].double().t(), x @ s["up"].double().t()
    gated = gate * torch.sigmoid(gate) * up
    h = s["h"].double() + gated @ s["down"].dense.double().t()
    return h, _rms64(h, s["norm"])


def _exact_sample(s):
    out = torch.zeros(s["logits"].shape, dtype=torch.float64, device=DEVICE)
    for row, logits, p in zip(out, s["logits"].double(), s["params"]):
        if p.temperature == 0:
            row[logits.argmax()] = 1.0
            continue
        probs, order = (logits / p.temperature).softmax(dim=-1).sort(descending=True, stable=True)
        before = probs.cumsum(dim=-1) - probs
        keep = torch.ones_like(probs, dtype=torch.bool)
        if p.top_k:
            keep[p.top_k:] = False
        if p.top_p < 1.0:
            keep &= before < p.top_p
        keep[0] = True
        row[order] = torch.where(keep, probs, torch.zeros_like(probs)) / probs[keep].sum()
    return out


def _exact_model(s):
    """The forward pass of a scheduled batch; the pools' new rows for a few layers."""
    model, scheduled = s["model"], s["scheduled"]
    c, w, manager = model.config, model.weights, model.manager
    ids, positions, spans, rows = [], [], [], 0
    for seq, n in scheduled:
        start = seq.num_computed_tokens
        ids += seq.tokens(start, n)
        positions += range(start, start + n)
        spans.append((rows, n, start, torch.tensor(manager.table(seq.seq_id), device=DEVICE)))
        rows += n
    positions = torch.tensor(positions, device=DEVICE)
    h = w["embedding"][torch.tensor(ids, device=DEVICE)].double()
    whole = c.num_hidden_layers <= 2
    pools = (manager.kv.keys.double(), manager.kv.values.double()) if whole else None
    for layer in range(c.num_hidden_layers):
        g = {n: w[f"layers.{layer}.{n}"].double() for n in
             ("wq", "wk", "wv", "wo", "gate", "up", "down", "q_norm", "k_norm", "attn_norm",
              "mlp_norm")}
        x = _rms64(h, g["attn_norm"])
        q = _rope64(_rms64((x @ g["wq"].t()).view(rows, -1, D), g["q_norm"]), positions)
        k = _rope64(_rms64((x @ g["wk"].t()).view(rows, -1, D), g["k_norm"]), positions)
        v = (x @ g["wv"].t()).view(rows, -1, D)
        out = torch.empty_like(q)
        for at, n, start, table in spans:
            known = table[: -(-(start + n) // PAGE)]
            new = slice(at, at + n)
            kv = []
            for j, (pool, fresh) in enumerate(((manager.kv.keys, k), (manager.kv.values, v))):
                kv.append(torch.cat((_pool64(pool[layer], None, known)[:start], fresh[new])))
                if whole:
                    where = torch.arange(start, start + n, device=DEVICE)
                    pools[j][layer][table[where // PAGE], where % PAGE] = fresh[new]
            out[new] = _attend64(q[new], *kv, 1.0 / math.sqrt(D))
        h = h + out.reshape(rows, -1) @ g["wo"].t()
        x = _rms64(h, g["mlp_norm"])
        gate = x @ g["gate"].t()
        h = h + (gate * torch.sigmoid(gate) * (x @ g["up"].t())) @ g["down"].t()
    last = torch.tensor([at + n - 1 for at, n, _, _ in spans], device=DEVICE)
    logits = _rms64(h[last], w["final_norm"]) @ w["embedding"].double().t()
    return (logits, *pools) if whole else (logits, None, None)


_EXACT = {"paged": _exact_paged, "step": _exact_step, "dense": _exact_dense, "mlp": _exact_mlp,
          "sample": _exact_sample, "forward": _exact_model, "graph": _exact_model}
