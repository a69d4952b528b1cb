"""The work a user of this framework has it do, as cases a timer can run.

Five kinds of pass, each through the public entry points:

  prefill    the fused forward over a grid of tiles, prepared once as a layer
             does whose tiles keep their addresses (plan_grid)
  step       one step of generation through the key/value cache: the new rows
             join the cache, the new queries attend to all of it
             (KVCache.append_attend; one token, a few, or a long chunk)
  tasks      the reference's own submission: one kernel call per pair of
             square tiles with an additive mask tile, forward or backward
             (flash_sdpa_fwd, flash_sdpa_bwd), after the running logsumexp
             or the gradients were cleared
  train      the fused backward over a grid of tiles (plan_bwd_grid)
  layer_io   what stands either side of the attention in a layer: transposes
             of the projections and of the output, rotary embedding of Q and K

A case is a dict of plain values.  Tensors are C-ordered views of NNTile's
Fortran tiles: K, V [n_batch * n_head_kv, rows, head], Q, A
[n_batch * kv_group * n_head_kv, rows, head].
"""
import math

import torch

from nntile_amd import hip_sdpa as hs
from nntile_amd.kv_cache import KVCache

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # generation of one sequence, token by token, grouped-query heads:
        # nothing but latency, the call a chat makes most often
        dict(name="step_one_token_bf16", op="step", dtype="bf16", head=128, n_batch=1, n_head_kv=8,
             kv_group=4, q_seq=1, filled=1023, capacity=4096),
        # the decode configuration: 8 sequences, 16 new tokens each, 8192 keys
        dict(name="step_gqa_bf16", op="step", dtype="bf16", head=128, n_batch=8, n_head_kv=8,
             kv_group=4, q_seq=16, filled=8176, capacity=8192),
        # generation with the small fp32 model, an odd number of sequences
        # and of keys
        dict(name="step_gpt2_fp32", op="step", dtype="fp32", head=64, n_batch=5, n_head_kv=12,
             kv_group=1, q_seq=1, filled=777, capacity=1024),
        # a long prompt taken in chunks: 333 tokens behind 1500 in the cache
        dict(name="step_chunk_fp16", op="step", dtype="fp16", head=128, n_batch=2, n_head_kv=8,
             kv_group=4, q_seq=333, filled=1500, capacity=2048),
        # the prefill configuration: 32 heads, 4096 tokens, tiles of 1024
        dict(name="prefill_llama_bf16", op="prefill", dtype="bf16", head=128, n_batch=1,
             n_head_kv=32, kv_group=1, seq=4096, tile=1024, causal=True),
        # the long-sequence configuration: 16384 tokens, 8 heads
        dict(name="prefill_long_bf16", op="prefill", dtype="bf16", head=128, n_batch=1,
             n_head_kv=8, kv_group=1, seq=16384, tile=1024, causal=True),
        # the small fp32 model's layer: 12 heads, 1024 tokens, 4 sequences
        dict(name="prefill_gpt2_fp32", op="prefill", dtype="fp32", head=64, n_batch=4,
             n_head_kv=12, kv_group=1, seq=1024, tile=1024, causal=True),
        # the smallest tile of the reference's kernel benchmark, as one task
        dict(name="task_small_bf16", op="tasks", dtype="bf16", head=64, batch=4, tile=128,
             n_tiles=1, mask="causal", backward=False),
        # the prefill configuration as the reference submits it: 4 x 4 tasks,
        # each with its mask tile
        dict(name="tasks_llama_bf16", op="tasks", dtype="bf16", head=128, batch=32, tile=1024,
             n_tiles=4, mask="causal", backward=False),
        # a training step's backward as the reference submits it, on tiles of
        # an odd size
        dict(name="tasks_backward_fp16", op="tasks", dtype="fp16", head=64, batch=12, tile=500,
             n_tiles=2, mask="causal", backward=True),
        # the backward of the prefill configuration in one call
        dict(name="train_llama_bf16", op="train", dtype="bf16", head=128, n_batch=1, n_head_kv=32,
             kv_group=1, seq=4096, tile=1024, causal=True),
        # what surrounds the attention in a grouped-query layer of 2048 tokens
        dict(name="layer_io_bf16", op="layer_io", dtype="bf16", head=128, n_batch=1, n_head_kv=8,
             kv_group=4, seq=2048, backward=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


#: the most a drawn case may cost, below the largest listed ones: operations
#: (fp32 runs on matrix units of a sixteenth of the rate) and bytes
_MOST_FLOPS = {"bf16": 3.0e11, "fp16": 3.0e11, "fp32": 1.9e10}
_MOST_BYTES = 2.8e8


def _draw(rng):
    op = rng.choice(["step", "step", "step", "prefill", "prefill", "prefill", "tasks", "tasks", "train",
                     "layer_io"])
    # 16-bit tiles are the rule, fp32 what the small models use
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    head = rng.choice([64, 128, 128])
    heads = rng.choice([(4, 1), (8, 1), (12, 1), (16, 1), (32, 1), (8, 4), (4, 4), (2, 8)])
    if op == "step":
        q_seq = rng.choice([1, 1, 1, _log(rng, 2, 16), _log(rng, 17, 1024)])
        filled = _log(rng, 16, 16000)
        return dict(op=op, dtype=dtype, head=head, n_batch=_log(rng, 1, 24), n_head_kv=heads[0],
                    kv_group=heads[1], q_seq=q_seq, filled=filled,
                    capacity=filled + q_seq + rng.choice([0, 1, 100, 1024]))
    if op == "tasks":
        backward = dtype != "fp32" and rng.random() < 0.5
        return dict(op=op, dtype=dtype, head=head, batch=_log(rng, 1, 64), tile=_log(rng, 48, 2048),
                    n_tiles=rng.randint(1, 4), mask=rng.choice(["causal", "causal", "full", "window"]),
                    backward=backward)
    if op == "layer_io":
        return dict(op=op, dtype=dtype, head=head, n_batch=_log(rng, 1, 8), n_head_kv=heads[0],
                    kv_group=heads[1], seq=_log(rng, 16, 8192), backward=rng.random() < 0.5)
    if op == "train" and dtype == "fp32":
        dtype = "bf16"      # the backward's tiles are 16-bit, as the reference's
    seq = _log(rng, 50, 16384 if op == "prefill" else 8192)
    tile = rng.choice([512, 1024, 2048])
    # (whole tiles in front, a ragged one last; one tile when it is shorter)
    if seq <= tile:
        tile = seq
    elif -(-seq // tile) > 8:
        tile = 2048
    return dict(op=op, dtype=dtype, head=head, n_batch=_log(rng, 1, 8), n_head_kv=heads[0],
                kv_group=heads[1], seq=seq, tile=tile, causal=rng.random() < 0.75)


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= _MOST_FLOPS[case["dtype"]] and w["bytes"] <= _MOST_BYTES:
            return case


class _Inputs:
    """N(0, 1) values in the tile type, from one seeded generator."""

    def __init__(self, case, seed):
        self.dtype = DTYPES[case["dtype"]]
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def __call__(self, *shape):
        return torch.randn(*shape, generator=self.gen, device="cuda", dtype=torch.float32).to(self.dtype)


def _split(t, tile):
    """The tiles of t along its rows, each in memory of its own."""
    return [t[:, s:s + tile].contiguous() for s in range(0, t.shape[1], tile)]


def _lse_tiles(batch, seq, tile):
    return [torch.full((batch, min(tile, seq - s)), float("-inf"), device="cuda")
            for s in range(0, seq, tile)]


def _prepare_prefill(case, seed, backward):
    """Forward and backward over a grid: one slab holding the whole batch."""
    rand = _Inputs(case, seed)
    seq, tile, head = case["seq"], case["tile"], case["head"]
    b_kv = case["n_batch"] * case["n_head_kv"]
    b_q = b_kv * case["kv_group"]
    K, V = (_split(rand(b_kv, seq, head), tile) for _ in range(2))
    Q = _split(rand(b_q, seq, head), tile)
    A = [torch.empty_like(t) for t in Q]
    lse = _lse_tiles(b_q, seq, tile)
    mode = hs.MASK_CAUSAL if case["causal"] else hs.MASK_NONE
    common = dict(n_batch=case["n_batch"], kv_group=case["kv_group"], flags=hs.OVERWRITE)
    fwd = hs.plan_grid(K, Q, lse, V, A, seq, seq, tile, tile, mode, **common)
    if not backward:
        return {"plan": fwd, "out": {"A": A, "lse": lse}}
    fwd.launch()
    dA = _split(rand(b_q, seq, head), tile)
    dK, dV, dQ = ([torch.empty_like(t) for t in x] for x in (K, V, Q))
    workspace = torch.empty(4 * seq * b_q, dtype=torch.uint8, device="cuda")
    bwd = hs.plan_bwd_grid(K, Q, V, A, dA, lse, dK, dQ, dV, seq, seq, tile, tile, mode, workspace, **common)
    return {"plan": bwd, "out": {"dK": dK, "dQ": dQ, "dV": dV}}


def _prepare_step(case, seed):
    rand = _Inputs(case, seed)
    head, q_seq, filled = case["head"], case["q_seq"], case["filled"]
    b_kv = case["n_batch"] * case["n_head_kv"]
    b_q = b_kv * case["kv_group"]
    cache = KVCache(case["capacity"])
    cache.append(rand(b_kv, filled, head), rand(b_kv, filled, head))
    Q = rand(b_q, q_seq, head)
    return {"cache": cache, "k": rand(b_kv, q_seq, head), "v": rand(b_kv, q_seq, head), "Q": Q,
            "lse": torch.empty(b_q, q_seq, device="cuda"), "A": torch.empty_like(Q)}


def _run_step(case, s):
    cache = s["cache"]
    # every pass takes the step at the same place: the rows of the pass before
    # are given up, as when drafted tokens are drawn back
    cache.k_cache_size = cache.v_cache_size = case["filled"]
    cache.append_attend(s["k"], s["v"], s["Q"], s["lse"], s["A"], case["n_batch"], case["kv_group"])
    return {"A": s["A"], "lse": s["lse"], "k": cache.k, "v": cache.v}


def _mask_tile(case, qi, ki, dtype):
    """0 where visible, -inf where hidden, [queries, keys] of one tile pair."""
    tile = case["tile"]
    q = (torch.arange(tile, device="cuda") + qi * tile)[:, None]
    k = (torch.arange(tile, device="cuda") + ki * tile)[None, :]
    if case["mask"] == "causal":
        seen = k <= q
    elif case["mask"] == "window":
        seen = (q - k).abs() <= 32
    else:
        seen = torch.ones(tile, tile, dtype=torch.bool, device="cuda")
    zero, hidden = (torch.tensor(x, dtype=dtype, device="cuda") for x in (0.0, float("-inf")))
    return torch.where(seen, zero, hidden).contiguous()


def _prepare_tasks(case, seed):
    rand = _Inputs(case, seed)
    n, tile, head, batch = case["n_tiles"], case["tile"], case["head"], case["batch"]
    K, Q, V = ([rand(batch, tile, head) for _ in range(n)] for _ in range(3))
    # the running results of all tiles lie in one allocation, so that one fill
    # clears them
    lse = torch.empty(n, batch, tile, device="cuda")
    A = torch.zeros(n, batch, tile, head, device="cuda", dtype=rand.dtype)
    s = {"K": K, "Q": Q, "V": V, "lse": lse, "A": A,
         "mask": [[_mask_tile(case, i, j, rand.dtype) for j in range(n)] for i in range(n)],
         "scratch_lse": torch.empty(batch, tile, device="cuda"), "scratch": torch.empty_like(Q[0])}
    if case["backward"]:
        _tasks_forward(case, s)
        s["dA"] = [rand(batch, tile, head) for _ in range(n)]
        s["grads"] = torch.empty(3, n, batch, tile, head, device="cuda", dtype=rand.dtype)
    return s


def _tasks_forward(case, s):
    s["lse"].fill_(float("-inf"))
    for i in range(case["n_tiles"]):
        for j in range(case["n_tiles"]):
            hs.flash_sdpa_fwd(s["K"][j], s["Q"][i], s["mask"][i][j], s["lse"][i], s["V"][j], s["A"][i],
                              s["scratch_lse"], s["scratch"])
    return {"A": s["A"], "lse": s["lse"]}


def _tasks_backward(case, s):
    s["grads"].zero_()
    dK, dQ, dV = s["grads"]
    for i in range(case["n_tiles"]):
        for j in range(case["n_tiles"]):
            hs.flash_sdpa_bwd(s["K"][j], s["Q"][i], s["V"][j], s["A"][i], s["dA"][i], s["mask"][i][j],
                              s["lse"][i], s["scratch"], dK[j], dQ[i], dV[j])
    return {"dK": dK, "dQ": dQ, "dV": dV}


def _prepare_layer_io(case, seed):
    """q, k, v: projections, heads slowest in NNTile's axes (fastest here is
    the head index, so an attention tile is their transpose)."""
    rand = _Inputs(case, seed)
    n_kv, group = case["n_head_kv"], case["kv_group"]
    rows = case["head"] * case["seq"] * case["n_batch"]     # elements of one head
    angle = torch.rand(rows // 2, generator=rand.gen, device="cuda") * (2 * math.pi)
    s = {"sin": angle.sin().to(rand.dtype), "cos": angle.cos().to(rand.dtype)}
    for name, heads in (("q", n_kv * group), ("k", n_kv), ("v", n_kv), ("a", n_kv * group)):
        s[name] = rand(rows, heads)
        s[name + "_t"] = torch.empty_like(s[name])
    for name in ("q", "k"):
        s[name + "_r"] = torch.empty_like(s[name])
    return s


def _run_layer_io(case, s):
    n_kv, group = case["n_head_kv"], case["kv_group"]
    rows = case["head"] * case["seq"] * case["n_batch"]
    for name, heads in (("q", n_kv * group), ("k", n_kv)):
        if case["backward"]:
            # the gradient arrives in the attention layout and leaves in the
            # projections'
            hs.rope(s["sin"], s["cos"], s[name], s[name + "_r"], backward=True)
            hs.transpose(1.0, s[name + "_r"], s[name + "_t"], rows, heads)
        else:
            hs.transpose(1.0, s[name], s[name + "_t"], heads, rows)
            hs.rope(s["sin"], s["cos"], s[name + "_t"], s[name + "_r"])
    if case["backward"]:
        hs.transpose(1.0, s["v"], s["v_t"], rows, n_kv)
        hs.transpose(1.0, s["a"], s["a_t"], n_kv * group, rows)
        return {name: s[name + "_t"] for name in ("q", "k", "v", "a")}
    hs.transpose(1.0, s["v"], s["v_t"], n_kv, rows)
    hs.transpose(1.0, s["a"], s["a_t"], rows, n_kv * group)
    return {"q": s["q_r"], "k": s["k_r"], "v": s["v_t"], "a": s["a_t"]}


def prepare(case, seed):
    op = case["op"]
    if op == "step":
        s = _prepare_step(case, seed)
    elif op == "tasks":
        s = _prepare_tasks(case, seed)
    elif op == "layer_io":
        s = _prepare_layer_io(case, seed)
    else:
        s = _prepare_prefill(case, seed, op == "train")
    s["case"] = case
    return s


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "step":
        return _run_step(case, state)
    if op == "tasks":
        return _tasks_backward(case, state) if case["backward"] else _tasks_forward(case, state)
    if op == "layer_io":
        return _run_layer_io(case, state)
    state["plan"].launch()
    return state["out"]


def _visible(seq, mask):
    """(query, key) pairs of one batch entry that the mask leaves visible."""
    if mask == "causal":
        return seq * (seq + 1) // 2
    if mask == "window":
        w = min(32, seq - 1)
        return seq * (2 * w + 1) - w * (w + 1)
    return seq * seq


def work(case):
    """Inputs read once, outputs written once; products of visible pairs only
    (two per pair in the forward, five in the backward)."""
    e = 4 if case["dtype"] == "fp32" else 2
    op, head = case["op"], case["head"]
    if op == "layer_io":
        elems = head * case["seq"] * case["n_batch"]
        n_kv, n_q = case["n_head_kv"], case["n_head_kv"] * case["kv_group"]
        # four transposes and the rotary embedding of Q and K, each entry
        # point reading and writing its tensor once, and the sines and cosines
        return {"bytes": e * elems * (2 * (2 * n_q + 2 * n_kv) + 2 * (n_q + n_kv) + 2),
                "flops": 3 * elems * (n_q + n_kv)}
    if op == "step":
        b_kv = case["n_batch"] * case["n_head_kv"]
        b_q, q_seq = b_kv * case["kv_group"], case["q_seq"]
        keys = case["filled"] + q_seq
        pairs = q_seq * case["filled"] + q_seq * (q_seq + 1) // 2
        # the keys and values, the new rows' writes into the caches, Q, A, lse
        return {"bytes": e * head * (2 * b_kv * (keys + q_seq) + 2 * b_q * q_seq) + 4 * b_q * q_seq,
                "flops": 4 * head * pairs * b_q}
    if op == "tasks":
        b_q = b_kv = case["batch"]
        seq = case["tile"] * case["n_tiles"]
        mask, backward = case["mask"], case["backward"]
        mask_bytes = e * seq * seq
    else:
        b_kv = case["n_batch"] * case["n_head_kv"]
        b_q = b_kv * case["kv_group"]
        seq, mask_bytes = case["seq"], 0
        mask, backward = "causal" if case["causal"] else "full", op == "train"
    pairs = _visible(seq, mask)
    if backward:    # K, V, Q, A, dA, lse in; dK, dV, dQ out
        moved = e * head * seq * (4 * b_kv + 4 * b_q) + 4 * seq * b_q
    else:
        moved = e * head * seq * (2 * b_kv + 2 * b_q) + 4 * seq * b_q
    return {"bytes": moved + mask_bytes, "flops": (10 if backward else 4) * head * pairs * b_q}


def tolerance(case):
    """What two correct implementations differ by in the tile type, with sums
    and statistics in fp32."""
    if case["op"] == "layer_io":
        return {"rel": {"bf16": 4e-3, "fp16": 5e-4, "fp32": 1e-6}[case["dtype"]]}
    return {"rel": {"bf16": 1e-2, "fp16": 2e-3, "fp32": 1e-5}[case["dtype"]]}
