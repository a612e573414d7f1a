"""Workloads of the decode hot path, as a rollout program issues them.

Each case is one call (or one short run of calls) through the C ABI that
rlrt.py binds, on inputs that are already in HBM:

  attn    rl_hip_decode_step: paged GQA decode attention of one batch with the
          append of the step's K/V token, or rl_hip_attn_decode without it
  step    rl_hip_decode_sample_step: one micro-batch's decode step beside the
          sampling of another micro-batch's logits
  lanes   rl_hip_decode_lane_step / _flush: four micro-batches pipelined on
          the two lanes
  sample  rl_hip_sample: greedy, temperature, top-k and top-p
  proj    rl_hip_logits_proj: the vocabulary projection
  ring    infer_submit_decode into the command ring, the batched steps of
          rl_hip_ring_step_enqueue, and the completions read back

listed() names the cases, draw() gives more of the same ranges, prepare()
makes a case's inputs from a seed, run() is one pass, work() what a pass
cannot do without, tolerance() how far a correct result may be off, and
exact() the results in 64 bits from plain torch and numpy.
"""
import ctypes as C
import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gb300-rl-runtime_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import rlrt  # noqa: E402

DTYPES = {"bf16": (torch.bfloat16, rlrt.DTYPE_BF16), "fp16": (torch.float16, rlrt.DTYPE_FP16)}


def listed():
    return [
        # a single rollout with a short prompt: latency of one step's launches
        dict(name="attn_b1_ctx517", kind="attn", batch=1, q_heads=32, kv_heads=8, head_dim=128, dtype="bf16",
             block=16, ctx_lo=517, ctx_hi=517, group=1, prefix=0, append=True),
        # the small-head configuration of the ring worker (MHA 8 x d64, fp16), batched, in 32-token blocks
        dict(name="attn_b24_d64_fp16", kind="attn", batch=24, q_heads=8, kv_heads=8, head_dim=64, dtype="fp16",
             block=32, ctx_lo=64, ctx_hi=2048, group=1, prefix=0, append=True),
        # a GRPO step: 256 slots in groups of 8 that share a 512-token prompt prefix
        dict(name="attn_b256_grpo", kind="attn", batch=256, q_heads=32, kv_heads=8, head_dim=128, dtype="bf16",
             block=16, ctx_lo=513, ctx_hi=1280, group=8, prefix=512, append=True),
        # long-context decode, GQA 8
        dict(name="attn_b8_ctx32k", kind="attn", batch=8, q_heads=64, kv_heads=8, head_dim=128, dtype="bf16",
             block=16, ctx_lo=32768, ctx_hi=32768, group=1, prefix=0, append=False),
        # one micro-batch of 64 rollouts, decode and sampling in one call
        dict(name="step_b64", kind="step", batch=64, q_heads=32, kv_heads=8, head_dim=128, dtype="bf16", block=16,
             ctx_lo=512, ctx_hi=4096, vocab=128256, greedy=False, temperature=0.8, top_k=50, top_p=0.9),
        # 256 rollouts in flight as four micro-batches on two lanes, eight steps
        dict(name="lanes_b64x4", kind="lanes", batch=64, q_heads=32, kv_heads=8, head_dim=128, dtype="bf16",
             block=16, ctx_lo=512, ctx_hi=4096, vocab=128256, greedy=False, temperature=0.8, top_k=50, top_p=0.9,
             steps=8),
        # a full batch sampled with top-k and top-p over a large vocabulary
        dict(name="sample_b256_topk", kind="sample", rows=256, vocab=128256, std=1.0, spikes=5, greedy=False,
             temperature=0.8, top_k=50, top_p=0.9),
        # the GRPO loop's sampler: top-p over the whole of a small vocabulary
        dict(name="sample_b256_topp_32k", kind="sample", rows=256, vocab=32000, std=0.3, spikes=0, greedy=False,
             temperature=1.0, top_k=0, top_p=0.9),
        # top-p over the whole of a large vocabulary, an uneven number of rows
        dict(name="sample_b37_topp_128k", kind="sample", rows=37, vocab=128256, std=1.0, spikes=5, greedy=False,
             temperature=1.0, top_k=0, top_p=0.95),
        # the projection of a small decode batch
        dict(name="proj_r24", kind="proj", rows=24, vocab=32000, hidden=4096),
        # the projection of two full GRPO batches
        dict(name="proj_r512", kind="proj", rows=512, vocab=32000, hidden=4096),
        # 64 rollouts decoded through the rings, eight tokens each
        dict(name="ring_b64", kind="ring", batch=64, q_heads=32, kv_heads=8, head_dim=128, dtype="bf16", block=16,
             ctx_lo=512, ctx_hi=4096, vocab=32000, greedy=False, temperature=0.8, top_k=50, top_p=0.9, steps=8),
    ]


HEADS = ((32, 8, 128), (64, 8, 128), (16, 8, 128), (8, 8, 128), (8, 8, 64), (32, 8, 64), (16, 8, 64))
SAMPLERS = (dict(greedy=True, temperature=1.0, top_k=0, top_p=1.0), dict(greedy=False, top_k=50, top_p=0.9),
            dict(greedy=False, top_k=20, top_p=1.0), dict(greedy=False, top_k=0, top_p=0.9),
            dict(greedy=False, top_k=0, top_p=1.0))


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_attention(rng, most_batch, heads):
    h = rng.choice(heads)
    batch = _log_int(rng, 1, most_batch)
    # at most 300,000 tokens of context in a batch
    hi = _log_int(rng, 100, max(100, min(32768, 300000 // batch)))
    return dict(batch=batch, q_heads=h[0], kv_heads=h[1], head_dim=h[2], dtype=rng.choice(("bf16", "bf16", "fp16")),
                block=rng.choice((16, 16, 32)), ctx_lo=rng.randint(1, hi), ctx_hi=hi)


def _draw_sampler(rng):
    s = dict(rng.choice(SAMPLERS))
    if "temperature" not in s:
        s["temperature"] = round(rng.uniform(0.6, 1.2), 2)
    if s["top_k"]:
        s["top_k"] = _log_int(rng, 5, 200)
    if s["top_p"] < 1.0:
        s["top_p"] = round(rng.uniform(0.7, 0.98), 3)
    return s


def draw(rng):
    kind = rng.choice(("attn", "attn", "attn", "step", "step", "sample", "sample", "sample", "proj", "proj", "ring"))
    if kind == "attn":
        c = dict(kind=kind, **_draw_attention(rng, 256, HEADS), group=1, prefix=0, append=rng.random() < 0.75)
        if rng.random() < 0.25 and c["ctx_lo"] > 64:
            c["group"], c["prefix"] = rng.choice((2, 4, 8)), c["ctx_lo"] // 2 // c["block"] * c["block"]
        return c
    if kind == "step":
        return dict(kind=kind, **_draw_attention(rng, 256, HEADS), vocab=4 * _log_int(rng, 1000, 32768),
                    **_draw_sampler(rng))
    if kind == "sample":
        return dict(kind=kind, rows=_log_int(rng, 1, 512), vocab=_log_int(rng, 4000, 131072),
                    std=rng.choice((0.3, 1.0, 2.0)), spikes=rng.choice((0, 5)), **_draw_sampler(rng))
    if kind == "proj":
        return dict(kind=kind, rows=_log_int(rng, 1, 512), vocab=_log_int(rng, 8000, 40000),
                    hidden=64 * rng.randint(16, 64))
    c = dict(kind=kind, **_draw_attention(rng, 128, HEADS), vocab=4 * _log_int(rng, 1000, 12000), **_draw_sampler(rng),
             steps=rng.randint(2, 8))
    c["ctx_lo"], c["ctx_hi"] = max(32, c["ctx_lo"]), max(64, c["ctx_hi"])
    return c


# ---------------------------------------------------------------- inputs
def _open():
    if not rlrt.lib().rl_hip_is_open():
        rlrt.open_device(torch.cuda.current_device())


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype, std=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype).mul_(std)


def _buf(t):
    return SimpleNamespace(ptr=t.data_ptr(), nbytes=t.numel() * t.element_size())


def _device_bytes(n):
    return torch.zeros(n, dtype=torch.uint8, device="cuda")


def _contexts(case, seed, reach=1):
    """The batch's ragged context lengths. With several steps between two
    reward points (multiples of 32 tokens) no rollout crosses one."""
    ctx = np.random.default_rng(seed).integers(case["ctx_lo"], case["ctx_hi"] + 1, case["batch"])
    if reach > 1:
        ctx = ctx // 32 * 32 + np.minimum(ctx % 32, 32 - 1 - reach)
    return np.maximum(ctx, 1).astype(np.int64)


def _attention(case, seed, reach=1):
    """KV arena, block table, contexts and queries of one batch. The arena holds
    the longest contexts for every rollout; blocks sit at random places of it,
    and the rollouts of a group share the blocks of their prefix."""
    g, tdt = _gen(seed), DTYPES[case["dtype"]][0]
    b, kvh, d, t = case["batch"], case["kv_heads"], case["head_dim"], case["block"]
    ctx = _contexts(case, seed, reach)
    need = -(-(ctx + reach) // t)
    stride = -(-(case["ctx_hi"] + reach) // t)
    shared, group = case.get("prefix", 0) // t, case.get("group", 1)
    own = np.arange(stride)[None, :] < need[:, None]                       # [batch][stride]: the row has such a block
    rows = np.arange(b)
    owner = np.where(np.arange(stride)[None, :] < shared, (rows // group * group)[:, None], rows[:, None])
    mine = own & (owner == rows[:, None])
    ids = np.zeros((b, stride), np.int64)
    ids[mine] = np.arange(int(mine.sum()))
    ids = np.where(own, ids[owner, np.arange(stride)[None, :]], 0)
    n = b * stride * kvh
    perm = torch.randperm(n, generator=g, device="cuda")
    at = torch.from_numpy(ids).cuda()[:, None, :] * kvh + torch.arange(kvh, device="cuda")[None, :, None]
    table = torch.where(torch.from_numpy(own).cuda()[:, None, :], perm[at], 0).to(torch.int32).contiguous()
    return SimpleNamespace(arena=_normal(g, (n, 2, t, d), tdt), table=table, stride=stride, ctx_host=ctx,
                           ctx=torch.from_numpy(ctx).cuda().to(torch.int32),
                           q=_normal(g, (b, case["q_heads"], d), tdt), k_new=_normal(g, (b, kvh, d), tdt),
                           v_new=_normal(g, (b, kvh, d), tdt))


def _logits(g, rows, vocab, std, spikes):
    """fp32 logits ~N(0, std^2), each row with `spikes` tokens well above the
    rest, rows at a stride of whole 16-byte quads."""
    x = _normal(g, (rows, -(-vocab // 4) * 4), torch.float32, std)
    if spikes:
        x.scatter_(1, torch.randint(0, vocab, (rows, spikes), generator=g, device="cuda"), 8.0)
    return x


def _seeds(seed, n):
    return np.random.default_rng(seed + 1).integers(0, 2**63, n, dtype=np.uint64)


def _attn_args(case, s):
    layout = rlrt.KvLayoutDesc.paged(case["block"], case["head_dim"])
    s.out = torch.zeros_like(s.q)
    return rlrt.attn_args(_buf(s.arena), layout, _buf(s.table), s.stride, case["batch"], case["q_heads"],
                          case["kv_heads"], DTYPES[case["dtype"]][1], _buf(s.ctx), case["ctx_hi"], _buf(s.q),
                          _buf(s.out))


def _append_args(case, s):
    return rlrt.AppendArgs(arena_base=s.arena.data_ptr(), arena_bytes=_buf(s.arena).nbytes,
                           layout=rlrt.KvLayoutDesc.paged(case["block"], case["head_dim"]),
                           block_table=s.table.data_ptr(), table_stride=s.stride, batch=case["batch"],
                           kv_heads=case["kv_heads"], positions=s.ctx.data_ptr(), cow_src=None,
                           k_new=s.k_new.data_ptr(), v_new=s.v_new.data_ptr())


def _sample_args(case, s, logits, rows, seed):
    s.logits, s.seeds = logits, torch.from_numpy(_seeds(seed, rows).view(np.int64)).cuda()
    s.tokens = torch.zeros(rows, dtype=torch.int32, device="cuda")
    s.logprobs = torch.zeros(rows, dtype=torch.float32, device="cuda")
    return rlrt.sample_args(_buf(logits), rows, case["vocab"], logits.shape[1], _buf(s.tokens), _buf(s.logprobs),
                            greedy=case["greedy"], temperature=case["temperature"], top_k=case["top_k"],
                            top_p=case["top_p"], step=3, seeds=_buf(s.seeds))


def _micro_batch(case, seed):
    s = _attention(case, seed)
    s.attn, s.append = _attn_args(case, s), _append_args(case, s)
    s.samp = _sample_args(case, s, _logits(_gen(seed + 7), case["batch"], case["vocab"], 1.0, 5), case["batch"], seed)
    s.ws = _device_bytes(rlrt.decode_sample_step_workspace_bytes(s.attn, s.samp))
    return s


class _Ring:
    """The rings, slotted inputs and outputs, and arguments of a ring-driven run."""

    def __init__(self, case, seed):
        lib = rlrt.lib()
        n, b, tdt = case["steps"], case["batch"], DTYPES[case["dtype"]][0]
        qh, kvh, d, v = case["q_heads"], case["kv_heads"], case["head_dim"], case["vocab"]
        s = self.s = _attention(case, seed, reach=n)
        g = _gen(seed + 9)
        self.q, self.k = _normal(g, (n, b, qh, d), tdt), _normal(g, (n, b, kvh, d), tdt)
        self.v, self.logits = _normal(g, (n, b, kvh, d), tdt), _logits(g, n * b, v, 1.0, 5)
        self.seeds = torch.from_numpy(_seeds(seed, b).view(np.int64)).cuda()
        self.out, self.lp = torch.zeros_like(self.q), torch.zeros(n, b, device="cuda")
        self.tok = torch.zeros(n, b, dtype=torch.int32, device="cuda")
        self.rows, self.stats = torch.zeros_like(self.tok), torch.zeros(4, dtype=torch.int64, device="cuda")
        self.cq, self.dq = lib.hw_ring_create(), lib.hw_ring_create()
        self.stop, self.doorbell = lib.rl_hip_host_alloc_coherent(64), lib.rl_hip_host_alloc_coherent(64)
        self.hw = rlrt.InferHwCtx(cmdq=self.cq, doneq=self.dq, doorbell=self.doorbell, gpu_group_id=0, kv_arena_id=0)
        self.args = rlrt.RingStepArgs(
            cmdq=self.cq, doneq=self.dq, stop=self.stop, max_idle_polls=1 << 18, batch=b,
            arena_base=s.arena.data_ptr(), arena_bytes=_buf(s.arena).nbytes,
            layout=rlrt.KvLayoutDesc.paged(case["block"], d), block_table=s.table.data_ptr(), table_stride=s.stride,
            rollouts=b, q_heads=qh, kv_heads=kvh, dtype=DTYPES[case["dtype"]][1], scale=0.0,
            max_ctx=case["ctx_hi"] + n, input_slots=n, q=self.q.data_ptr(), k_new=self.k.data_ptr(),
            v_new=self.v.data_ptr(), logits=self.logits.data_ptr(), vocab=v, greedy=int(case["greedy"]),
            temperature=case["temperature"], top_k=case["top_k"], top_p=case["top_p"], seeds=self.seeds.data_ptr(),
            output_slots=n, attn_out=self.out.data_ptr(), attn_out_f32=None, token_out=self.tok.data_ptr(),
            logprob_out=self.lp.data_ptr(), row_rollout_out=self.rows.data_ptr(), stats=self.stats.data_ptr())
        self.ws = _device_bytes(lib.rl_hip_ring_step_workspace(C.byref(self.args)))
        self.args.workspace, self.args.workspace_bytes = self.ws.data_ptr(), self.ws.numel()
        self.ctx, self.steps, self.done_steps = s.ctx_host.tolist(), n, 0

    def run(self):
        lib = rlrt.lib()
        for i, c in enumerate(self.ctx):
            rlrt.check(lib.infer_submit_decode(C.byref(self.hw), i, 0, 0, 0, c, c + self.steps), "infer_submit_decode")
        rlrt.check(lib.rl_hip_ring_step_enqueue(C.byref(self.args), self.steps, self.done_steps),
                   "rl_hip_ring_step_enqueue")
        self.done_steps += self.steps
        rlrt.sync()
        head, tail = rlrt.hw_ring_indices(self.dq)
        at = (head + np.arange((tail - head) & 0xFFFFFFFF)) & (rlrt.HW_RING_SIZE - 1)
        words = np.frombuffer((C.c_char * (64 * rlrt.HW_RING_SIZE)).from_address(self.dq + 128), np.uint32)
        done = words.reshape(-1, 16)[at].astype(np.int64)
        lib.hw_ring_store_release(self.dq, tail)
        return self.out, self.tok, self.lp, self.rows, self.s.arena, done

    def __del__(self):
        try:
            lib = rlrt.lib()
            lib.hw_ring_destroy(self.cq)
            lib.hw_ring_destroy(self.dq)
            lib.rl_hip_host_free(self.stop)
            lib.rl_hip_host_free(self.doorbell)
        except Exception:
            pass


def prepare(case, seed):
    _open()
    s = SimpleNamespace(case=case)
    if case["kind"] == "attn":
        s.m = _attention(case, seed)
        s.m.attn, s.m.append = _attn_args(case, s.m), _append_args(case, s.m)
        s.ws = _device_bytes(rlrt.lib().rl_hip_attn_decode_workspace(C.byref(s.m.attn)))
        s.m.attn.workspace, s.m.attn.workspace_bytes = s.ws.data_ptr(), s.ws.numel()
    elif case["kind"] == "step":
        s.m = _micro_batch(case, seed)
    elif case["kind"] == "lanes":
        s.m = [_micro_batch(case, seed + 1000 * k) for k in range(4)]
    elif case["kind"] == "sample":
        x = _logits(_gen(seed), case["rows"], case["vocab"], case["std"], case["spikes"])
        s.samp = _sample_args(case, s, x, case["rows"], seed)
        s.ws = _device_bytes(rlrt.lib().rl_hip_sample_workspace(C.byref(s.samp)))
        s.samp.workspace, s.samp.workspace_bytes = s.ws.data_ptr(), s.ws.numel()
    elif case["kind"] == "proj":
        g = _gen(seed)
        s.x = _normal(g, (case["rows"], case["hidden"]), torch.bfloat16)
        s.w = _normal(g, (case["vocab"], case["hidden"]), torch.bfloat16, 0.02)
        s.logits = torch.zeros(case["rows"], -(-case["vocab"] // 4) * 4, device="cuda")
        s.args = rlrt.ProjArgs(x=s.x.data_ptr(), w=s.w.data_ptr(), logits=s.logits.data_ptr(), rows=case["rows"],
                               vocab=case["vocab"], hidden=case["hidden"], x_stride=case["hidden"],
                               w_stride=case["hidden"], logits_stride=s.logits.shape[1])
    else:
        s.ring = _Ring(case, seed)
    return s


# ---------------------------------------------------------------- one pass
def run(state):
    kind = state.case["kind"]
    if kind == "attn":
        m = state.m
        if state.case["append"]:
            rlrt.decode_step(m.attn, m.append)
            return m.out, m.arena
        rlrt.attn_decode(m.attn)
        return m.out
    if kind == "step":
        m = state.m
        rlrt.decode_sample_step(m.attn, m.append, m.samp, _buf(m.ws))
        return m.out, m.tokens, m.logprobs, m.arena
    if kind == "lanes":
        ms, n = state.m, state.case["steps"]
        ws = [_buf(m.ws) for m in ms]
        rlrt.lanes_fork()
        for t in range(n):
            m, prev = ms[t % 4], ()
            m.samp.step = t
            if t >= 2:
                p = (t - 2) % 4
                prev = (ms[p].attn, ms[p].append, ws[p])
            rlrt.decode_lane_step(t % 2, m.attn, m.samp, ws[t % 4], *prev)
        for t in (n - 2, n - 1):
            rlrt.decode_lane_flush(t % 2, ms[t % 4].attn, ms[t % 4].append, ws[t % 4])
        rlrt.lanes_join()
        return [(m.out, m.tokens, m.logprobs, m.arena) for m in ms]
    if kind == "sample":
        rlrt.sample(state.samp)
        return state.tokens, state.logprobs
    if kind == "proj":
        rlrt.check(rlrt.lib().rl_hip_logits_proj(C.byref(state.args)), "rl_hip_logits_proj")
        return state.logits
    return state.ring.run()


# ---------------------------------------------------------------- what a pass cannot do without
def _attention_work(case, tokens, unique, rows):
    """K and V of `unique` tokens read once, queries, outputs and table; `tokens` attended, `rows` queries."""
    d, qh, kvh = case["head_dim"], case["q_heads"], case["kv_heads"]
    kv = unique * kvh * d * 2 * 2
    return (kv + rows * qh * d * 2 * 2 + -(-tokens // case["block"]) * kvh * 4 + rows * kvh * d * 2 * 2 * 2,
            4 * tokens * qh * d)


def work(case):
    kind = case["kind"]
    if kind == "proj":
        r, v, h = case["rows"], case["vocab"], case["hidden"]
        return {"bytes": (r + v) * h * 2 + r * v * 4, "flops": 2 * r * v * h}
    if kind == "sample":
        return {"bytes": case["rows"] * case["vocab"] * 4 + case["rows"] * 16, "flops": 0}
    steps = case.get("steps", 1)
    mean = (case["ctx_lo"] + case["ctx_hi"]) // 2
    b = case["batch"]
    tokens = b * mean
    unique = tokens - (b - -(-b // case.get("group", 1))) * case.get("prefix", 0)
    nbytes, flops = _attention_work(case, tokens, unique, b)
    nbytes += b * case.get("vocab", 0) * 4
    return {"bytes": steps * nbytes, "flops": steps * flops}


def tolerance(case):
    # The stored attention rounds an fp32 result to 16 bits: another summation
    # order moves a result across a rounding boundary now and then. Tokens are
    # whole numbers of a draw that is defined bit for bit; logprobs are fp32.
    # Measured against exact(): logprobs up to 1.6e-7, the projection 3.9e-7,
    # attention 1.7e-3 in bf16 and 2.1e-4 in fp16.
    if case["kind"] == "sample":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    if case["kind"] == "proj":
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 6e-3 if case["dtype"] == "bf16" else 8e-4, "max": 3e-2, "differ": 0.0}


# ---------------------------------------------------------------- the same in 64 bits
def _attend(case, arena, table, ctx, q):
    """softmax(q K^T / sqrt(d)) V in float64, rollout by rollout."""
    kvh, d, t = case["kv_heads"], case["head_dim"], case["block"]
    out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    for b, n in enumerate(ctx):
        ids = table[b, :, :-(-int(n) // t)].long()
        k = arena[ids, 0].reshape(kvh, -1, d)[:, :n].double()
        v = arena[ids, 1].reshape(kvh, -1, d)[:, :n].double()
        x = torch.matmul(q[b].double().reshape(kvh, -1, d), k.transpose(1, 2).contiguous()) / math.sqrt(d)
        out[b] = torch.matmul(torch.softmax(x, -1), v).reshape(-1, d)
    return out


def _appended(case, arena, table, pos, k_new, v_new):
    t = case["block"]
    at = torch.from_numpy(np.asarray(pos)).cuda()
    ids = table[torch.arange(len(pos), device="cuda"), :, at // t].long()     # [batch][kv heads]
    slot = (at % t)[:, None].expand_as(ids)
    arena[ids, 0, slot], arena[ids, 1, slot] = k_new, v_new
    return arena


def _draw64(seed, step, row):
    """Philox4x32-10 (Salmon et al., SC'11): key = seed, counter = (step, row)."""
    m = 0xFFFFFFFF
    c, k = [step & m, step >> 32, row, 0], [seed & m, seed >> 32]
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [(p1 >> 32) ^ c[1] ^ k[0], p1 & m, (p0 >> 32) ^ c[3] ^ k[1], p0 & m]
        k = [(k[0] + 0x9E3779B9) & m, (k[1] + 0xBB67AE85) & m]
    return c[0] | c[1] << 32


def _fma(a, b, c):
    return (a.double() * b + c.double()).float()


def _weights(d):
    """The integer weight of a logit d below the row's maximum: e^d 2^24 by the
    sampling specification's own fp32 range reduction and polynomial."""
    x = d.clamp(min=-87.0)
    n = torch.floor(x * np.float32(1.44269504088896341).item() + 0.5)
    r = _fma(-n, 0.693359375, x)
    r = _fma(-n, float(np.float32(-2.12194440e-4)), r)
    p = torch.full_like(r, np.float32(1.0 / 5040.0).item())
    for c in (1 / 720, 1 / 120, 1 / 24, 1 / 6, 0.5, 1.0, 1.0):
        p = _fma(p, r.double(), torch.full_like(r, np.float32(c).item()))
    w = (p.double() * torch.exp2(n.double() + 24)).long()
    return torch.where(d >= -87.0, w, 0)


def _sample_row(case, l, seed, step, row):
    """(token, logprob) of one row by the sampling specification of sample.h."""
    if case["greedy"]:
        x, token = l, int(torch.nonzero(l == l.max())[0])
    else:
        x = l * float(np.float32(1.0) / np.float32(case["temperature"]))
        keep = torch.ones_like(x, dtype=torch.bool)
        if 0 < case["top_k"] < x.numel():
            keep = x >= torch.topk(x, min(case["top_k"], 256)).values[-1]
        w = torch.where(keep, _weights(x - x.max()), 0)
        if 0 < case["top_p"] < 1:
            order = torch.sort(x, descending=True, stable=True).indices
            cum = torch.cumsum(w[order], 0)
            need = math.ceil(float(np.float32(case["top_p"])) * float(int(cum[-1])))
            n = int(torch.searchsorted(cum, torch.tensor([need], device="cuda"))[0]) + 1
            w = torch.zeros_like(w).scatter_(0, order[:n], w[order[:n]])
        cum = torch.cumsum(w, 0)
        u = (_draw64(seed, step, row) * int(cum[-1])) >> 64
        token = int(torch.searchsorted(cum, torch.tensor([u], device="cuda"), right=True)[0])
    return token, float(x[token].double() - torch.logsumexp(x.double(), 0))


def _sample_all(case, logits, seeds, steps, rows):
    got = [_sample_row(case, logits[i, : case["vocab"]], int(seeds[i]), steps[i], rows[i]) for i in range(len(seeds))]
    return (torch.tensor([t for t, _ in got], dtype=torch.int32), torch.tensor([p for _, p in got], dtype=torch.float64))


def _micro_batch_exact(case, seed, step):
    s = _attention(case, seed)
    out = _attend(case, s.arena, s.table, s.ctx_host, s.q)
    b = case["batch"]
    x = _logits(_gen(seed + 7), b, case["vocab"], 1.0, 5)
    tok, lp = _sample_all(case, x, _seeds(seed, b), [step] * b, range(b))
    return out, tok, lp, _appended(case, s.arena, s.table, s.ctx_host, s.k_new, s.v_new).double()


def exact(case, seed):
    kind = case["kind"]
    if kind == "attn":
        s = _attention(case, seed)
        out = _attend(case, s.arena, s.table, s.ctx_host, s.q)
        if not case["append"]:
            return out
        return out, _appended(case, s.arena, s.table, s.ctx_host, s.k_new, s.v_new).double()
    if kind == "step":
        return _micro_batch_exact(case, seed, 3)
    if kind == "lanes":
        return [_micro_batch_exact(case, seed + 1000 * k, case["steps"] - 4 + k) for k in range(4)]
    if kind == "sample":
        x = _logits(_gen(seed), case["rows"], case["vocab"], case["std"], case["spikes"])
        return _sample_all(case, x, _seeds(seed, case["rows"]), [3] * case["rows"], range(case["rows"]))
    if kind == "proj":
        g, v = _gen(seed), case["vocab"]
        x = _normal(g, (case["rows"], case["hidden"]), torch.bfloat16).double()
        w = _normal(g, (v, case["hidden"]), torch.bfloat16, 0.02)
        logits = torch.zeros(case["rows"], -(-v // 4) * 4, dtype=torch.float64, device="cuda")
        for at in range(0, v, 4096):
            logits[:, at:min(at + 4096, v)] = torch.matmul(x, w[at:at + 4096].double().t().contiguous())
        return logits
    n, b, v, tdt = case["steps"], case["batch"], case["vocab"], DTYPES[case["dtype"]][0]
    s, g = _attention(case, seed, reach=n), _gen(seed + 9)
    q = _normal(g, (n, b, case["q_heads"], case["head_dim"]), tdt)
    k = _normal(g, (n, b, case["kv_heads"], case["head_dim"]), tdt)
    vv, logits = _normal(g, (n, b, case["kv_heads"], case["head_dim"]), tdt), _logits(g, n * b, v, 1.0, 5)
    outs, toks, lps = [], [], []
    for t in range(n):
        outs.append(_attend(case, s.arena, s.table, s.ctx_host + t, q[t]))
        tok, lp = _sample_all(case, logits[t * b:(t + 1) * b], _seeds(seed, b), (s.ctx_host + t).tolist(), range(b))
        toks.append(tok)
        lps.append(lp)
        _appended(case, s.arena, s.table, s.ctx_host + t, k[t], vv[t])
    rows = torch.arange(b, dtype=torch.int32).repeat(n, 1)
    return torch.stack(outs), torch.stack(toks), torch.stack(lps), rows, s.arena.double(), None
