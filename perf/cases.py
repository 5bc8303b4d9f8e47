"""Timed cases of the kda355 entry points: what a serving or evaluation program asks of one GPU.

A case is a dict of plain values.  `op` names the entry point:
  chunk_kda    the plain call with given fp32 log-decays and activated beta; `lens` are the packed sequence lengths,
               `state` is "none", "dense" (initial_state [N, H, 128, 128]) or "pool" (paged pool, one slot per
               sequence), `every` > 0 writes checkpoints every so many tokens into `ck` ("bf16" / "fp32") rows
  kda_prefill  the plain call with gates, beta and q / k norms in the kernel and dense initial states
  prefill      one chunked-prefill step of a serving engine on its page layout; `seqs` lists
               tokens:has_initial_state:checkpoint offset per sequence
  decode       the fused decode step (conv, norms, recurrence, gated RMSNorm) on the page layout; S > 1 is a
               speculative verify of S tokens
  recurrent    fused_recurrent_kda on a state pool; S > 1 verifies S draft tokens into a scratch and commits the
               accepted length
Layouts are planned in prepare() as an engine plans them: once per step, shared by every layer.
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "eat-kernels_amd"))
import kda355  # noqa: E402

D = 128
LOWER_BOUND = -5.0
NORM_EPS = 1e-5
PAGE_TAPS = 10  # conv taps a page holds: 2 + 8 speculative tokens
DEV = "cuda"


def listed():
    return [
        # an evaluation or training-style batch of ragged documents through the fla call (the benchmark's headline)
        dict(name="plain_8seq_39k_h32", op="chunk_kda", lens="4011,4318,6249,7799,532,1400,6787,7785", H=32, state="dense",
             every=0, ck="bf16", precise=False),
        # one long document, state in a paged pool, bf16 prefix-cache checkpoints every 4,096 tokens
        dict(name="plain_1seq_131k_h32_ck", op="chunk_kda", lens="131072", H=32, state="pool", every=4096, ck="bf16",
             precise=False),
        # a first look at the operator: one short document, few heads, no initial state
        dict(name="plain_1seq_1k_h4", op="chunk_kda", lens="1024", H=4, state="none", every=0, ck="bf16", precise=False),
        # serving under light load: one request's next turn at 12 heads (a tensor-parallel share)
        dict(name="step_1600_h12", op="prefill", seqs="1600:1:640", H=12, precise=False),
        # serving under load at 12 heads: a 16k-token step of many requests, most with a prefix hit and a checkpoint
        dict(name="step_12seq_16k_h12", op="prefill", H=12, precise=False,
             seqs="3008:1:3008,1536:1:1536,256:1:64,128:0:0,1600:1:832,640:1:0,576:1:0,512:1:0,448:1:0,2560:1:2560,"
                  "320:1:256,4288:1:3712"),
        # serving under load with all 96 heads on the GPU: one long prompt's chunk
        dict(name="step_8192_h96", op="prefill", seqs="8192:1:7616", H=96, precise=False),
        # a batch of many short prompts of one length
        dict(name="gated_32x512_h12", op="kda_prefill", lens=",".join(["512"] * 32), H=12, precise=False),
        # prompts of very different lengths, ragged ends among them
        dict(name="gated_mixed_h12", op="kda_prefill", lens="8192,1024,777,512,256,130,64,17", H=12, precise=False),
        # the smallest call: one user's next token
        dict(name="decode_b1_h12", op="decode", H=12, B=1, S=1),
        # speculative verify of 8 tokens for a small batch
        dict(name="verify_b16_s8_h12", op="decode", H=12, B=16, S=8),
        # decode of a large batch through the recurrent entry point
        dict(name="recurrent_b256_h32", op="recurrent", H=32, B=256, S=1, raw=False),
        # speculative verify with a scratch and the commit of the accepted lengths
        dict(name="recurrent_verify_b64_s4_h64", op="recurrent", H=64, B=64, S=4, raw=False),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_lens(rng, tokens, most, longest):
    """About `tokens` tokens in up to `most` sequences of at most `longest`: equal, ragged or one of them dominant."""
    n = min(_log_uniform(rng, 1, most), max(1, tokens // 16))
    n = max(n, -(-tokens // longest))
    style = rng.randrange(3)
    if style == 0:
        w = [1.0] * n
    elif style == 1:
        w = [rng.uniform(0.1, 1.9) for _ in range(n)]
    else:
        w = [1.0] * n
        w[rng.randrange(n)] = float(n)
    return [max(1, min(longest, int(tokens * x / sum(w)))) for x in w]


def draw(rng):
    op = rng.choice(["chunk_kda", "chunk_kda", "kda_prefill", "kda_prefill", "prefill", "prefill", "decode", "recurrent"])
    if op in ("chunk_kda", "kda_prefill", "prefill"):
        H = rng.choice([1, 2, 4, 8, 12, 12, 16, 24, 32, 48, 64, 96])
        tokens = max(1, _log_uniform(rng, 2000, 1200000) // H)
        lens = _draw_lens(rng, tokens, 64, 32768)
        precise = rng.random() < 0.15
        if op == "prefill":
            seqs = []
            for n in lens:
                off = 64 * rng.randrange(n // 64 + 1) if rng.random() < 0.6 else 0
                seqs.append("%d:%d:%d" % (n, rng.random() < 0.75, off))
            return dict(op=op, H=H, seqs=",".join(seqs), precise=precise)
        text = ",".join(str(n) for n in lens)
        if op == "kda_prefill":
            return dict(op=op, H=H, lens=text, precise=precise)
        return dict(op=op, H=H, lens=text, state=rng.choice(["none", "dense", "dense", "pool"]),
                    every=rng.choice([0, 0, 0, 64 * _log_uniform(rng, 4, 64)]), ck=rng.choice(["bf16", "fp32"]),
                    precise=precise)
    H = rng.choice([8, 12, 12, 16, 24, 32, 64, 96])
    S = rng.choice([1, 1, 1, 2, 3, 4, 6, 8])
    S = S if op == "decode" else min(S, 4)
    B = _log_uniform(rng, 1, 12288 // (H * S))
    if op == "decode":
        return dict(op=op, H=H, B=B, S=S)
    return dict(op=op, H=H, B=B, S=S, raw=rng.random() < 0.5)


# ---------------------------------------------------------------------------------------------------- inputs
def _lens(case):
    if case["op"] == "prefill":
        return [int(s.split(":")[0]) for s in case["seqs"].split(",")]
    return [int(s) for s in case["lens"].split(",")]


def _offsets(lens):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return cu


class _Random:
    """Device normals from one seeded generator."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV).manual_seed(seed)
        self.cpu = torch.Generator().manual_seed(seed)

    def normal(self, *shape, scale=1.0):
        x = torch.randn(*shape, generator=self.gen, device=DEV)
        return x.mul_(scale) if scale != 1.0 else x

    def bf16(self, *shape):
        return self.normal(*shape).bfloat16()

    def slots(self, count, slots):
        """Distinct rows of a pool whose row 0 is reserved."""
        return (torch.randperm(slots - 1, generator=self.cpu)[:count] + 1).to(torch.int32)


def _plain_tokens(r, T, H):
    """q, k unit vectors, v normal (bf16); g = -softplus(N(0, 1)) and beta = sigmoid(N(0, 1)) (fp32)."""
    unit = lambda: torch.nn.functional.normalize(r.normal(1, T, H, D), dim=-1).bfloat16()  # noqa: E731
    q, k, v = unit(), unit(), r.bf16(1, T, H, D)
    g = -torch.nn.functional.softplus(r.normal(1, T, H, D))
    return q, k, v, g, torch.sigmoid(r.normal(1, T, H))


def _gate_params(r, H):
    A_log = torch.rand(H, generator=r.gen, device=DEV) * 2 - 1
    return A_log, r.normal(H * D, scale=0.5)


def _page_pool(r, slots, taps, H):
    """Conv and SSM states as strided views into one byte pool of pages (conv first, the page padded)."""
    dim = H * D
    conv_bytes = taps * 3 * dim * 2
    page = -(-(conv_bytes + H * D * D * 4 + 4096) // 256) * 256
    raw = torch.zeros(slots * page, dtype=torch.uint8, device=DEV)
    conv = torch.as_strided(raw.view(torch.bfloat16), (slots, taps, 3 * dim), (page // 2, 3 * dim, 1), 0)
    ssm = torch.as_strided(raw.view(torch.float32), (slots, H, D, D), (page // 4, D * D, D, 1), conv_bytes // 4)
    conv.copy_(r.bf16(slots, taps, 3 * dim))
    ssm.copy_(r.normal(slots, H, D, D, scale=0.05))
    return conv, ssm


def _projection(r, T, H):
    """One input projection's rows: q | k | v | out_gate | 128 others | beta, as column slices."""
    dim = H * D
    width = -(-(4 * dim + D + H) // 16) * 16
    P = r.bf16(T, width)
    return P[:, :3 * dim], P[:, 3 * dim:4 * dim], P[:, 4 * dim + D:4 * dim + D + H]


def prepare(case, seed):
    r = _Random(seed)
    return dict(_PREPARE[case["op"]](case, r), case=dict(case))


def _prepare_chunk(case, r):
    lens, H = _lens(case), case["H"]
    T, N, every = sum(lens), len(lens), case["every"]
    s = dict(zip("qkvgb", _plain_tokens(r, T, H)))
    cu = torch.tensor(_offsets(lens), dtype=torch.int32)
    s["meta"] = kda355.plan(cu, H, ck_every=every, device=DEV)
    s["kw"] = kw = dict(precise=case["precise"])
    s["init"] = None
    if case["state"] == "dense":
        s["init"] = r.normal(N, H, D, D, scale=0.02)
    elif case["state"] == "pool":
        slots = 2 * N + 6
        s["init"] = r.normal(slots, H, D, D, scale=0.02)
        kw["ssm_state_indices"] = r.slots(N, slots).to(DEV)
    if every:
        rows = s["meta"].ck_rows
        s["ck"] = torch.zeros(rows + 8, H, D, D, dtype=torch.bfloat16 if case["ck"] == "bf16" else torch.float32, device=DEV)
        kw.update(state_checkpoints=s["ck"], checkpoint_every_n_tokens=every,
                  checkpoint_state_indices=torch.randperm(rows + 8, generator=r.cpu)[:rows].to(torch.int32).to(DEV))
    s["workspace"] = torch.empty(max(256, s["meta"].workspace_bytes), dtype=torch.uint8, device=DEV)
    return s


def _prepare_gated(case, r):
    lens, H = _lens(case), case["H"]
    T, N = sum(lens), len(lens)
    s = {n: r.bf16(1, T, H, D) for n in "qkvg"}
    s["b"] = r.bf16(1, T, H)
    s["A_log"], s["dt_bias"] = _gate_params(r, H)
    s["init"] = r.normal(N, H, D, D, scale=0.05)
    cu = torch.tensor(_offsets(lens), dtype=torch.int32)
    s["meta"], s["cu"] = kda355.plan(cu, H, device=DEV), cu.to(DEV)
    return s


def _prepare_step(case, r):
    lens, H = _lens(case), case["H"]
    T, N, dim = sum(lens), len(lens), case["H"] * D
    slots = 2 * N + 9
    s = {}
    _, s["pool"] = _page_pool(r, slots, PAGE_TAPS, H)
    for n in "qkvg":
        s[n] = r.bf16(1, T, H, D)
    s["b"] = _projection(r, T, H)[2].unsqueeze(0)
    s["A_log"], s["dt_bias"] = _gate_params(r, H)
    parts = [p.split(":") for p in case["seqs"].split(",")]
    rows = r.slots(2 * N, slots)
    off = torch.tensor([int(p[2]) for p in parts], dtype=torch.int32)
    ck = torch.where(off > 0, rows[N:], torch.full_like(off, -1))
    cu = torch.tensor(_offsets(lens), dtype=torch.int32)
    s["meta"] = kda355.prefill_prepare(cu, H, off, ck, device=DEV)
    s["idx"], s["off"], s["ck"], s["cu"] = rows[:N].contiguous().to(DEV), off.to(DEV), ck.to(DEV), cu.to(DEV)
    s["has_init"] = torch.tensor([p[1] == "1" for p in parts], device=DEV)
    s["out"] = torch.zeros(1, T + 64, H, D, dtype=torch.bfloat16, device=DEV)[:, 64:]
    s["workspace"] = torch.empty(max(256, s["meta"].workspace_bytes), dtype=torch.uint8, device=DEV)
    return s


def _prepare_decode(case, r):
    H, B, S = case["H"], case["B"], case["S"]
    T, dim = B * S, case["H"] * D
    slots = 2 * T + 16
    s = {}
    s["conv"], s["pool"] = _page_pool(r, slots, 3 if S == 1 else 2 + S, H)
    s["mixed"], s["out_gate"], s["b"] = _projection(r, T, H)
    s["g"] = r.bf16(T, H, D)
    s["conv_weight"] = r.normal(3, 4, dim, scale=0.4)
    s["A_log"], s["dt_bias"] = _gate_params(r, H)
    s["norm_weight"] = 1 + r.normal(D, scale=0.1)
    rows = r.slots(T, slots)
    s["idx"] = (rows if S == 1 else rows.view(B, S)).contiguous().to(DEV)
    s["acc"] = None if S == 1 else torch.randint(1, S + 1, (B,), generator=r.cpu, dtype=torch.int32).to(DEV)
    s["cu"] = torch.arange(0, T + 1, S, dtype=torch.int32, device=DEV)
    s["out"] = torch.zeros(T, dim, dtype=torch.bfloat16, device=DEV)
    return s


def _prepare_recurrent(case, r):
    H, B, S = case["H"], case["B"], case["S"]
    T, slots = B * S, 2 * B + 8
    s = dict(zip("qkvgb", _plain_tokens(r, T, H)))
    if case["raw"]:
        s["g"], s["b"] = r.bf16(1, T, H, D), r.bf16(1, T, H)
        s["A_log"], s["dt_bias"] = _gate_params(r, H)
    s["pool"] = r.normal(slots, H, D, D, scale=0.05)
    rows = r.slots(B, slots).to(DEV)
    s["slot"] = rows
    s["cu"] = torch.arange(0, T + 1, S, dtype=torch.int32, device=DEV)
    s["out"] = torch.zeros(1, T, H, D, dtype=torch.bfloat16, device=DEV)
    if S > 1:
        s["idx"] = rows.view(B, 1).expand(B, S).contiguous()
        s["scratch"] = torch.zeros(T, H, D, D, device=DEV)
        s["scratch_idx"] = torch.arange(T, dtype=torch.int32, device=DEV).view(B, S)
        s["acc"] = torch.randint(1, S + 1, (B,), generator=r.cpu, dtype=torch.int32).to(DEV)
    return s


_PREPARE = dict(chunk_kda=_prepare_chunk, kda_prefill=_prepare_gated, prefill=_prepare_step, decode=_prepare_decode,
                recurrent=_prepare_recurrent)


# ---------------------------------------------------------------------------------------------------- one pass
def run(s):
    case = s["case"]
    op = case["op"]
    if op == "chunk_kda":
        got = kda355.chunk_kda(s["q"], s["k"], s["v"], s["g"], s["b"], initial_state=s["init"], meta=s["meta"],
                               workspace=s["workspace"], **s["kw"])
        return dict(zip(("out", "state", "checkpoints"), got))
    if op == "kda_prefill":
        out, state = kda355.kda_prefill(s["q"], s["k"], s["v"], s["g"], s["b"], s["A_log"], s["dt_bias"], s["init"], s["cu"],
                                        lower_bound=LOWER_BOUND, meta=s["meta"], precise=case["precise"])
        return dict(out=out, state=state)
    if op == "prefill":
        kda355.prefill(s["q"], s["k"], s["v"], s["g"], s["b"], s["A_log"], s["dt_bias"], D ** -0.5, LOWER_BOUND, s["pool"],
                       s["idx"], s["has_init"], s["cu"], s["out"], s["off"], s["ck"], meta=s["meta"],
                       workspace=s["workspace"], precise=case["precise"])
        return dict(out=s["out"], pool=s["pool"])
    if op == "decode":
        kda355.decode(s["mixed"], s["conv"], s["conv_weight"], s["g"], s["b"], s["out_gate"], s["A_log"], s["dt_bias"],
                      s["norm_weight"], s["pool"], s["idx"], s["acc"], s["cu"], NORM_EPS, LOWER_BOUND, s["out"])
        return dict(out=s["out"], conv=s["conv"], pool=s["pool"])
    gates = (dict(raw_g=s["g"], raw_beta=s["b"], A_log=s["A_log"], dt_bias=s["dt_bias"], lower_bound=LOWER_BOUND)
             if case["raw"] else dict(g=s["g"], beta=s["b"]))
    if case["S"] == 1:
        kda355.fused_recurrent_kda(s["q"], s["k"], s["v"], initial_state=s["pool"], cu_seqlens=s["cu"],
                                   ssm_state_indices=s["slot"], out=s["out"], **gates)
        return dict(out=s["out"], pool=s["pool"])
    kda355.fused_recurrent_kda(s["q"], s["k"], s["v"], initial_state=s["pool"], cu_seqlens=s["cu"],
                               ssm_state_indices=s["idx"], num_accepted_tokens=s["acc"], out=s["out"],
                               write_pool=s["scratch"], write_indices=s["scratch_idx"], **gates)
    kda355.spec_commit(s["scratch"], s["scratch_idx"], s["pool"], s["slot"], s["acc"])
    return dict(out=s["out"], pool=s["pool"], scratch=s["scratch"])


# ---------------------------------------------------------------------------------------------------- work
def work(case):
    """Compulsory bytes (inputs read once, outputs written once) and the chunked or recurrent form's FLOPs."""
    H, state = case["H"], D * D * 4
    if case["op"] in ("decode", "recurrent"):
        B, S = case["B"], case["S"]
        flops = B * S * H * 7.0 * D * D  # decay, S k, rank-1 update, S q
        if case["op"] == "decode":
            taps = 3 if S == 1 else 2 + S
            bytes_ = B * H * (state * (1 + S) + (3 + taps) * 3 * D * 2 + S * (3 * D * 2 + D * 2 + 2 + D * 2 + D * 2))
            return dict(bytes=bytes_ + H * (12 * D * 4 + D * 4 + 4), flops=flops)
        token = 3 * D * 2 + (D * 2 + 2 if case["raw"] else D * 4 + 4) + D * 2
        commit = 2 if S > 1 else 0
        return dict(bytes=B * H * (state * (1 + S + commit) + S * token), flops=flops)
    lens = _lens(case)
    T, N = sum(lens), len(lens)
    flops = 0.0
    for n in lens:
        for c, count in ((64, n // 64), (n % 64, 1)):
            flops += count * (6.0 * c * D * D + 10.0 * c * c * D + 2.0 / 3.0 * c ** 3)
    given = case["op"] == "chunk_kda"
    bytes_ = T * H * (3 * D * 2 + (D * 4 + 4 if given else D * 2 + 2) + D * 2)
    if case["op"] == "prefill":
        parts = [p.split(":") for p in case["seqs"].split(",")]
        rows = N + sum(p[1] == "1" for p in parts) + sum(int(p[2]) > 0 for p in parts)
    else:
        rows = N * (1 if given and case["state"] == "none" else 2)
        if given and case["every"]:
            rows += sum(-(-n // case["every"]) for n in lens) * (0.5 if case["ck"] == "bf16" else 1)
    return dict(bytes=bytes_ + rows * H * state, flops=flops * H)


def tolerance(case):
    # Outputs are bf16: two correct implementations differ by about one rounding (2^-9 relative), twice for the fused
    # decode, whose recurrence output is rounded before its norm; measured against exact(): 1.7e-3, decode 2.3e-3.  A single
    # output near a rounding boundary differs by one bf16 step of its own size, or, where large terms cancel, by the
    # fp16 operands' error of a typical output.
    return dict(rel=8e-3, max=0.1)


# ---------------------------------------------------------------------------------------------------- 64-bit results
def _walk64(q, k, v, g, beta, lens, S0, scale, marks=()):
    """Token recurrence in fp64 over [T, H, ...] inputs, all sequences side by side.  S0 [N, H, V, K].  Returns the
    outputs, the final states and {(n, t): state of sequence n after t tokens} for the (n, t) in marks."""
    N, H = S0.shape[0], S0.shape[1]
    order = sorted(range(N), key=lambda n: -lens[n])
    start = torch.tensor([_offsets(lens)[n] for n in order], device=DEV)
    S = S0[order].double().contiguous()
    out = torch.zeros(q.shape[0], H, D, dtype=torch.float64, device=DEV)
    want = {}
    for n, t in marks:
        want.setdefault(t, []).append(n)
    place = {n: i for i, n in enumerate(order)}
    snaps = {(n, 0): S[place[n]].clone() for n in want.get(0, [])}
    live = N
    for t0 in range(0, max(lens), 256):
        while lens[order[live - 1]] <= t0:
            live -= 1
        n = live
        steps = min(256, max(lens) - t0)
        tok = (start[:live].view(1, -1) + torch.arange(t0, t0 + steps, device=DEV).view(-1, 1)).clamp(max=q.shape[0] - 1)
        bq, bk, bv, bd = q[tok].double(), k[tok].double(), v[tok].double(), g[tok].double().exp()
        bb = beta[tok].double()
        bo = torch.zeros_like(bq)
        for i in range(steps):
            while lens[order[n - 1]] <= t0 + i:  # sequences run longest first, so the ones still running lead
                n -= 1
            X = S[:n]
            X.mul_(bd[i, :n].unsqueeze(-2))
            kk = bk[i, :n]
            u = bb[i, :n].unsqueeze(-1) * (bv[i, :n] - (X @ kk.unsqueeze(-1)).squeeze(-1))
            X.addcmul_(u.unsqueeze(-1), kk.unsqueeze(-2))
            bo[i, :n] = (X @ bq[i, :n].unsqueeze(-1)).squeeze(-1)
            for m in want.get(t0 + i + 1, ()):
                snaps[m, t0 + i + 1] = S[place[m]].clone()
        for j in range(live):
            c = min(steps, lens[order[j]] - t0)
            a = int(start[j]) + t0
            out[a:a + c] = bo[:c, j] * scale
    final = torch.empty_like(S)
    final[order] = S
    return out, final, snaps


def _unit64(x):
    x = x.double()
    return x / x.norm(dim=-1, keepdim=True).clamp(min=1e-6)


def _gate64(raw, A_log, dt_bias):
    H = A_log.numel()
    return LOWER_BOUND * torch.sigmoid(A_log.double().exp().view(H, 1) * (raw.double() + dt_bias.double().view(H, D)))


def exact(case, seed):
    return _EXACT[case["op"]](case, prepare(case, seed))


def _exact_chunk(case, s):
    lens, H, every = _lens(case), case["H"], case["every"]
    N = len(lens)
    if case["state"] == "none":
        S0 = torch.zeros(N, H, D, D, device=DEV)
    else:
        S0 = s["init"] if case["state"] == "dense" else s["init"][s["kw"]["ssm_state_indices"].long()]
    marks = [(n, j * every) for n in range(N) for j in range(-(-lens[n] // every))] if every else []
    o, fin, snaps = _walk64(_unit64(s["q"][0]), _unit64(s["k"][0]), s["v"][0], s["g"][0], s["b"][0], lens, S0, D ** -0.5, marks)
    state = fin
    if case["state"] == "pool":
        state = s["init"].double()
        state[s["kw"]["ssm_state_indices"].long()] = fin
    got = dict(out=o.unsqueeze(0), state=state)
    if every:
        got["checkpoints"] = s["ck"].double()
        for row, m in zip(s["kw"]["checkpoint_state_indices"].tolist(), marks):
            got["checkpoints"][row] = snaps[m]
    return got


def _exact_gated(case, s):
    o, fin, _ = _walk64(_unit64(s["q"][0]), _unit64(s["k"][0]), s["v"][0], _gate64(s["g"][0], s["A_log"], s["dt_bias"]),
                        torch.sigmoid(s["b"][0].double()), _lens(case), s["init"], D ** -0.5)
    return dict(out=o.unsqueeze(0), state=fin)


def _exact_step(case, s):
    lens = _lens(case)
    S0 = s["pool"][s["idx"].long()] * s["has_init"].view(-1, 1, 1, 1)
    ck = s["ck"].tolist()
    marks = [(n, int(s["off"][n])) for n in range(len(lens)) if ck[n] >= 0]
    o, fin, snaps = _walk64(_unit64(s["q"][0]), _unit64(s["k"][0]), s["v"][0], _gate64(s["g"][0], s["A_log"], s["dt_bias"]),
                            torch.sigmoid(s["b"][0].double()), lens, S0, D ** -0.5, marks)
    pool = s["pool"].double()
    pool[s["idx"].long()] = fin
    for m in marks:
        pool[ck[m[0]]] = snaps[m]
    return dict(out=o.unsqueeze(0), pool=pool)


def _token64(S, q, k, v, g, beta):
    """One token for every (sequence, head): S [B, H, V, K] updated in place; returns S q."""
    S.mul_(g.exp().unsqueeze(-2))
    u = beta.unsqueeze(-1) * (v - (S @ k.unsqueeze(-1)).squeeze(-1))
    S.addcmul_(u.unsqueeze(-1), k.unsqueeze(-2))
    return (S @ q.unsqueeze(-1)).squeeze(-1)


def _rsqrt64(x):
    return x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def _exact_decode(case, s):
    H, B, S = case["H"], case["B"], case["S"]
    dim = H * D
    idx = s["idx"].long().view(B, S)
    start = (s["acc"] - 1).long() if S > 1 else torch.zeros(B, dtype=torch.long, device=DEV)
    conv, pool = s["conv"].double(), s["pool"].double()
    rows = idx[torch.arange(B, device=DEV), start]
    taps = start.view(B, 1) + torch.arange(3, device=DEV)
    window = torch.cat([conv[idx[:, :1], taps], s["mixed"].double().view(B, S, 3 * dim)], 1)  # [B, 3 + S, 3 dim]
    w = s["conv_weight"].double().permute(1, 0, 2).reshape(4, 3 * dim)
    x = sum(window[:, j:j + S] * w[j] for j in range(4))
    x = (x * torch.sigmoid(x)).view(B, S, 3, H, D)
    keep = 3 if S == 1 else 2 + S
    conv[idx[:, 0], :keep] = window[:, -keep:]
    g = _gate64(s["g"], s["A_log"], s["dt_bias"]).view(B, S, H, D)
    beta = torch.sigmoid(s["b"].double()).view(B, S, H)
    og = torch.sigmoid(s["out_gate"].double()).view(B, S, H, D)
    state = pool[rows]
    out = torch.empty(B, S, H, D, dtype=torch.float64, device=DEV)
    for t in range(S):
        o = _token64(state, _rsqrt64(x[:, t, 0]) * D ** -0.5, _rsqrt64(x[:, t, 1]), x[:, t, 2], g[:, t], beta[:, t])
        out[:, t] = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + NORM_EPS) * s["norm_weight"].double() * og[:, t]
        pool[idx[:, t]] = state
    return dict(out=out.view(B * S, dim), conv=conv, pool=pool)


def _exact_recurrent(case, s):
    H, B, S = case["H"], case["B"], case["S"]
    per = lambda t: t[0].double().view(B, S, *t.shape[2:])  # noqa: E731
    q, k, v = _rsqrt64(per(s["q"])), _rsqrt64(per(s["k"])), per(s["v"])
    g, beta = per(s["g"]), per(s["b"])
    if case["raw"]:
        g, beta = _gate64(g, s["A_log"], s["dt_bias"]), torch.sigmoid(beta)
    pool = s["pool"].double()
    state = pool[s["slot"].long()]
    out = torch.empty(B, S, H, D, dtype=torch.float64, device=DEV)
    scratch = torch.empty(B, S, H, D, D, dtype=torch.float64, device=DEV)
    for t in range(S):
        out[:, t] = _token64(state, q[:, t], k[:, t], v[:, t], g[:, t], beta[:, t]) * D ** -0.5
        scratch[:, t] = state
    got = dict(out=out.view(1, B * S, H, D))
    pool[s["slot"].long()] = state if S == 1 else scratch[torch.arange(B, device=DEV), (s["acc"] - 1).long()]
    got["pool"] = pool
    if S > 1:
        got["scratch"] = scratch.view(B * S, H, D, D)
    return got


_EXACT = dict(chunk_kda=_exact_chunk, kda_prefill=_exact_gated, prefill=_exact_step, decode=_exact_decode,
              recurrent=_exact_recurrent)
