"""What a user of this framework has it do, as cases that can be timed and compared.

Three families, through the public entry points only:

* ``kv``: one transfer of paged KV blocks between a pool and a staging buffer.  The pool and the
  buffer are prepared once as descriptor lists; every pass makes a request from two index
  vectors (the block list is new each time in a serving loop), posts it, polls it to completion
  and releases it.
* ``list``: transfers of descriptors that are no equal blocks.  ``small``: part of a prepared
  list of unequal lengths, by index; ``bytes``: explicit lists at any byte address and length;
  ``tensors``: whole tensors whose request is made once and posted again and again.
* ``ll`` and ``ht``: one mixture-of-experts layer's communication, low-latency (decode) and
  normal mode (prefill, training): dispatch, then combine of what the experts made of it.

Block shapes come from nixl_amd/kvshape.py, the expert-parallel shapes from the benchmark and
the tests of this repository.
"""
import itertools
import math

import numpy as np
import torch

from nixl_amd import kvshape, nixl_agent
from nixl_amd.ep import Buffer

_DEV = "cuda:0"
_names = itertools.count()
_MODELS = ("LLAMA3.1_8B", "LLAMA3.1_70B", "DEEPSEEK_R1", "QWEN3_8B", "GPT_OSS_20B")
_ONE_GIB = 1 << 30
_PIECES = 64  # consecutive pieces of a prepared list that belong to one block


def listed():
    return [
        # A decode instance pulls the one block a running sequence has just filled: 64 descriptors,
        # 2 MiB.  Time is latency.
        {"name": "kv_pull_one_block", "path": "kv", "op": "pull", "model": "LLAMA3.1_8B", "precision": "bfloat16",
         "block_tokens": 16, "blocks": 1, "pool_blocks": 512, "order": "layer"},
        # One prompt of 4000 tokens leaves a latent-attention cache: 61 layers, 9 KiB a block.
        {"name": "kv_gather_prompt", "path": "kv", "op": "gather", "model": "DEEPSEEK_R1", "precision": "fp8",
         "block_tokens": 16, "blocks": 250, "pool_blocks": 2048, "order": "layer"},
        # The benchmark's step: 1024 blocks of 8 tokens of a batch gathered (65 536 descriptors of
        # 16 KiB, 1 GiB), then scattered to other blocks of a second pool.
        {"name": "kv_batch_there_and_back", "path": "kv", "op": "both", "model": "LLAMA3.1_8B", "precision": "bfloat16",
         "block_tokens": 8, "blocks": 1024, "pool_blocks": 8192, "order": "layer"},
        # The small-descriptor stress of the benchmark: 262 144 pieces of 512 B to 4 KiB at random
        # 16-byte addresses, half of a list that was prepared once (caches whose layers keep states
        # of different sizes: a request names blocks, a block is 64 consecutive pieces).
        {"name": "list_small", "path": "list", "form": "small", "count": 262144, "min_bytes": 512, "max_bytes": 4096,
         "buffer_mib": 4096},
        # Odd leftovers that travel beside the blocks (token ids, scales, partial blocks): explicit
        # lists, any byte address, 1 B to 64 KiB.
        {"name": "list_bytes", "path": "list", "form": "bytes", "count": 3000, "min_bytes": 1, "max_bytes": 65536,
         "buffer_mib": 512},
        # New weights for an engine: 40 whole tensors of 1 to 128 MiB, the same request every time.
        {"name": "list_tensors", "path": "list", "form": "tensors", "count": 40, "min_bytes": 1 << 20, "max_bytes": 128 << 20,
         "buffer_mib": 0},
        # A decode step with two sequences a rank: latency and launches.
        {"name": "ll_step_two_tokens", "path": "ll", "ranks": 8, "tokens": 2, "hidden": 7168, "topk": 8, "experts": 256,
         "max_tokens": 128, "rows": "fp8", "scales": "float", "routed": False},
        # A full decode step: 32 ranks x 128 tokens, top-8 of 256 experts, fp8 rows.
        {"name": "ll_step", "path": "ll", "ranks": 32, "tokens": 128, "hidden": 7168, "topk": 8, "experts": 256,
         "max_tokens": 128, "rows": "fp8", "scales": "float", "routed": False},
        # A smaller layer in bf16 at an odd batch, from the router's logits.
        {"name": "ll_step_bf16_routed", "path": "ll", "ranks": 16, "tokens": 61, "hidden": 2560, "topk": 6, "experts": 64,
         "max_tokens": 64, "rows": "bf16", "scales": "float", "routed": True},
        # Prefill: 8 ranks x 4096 tokens, uneven (Zipf) expert popularity, bf16 rows.
        {"name": "ht_prefill", "path": "ht", "ranks": 8, "tokens": 4096, "hidden": 7168, "topk": 8, "experts": 256,
         "rows": "bf16", "backward": False},
        # Prefill of one short prompt, fp8 rows with their scales, odd token count.
        {"name": "ht_prompt_fp8", "path": "ht", "ranks": 4, "tokens": 333, "hidden": 4096, "topk": 6, "experts": 64,
         "rows": "fp8", "backward": False},
        # A training step's layer: forward, and backward through the kept layout (the gradient of
        # combine is a dispatch, that of dispatch a combine).
        {"name": "ht_train", "path": "ht", "ranks": 8, "tokens": 1024, "hidden": 4096, "topk": 4, "experts": 64,
         "rows": "bf16", "backward": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: blocks, lists and layers from the smallest listed to the largest."""
    path = rng.choice(["kv", "kv", "list", "ll", "ll", "ht", "ht"])
    if path == "kv":
        case = {"path": "kv", "op": rng.choice(["pull", "gather", "scatter"]), "model": rng.choice(_MODELS),
                "precision": rng.choice(["bfloat16", "fp8"]), "block_tokens": rng.choice([8, 16, 32, 64])}
        lay = _layout(case)
        case["blocks"] = _log_int(rng, 1, min(1024, _ONE_GIB // lay.bytes_per_block))
        case["pool_blocks"] = min(case["blocks"] * rng.choice([2, 5, 8]) + rng.randrange(1, 64), 8 * _ONE_GIB // lay.bytes_per_block)
        case["order"] = rng.choice(["layer", "block"])
        return case
    if path == "list":
        form = rng.choice(["small", "bytes", "tensors"])
        if form == "small":
            count = _PIECES * _log_int(rng, 1, 4096)
            return {"path": "list", "form": form, "count": count, "min_bytes": rng.choice([256, 512]),
                    "max_bytes": rng.choice([2048, 4096]), "buffer_mib": max(64, count * 16384 >> 20)}
        if form == "bytes":
            count = _log_int(rng, 16, 3000)
            return {"path": "list", "form": form, "count": count, "min_bytes": 1, "max_bytes": rng.choice([4096, 65536]),
                    "buffer_mib": 512}
        return {"path": "list", "form": form, "count": _log_int(rng, 2, 40), "min_bytes": 1 << 16, "max_bytes": rng.choice([8, 128]) << 20,
                "buffer_mib": 0}
    if path == "ll":
        ranks = rng.choice([2, 4, 8, 16, 32])
        rows = rng.choice(["fp8", "bf16"])
        tokens = _log_int(rng, 1, 128)
        return {"path": "ll", "ranks": ranks, "tokens": tokens, "hidden": rng.choice([2048, 2560, 4096, 5120, 7168]),
                "topk": rng.choice([2, 4, 6, 8]), "experts": rng.choice([32, 64, 128, 256]),
                "max_tokens": rng.choice([tokens, 128]), "rows": rows,
                "scales": rng.choice(["float", "ue8m0"]) if rows == "fp8" else "float", "routed": rng.random() < 0.35}
    backward = rng.random() < 0.3
    return {"path": "ht", "ranks": rng.choice([2, 4, 8]), "tokens": _log_int(rng, 32, 1500 if backward else 4096),
            "hidden": rng.choice([2048, 2560, 4096, 7168]), "topk": rng.choice([2, 4, 6, 8]), "experts": rng.choice([16, 64, 128, 256]),
            "rows": "bf16" if backward else rng.choice(["bf16", "fp8"]), "backward": backward}


# ---- transfers ---------------------------------------------------------------------------------


def _layout(case):
    return kvshape.paged_kv_layout(kvshape.model(case["model"]), case["block_tokens"], case["precision"])


def _triples(addrs, lens):
    lens = np.broadcast_to(np.asarray(lens, np.uint64), addrs.shape)
    return np.stack([addrs.astype(np.uint64), lens, np.zeros(addrs.size, np.uint64)], 1)


class _Mover:
    """What a transfer program keeps: its agent, the registered tensors, the prepared lists."""

    def __init__(self, tensors):
        self.name = f"perf{next(_names)}"
        self.agent = nixl_agent(self.name)
        self.tensors = tensors
        self.agent.register_memory(tensors)
        self.handles = []

    def keep(self, handle):
        self.handles.append(handle)
        return handle

    def prepare_list(self, triples, remote):
        return self.keep(self.agent.prep_xfer_dlist(self.name if remote else "", triples, "VRAM"))

    def post_and_wait(self, request):
        state = self.agent.transfer(request)
        while state == "PROC":
            state = self.agent.check_xfer_state(request)
        if state != "DONE":
            raise RuntimeError(f"the transfer ended in state {state}")

    def move(self, op, local, local_idx, remote, remote_idx):
        request = self.agent.make_prepped_xfer(op, local, local_idx, remote, remote_idx)
        self.post_and_wait(request)
        request.release()

    def __del__(self):
        for h in reversed(self.handles):
            h.release()
        self.agent.close()


def _normal_bytes(shape, gen):
    """Values as a bf16 cache or weight holds them (normal), seen as 16-bit words."""
    return torch.empty(shape, dtype=torch.bfloat16, device=_DEV).normal_(generator=gen).view(torch.int16)


def _prepare_kv(case, seed):
    lay = _layout(case)
    blk, lk, n_pool, n = lay.bytes_per_sub_block, lay.descriptors_per_block, case["pool_blocks"], case["blocks"]
    gen = torch.Generator(device=_DEV).manual_seed(seed)
    rng = np.random.default_rng(seed)
    op = case["op"]
    staging_shape = (lk * n, blk // 2)
    pool_shape = (lk, n_pool, blk // 2)
    filled_pool = op in ("gather", "pull", "both")
    pool = _normal_bytes(pool_shape, gen) if filled_pool else torch.zeros(pool_shape, dtype=torch.int16, device=_DEV)
    staging = torch.zeros(staging_shape, dtype=torch.int16, device=_DEV) if filled_pool else _normal_bytes(staging_shape, gen)
    tensors = [pool, staging]
    if op == "both":
        tensors.append(torch.zeros(pool_shape, dtype=torch.int16, device=_DEV))
    mover = _Mover(tensors)
    torch.cuda.synchronize()  # transfers run on the agent's own stream

    in_pool = np.arange(lk * n_pool, dtype=np.uint64) * np.uint64(blk)
    in_staging = np.arange(lk * n, dtype=np.uint64) * np.uint64(blk)

    def indices(ids):
        at = np.arange(lk, dtype=np.int64)[:, None] * n_pool + ids[None, :]
        return np.ascontiguousarray((at if case["order"] == "layer" else at.T).reshape(-1), dtype=np.int32)

    def handle(tensor, offsets, remote):
        return mover.prepare_list(_triples(np.uint64(tensor.data_ptr()) + offsets, blk), remote)

    there = indices(rng.permutation(n_pool)[:n])
    flat = np.arange(lk * n, dtype=np.int32)
    steps = []
    if op == "pull":  # the initiator reads the blocks of the remote pool
        steps.append(("READ", handle(staging, in_staging, False), flat, handle(pool, in_pool, True), there))
    if op in ("gather", "both"):
        steps.append(("WRITE", handle(pool, in_pool, False), there, handle(staging, in_staging, True), flat))
    if op in ("scatter", "both"):
        back = indices(rng.permutation(n_pool)[:n])
        steps.append(("WRITE", handle(staging, in_staging, False), flat, handle(tensors[-1] if op == "both" else pool, in_pool, True), back))
    out = [staging] if op in ("gather", "pull") else [pool] if op == "scatter" else tensors[1:]
    return {"mover": mover, "steps": steps, "out": out}


def _run_kv(s):
    for step in s["steps"]:
        s["mover"].move(*step)
    return s["out"]


def _prepare_list(case, seed):
    gen = torch.Generator(device=_DEV).manual_seed(seed)
    rng = np.random.default_rng(seed)
    n, lo, hi = case["count"] * (2 if case["form"] == "small" else 1), case["min_bytes"], case["max_bytes"]
    lens = np.exp(rng.uniform(math.log(lo), math.log(hi), n)).astype(np.int64)
    if case["form"] == "tensors":
        # lengths spread evenly over the logarithm, so that every seed moves the same number of bytes
        lens = np.exp(np.linspace(math.log(lo), math.log(hi), n)).astype(np.int64) // 2 * 2
        src = [_normal_bytes((int(b) // 2,), gen) for b in lens]
        dst = [torch.zeros_like(t) for t in src]
        mover = _Mover(src + dst)
        torch.cuda.synchronize()
        a = mover.agent
        request = mover.keep(a.initialize_xfer("WRITE", a.get_xfer_descs(src), a.get_xfer_descs(dst), mover.name))
        return {"mover": mover, "request": request, "out": dst}
    size = case["buffer_mib"] << 20
    src = torch.randint(0, 256, (size,), generator=gen, dtype=torch.uint8, device=_DEV)
    dst = torch.zeros(size, dtype=torch.uint8, device=_DEV)
    mover = _Mover([src, dst])
    torch.cuda.synchronize()
    unit = 16 if case["form"] == "small" else 1
    lens = np.maximum(lens // unit * unit, unit)
    # source anywhere (they may overlap), destination inside a slot of its own
    slot = 2 * hi
    so = rng.integers(0, (size - hi) // unit, n) * unit
    do = rng.permutation(size // slot)[:n] * slot + rng.integers(0, hi // unit, n) * unit
    s_triples = _triples(np.uint64(src.data_ptr()) + so.astype(np.uint64), lens)
    d_triples = _triples(np.uint64(dst.data_ptr()) + do.astype(np.uint64), lens)
    if case["form"] == "small":
        blocks = rng.permutation(n // _PIECES)[:n // _PIECES // 2]
        order = (blocks[:, None] * _PIECES + np.arange(_PIECES)).reshape(-1).astype(np.int32)
        return {"mover": mover, "local": mover.prepare_list(s_triples, False), "remote": mover.prepare_list(d_triples, True),
                "order": order, "out": [dst]}
    return {"mover": mover, "src": s_triples, "dst": d_triples, "out": [dst]}


def _run_list(s):
    mover = s["mover"]
    if "request" in s:
        mover.post_and_wait(s["request"])
    elif "order" in s:
        mover.move("WRITE", s["local"], s["order"], s["remote"], s["order"])
    else:
        a = mover.agent
        request = a.initialize_xfer("WRITE", a.get_xfer_descs(s["src"], "VRAM"), a.get_xfer_descs(s["dst"], "VRAM"), mover.name)
        mover.post_and_wait(request)
        request.release()
    return s["out"]


# ---- expert parallelism ------------------------------------------------------------------------


def _zipf_logits(ranks, tokens, experts, gen):
    """Scores whose top-k follows a Zipf(1.2) popularity over a random order of the experts (Gumbel noise)."""
    p = 1.0 / torch.arange(1, experts + 1, device=_DEV, dtype=torch.float32) ** 1.2
    logp = torch.log(p / p.sum())[torch.randperm(experts, generator=gen, device=_DEV)]
    u = torch.rand((ranks, tokens, experts), generator=gen, device=_DEV).clamp_(1e-9, 1 - 1e-7)
    return logp - torch.log(-torch.log(u))


class _ReceivedRows(list):
    """The rows a low-latency dispatch received.  The packed tensors have room for the worst case
    and only the first recv_count rows of an expert mean anything, to the experts as to anyone
    else: those are what this hands out, cut when it is looked at."""

    def __init__(self, packed, scales, src_info, count):
        super().__init__()
        self._parts = (packed, scales, src_info, count)

    def __iter__(self):
        packed, scales, src_info, count = self._parts
        n = packed.shape[2]
        valid = torch.arange(n, device=packed.device) < count.unsqueeze(-1)
        words = packed.view(torch.uint8 if packed.element_size() == 1 else torch.int16)
        yield words[valid]
        yield src_info[valid]
        if scales is not None:
            yield scales[valid]


def _prepare_ll(case, seed):
    R, T, H, E, M = case["ranks"], case["tokens"], case["hidden"], case["experts"], case["max_tokens"]
    gen = torch.Generator(device=_DEV).manual_seed(seed)
    buf = Buffer(R, device=_DEV)
    x = torch.empty((R, T, H), dtype=torch.bfloat16, device=_DEV).normal_(generator=gen)
    logits = torch.randn((R, T, E), generator=gen, device=_DEV)
    topk, weights = buf.route(logits, case["topk"])
    # what the experts hand back, in the layout they received
    y = torch.empty((R, E // R, R * M, H), dtype=torch.bfloat16, device=_DEV).normal_(generator=gen)
    return {"case": case, "buf": buf, "x": x, "logits": logits, "topk": topk, "weights": weights, "y": y}


def _run_ll(s):
    c, buf = s["case"], s["buf"]
    fp8, ue8m0 = c["rows"] == "fp8", c["scales"] == "ue8m0"
    topk, weights = s["topk"], s["weights"]
    if c["routed"]:
        topk, weights, recv, count, handle, _, _ = buf.route_dispatch(s["x"], s["logits"], c["topk"], c["max_tokens"], use_fp8=fp8,
                                                                     round_scale=ue8m0, use_ue8m0=ue8m0)
    else:
        recv, count, handle, _, _ = buf.dispatch(s["x"], topk, c["max_tokens"], c["experts"], use_fp8=fp8, round_scale=ue8m0,
                                                 use_ue8m0=ue8m0)
    combined, _, _ = buf.combine(s["y"], topk, weights, handle)
    packed, scales = recv if fp8 else (recv, None)
    return {"received": _ReceivedRows(packed, scales, handle[0], count), "count": count, "layout": handle[1],
            "topk": topk, "weights": weights, "combined": combined}


def _prepare_ht(case, seed):
    R, T, H, K, E = (case[k] for k in ("ranks", "tokens", "hidden", "topk", "experts"))
    gen = torch.Generator(device=_DEV).manual_seed(seed)
    buf = Buffer(R, low_latency_mode=False, device=_DEV)
    # one routing per shape, its tokens dealt out anew by the seed: every seed moves the same number of rows
    score, topk = torch.topk(_zipf_logits(R, T, E, torch.Generator(device=_DEV).manual_seed(R * T + E)).view(R * T, E), K, dim=1)
    deal = torch.randperm(R * T, generator=gen, device=_DEV)
    weights = torch.softmax(score[deal], dim=1).view(R, T, K).contiguous()
    topk = topk[deal].to(torch.int32).view(R, T, K).contiguous()
    s = {"case": case, "buf": buf, "topk": topk, "weights": weights}
    if case["rows"] == "fp8":
        x = torch.empty((R, T, H), dtype=torch.bfloat16, device=_DEV).normal_(generator=gen).to(torch.float8_e4m3fn)
        scales = torch.rand((R, H // 128, T), generator=gen, device=_DEV).transpose(1, 2)  # stored transposed, as quantisers leave them
        s["x"] = (x, scales)
    else:
        s["x"] = torch.empty((R, T, H), dtype=torch.bfloat16, device=_DEV).normal_(generator=gen)
    hit = torch.zeros((R, T, R), dtype=torch.bool, device=_DEV).scatter_(2, (topk // (E // R)).long(), True)
    s["y"] = torch.empty((int(hit.sum()), H), dtype=torch.bfloat16, device=_DEV).normal_(generator=gen)
    if case["backward"]:
        s["grad"] = torch.empty((R, T, H), dtype=torch.bfloat16, device=_DEV).normal_(generator=gen)
        s["grad_y"] = torch.empty_like(s["y"]).normal_(generator=gen)
    return s


def _bits(t):
    return t.view(torch.uint8 if t.element_size() == 1 else torch.int16)


def _run_ht(s):
    buf = s["buf"]
    per_rank, _, per_expert, in_rank, _ = buf.get_dispatch_layout(s["topk"], s["case"]["experts"])
    recv, idx, w, counts, handle, _ = buf.ht_dispatch(s["x"], num_tokens_per_rank=per_rank, is_token_in_rank=in_rank,
                                                      num_tokens_per_expert=per_expert, topk_idx=s["topk"], topk_weights=s["weights"])
    combined, combined_w, _ = buf.ht_combine(s["y"], handle, topk_weights=w)
    rows, scales = recv if isinstance(recv, tuple) else (recv, None)
    out = {"per_rank": per_rank, "per_expert": per_expert, "rows": _bits(rows), "scales": scales, "idx": idx, "w": w,
           "counts": np.array(counts), "handle": list(handle), "combined": combined, "combined_w": combined_w}
    if s["case"]["backward"]:
        grad_rows, _, _, _, _, _ = buf.ht_dispatch(s["grad"], handle=handle)
        grad_x, _, _ = buf.ht_combine(s["grad_y"], handle)
        out["grad_rows"], out["grad_x"] = _bits(grad_rows), grad_x
    return out


# ---- the interface -----------------------------------------------------------------------------


def prepare(case, seed):
    make = {"kv": _prepare_kv, "list": _prepare_list, "ll": _prepare_ll, "ht": _prepare_ht}[case["path"]]
    return {"run": case["path"], "state": make(case, seed)}


def run(state):
    return {"kv": _run_kv, "list": _run_list, "ll": _run_ll, "ht": _run_ht}[state["run"]](state["state"])


def _expected_rows_per_token(case):
    """Ranks that hold one of a token's experts: mean over a sample of the routing of _prepare_ht."""
    rng = np.random.default_rng(0)
    E, K, R = case["experts"], case["topk"], case["ranks"]
    seen = []
    for _ in range(8):
        logp = -1.2 * np.log(np.arange(1, E + 1))[rng.permutation(E)]
        sel = np.argpartition(-(logp + rng.gumbel(size=(256, E))), K - 1, axis=1)[:, :K] // (E // R)
        seen.append(np.mean([len(set(row)) for row in sel]))
    return float(np.mean(seen))


def work(case):
    if case["path"] == "kv":
        lay = _layout(case)
        n = case["blocks"] * lay.descriptors_per_block * (2 if case["op"] == "both" else 1)
        return {"bytes": n * (2 * lay.bytes_per_sub_block + 8), "flops": 0}  # payload read and written, two indices a block
    if case["path"] == "list":
        n, lo, hi = case["count"], case["min_bytes"], case["max_bytes"]
        mean = (hi - lo) / math.log(hi / lo)  # of a length whose logarithm is uniform
        if case["form"] == "tensors":
            mean = float(np.mean(np.exp(np.linspace(math.log(lo), math.log(hi), n))))
        return {"bytes": n * (2 * mean + 8), "flops": 0}
    tokens, H, K, E = case["ranks"] * case["tokens"], case["hidden"], case["topk"], case["experts"]
    if case["path"] == "ll":
        pairs = tokens * K
        row = H + H // 128 * (1 if case["scales"] == "ue8m0" else 4) if case["rows"] == "fp8" else 2 * H
        select = tokens * (E * 4 + K * 8) if case["routed"] else tokens * K * 4
        dispatch = tokens * H * 2 + select + pairs * (row + 4) + E * (case["ranks"] * 8 + 4)
        combine = pairs * H * 2 + tokens * K * 8 + tokens * H * 2
        return {"bytes": dispatch + combine, "flops": 2 * pairs * H}
    rows = tokens * _expected_rows_per_token(case)
    row = H + H // 128 * 4 if case["rows"] == "fp8" else 2 * H
    select = tokens * (K * 8 + case["ranks"]) + rows * (K * 8 + 8)
    dispatch = (tokens + rows) * row
    combine = (rows + tokens) * H * 2 + (rows + tokens) * K * 4
    back = 2 * (tokens + rows) * H * 2 if case["backward"] else 0
    return {"bytes": select + dispatch + combine + back, "flops": rows * H * (2 if case["backward"] else 1)}


def tolerance(case):
    """Transfers, rows, codes, counts and positions are bytes and whole numbers: exact.  Combine
    sums rows in fp32 and rounds to bf16: against sums in 64 bits the results are off by 1.66e-3
    (2-norm; a half step of bf16, 2^-9 of the value, is the most one value can be off by)."""
    return "exact" if case["path"] in ("kv", "list") else {"rel": 6.6e-3, "max": 8e-3}
