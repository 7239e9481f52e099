"""The work that users of this package have it do, as timed cases: training steps of the attention core, forward-only
evaluation, paged prefill and paged decode, from the smallest calls to the largest, through the public entry points.

`listed()` names them, `draw(rng)` gives further cases of the same ranges, `prepare(case, seed)` makes what a program
holds before the call, `run(state)` is one pass, `work(case)` the bytes and operations a pass cannot do without and
`tolerance(case)` how far another correct implementation at the same precision may be off."""
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "scalable-flash-native-sparse-attention_amd"))

from flash_nsa import HFNSACore, NSAConfig, NSACore, nsa_decode, nsa_prefill  # noqa: E402
from flash_nsa.inference import allocate_kv_pools, mean_pooling_prefill  # noqa: E402

# hyper-parameters of the attention, the same in every case: NSAConfig's defaults
KERNEL, STRIDE, BLOCK, TOP_N, WINDOW = 32, 16, 64, 16, 512

# (q heads, kv heads, qk head dim, v head dim)
WIDE = (64, 4, 128, 128)      # the benchmark's shape
NARROW = (16, 1, 128, 128)    # the shape of the CPU-runnable reference case; also one tensor-parallel shard of WIDE
QK192 = (32, 2, 192, 128)     # separate rotary channels in q and k
SMALL = (16, 2, 64, 64)       # a small model: 8 q-heads per kv head, 64 channels


def _heads(shape):
    return dict(zip(("q_heads", "kv_heads", "qk_dim", "v_dim"), shape))


def _train(shape, seqs, lo, hi, core="fused", cmp_k="mean", cmp_v="sigmoid-mul", host_lens=False, len_seed=1):
    """Forward + backward over `seqs` packed sequences of lo..hi tokens."""
    return dict(kind="train", **_heads(shape), seqs=seqs, lo=lo, hi=hi, core=core, cmp_k=cmp_k, cmp_v=cmp_v,
                host_lens=host_lens, len_seed=len_seed)


def _forward(shape, seqs, lo, hi, core="staged", cmp_k="mean", cmp_v="mean", len_seed=1):
    return dict(_train(shape, seqs, lo, hi, core, cmp_k, cmp_v, False, len_seed), kind="forward")


def _prefill(shape, seqs, prefix_lo, prefix_hi, lo, hi, page=256, store=False, len_seed=2):
    """lo..hi new tokens per request behind a cached prefix; store: the call also writes the new K/V rows."""
    return dict(kind="prefill", **_heads(shape), seqs=seqs, prefix_lo=prefix_lo, prefix_hi=prefix_hi, lo=lo, hi=hi,
                page=page, store=store, len_seed=len_seed)


def _decode(shape, seqs, lo, hi, page=256, store=False, graph=True, len_seed=3):
    """One token for each of `seqs` requests with lo..hi tokens of context; graph: replayed as serving engines do."""
    return dict(kind="decode", **_heads(shape), seqs=seqs, lo=lo, hi=hi, page=page, store=store, graph=graph,
                len_seed=len_seed)


def listed():
    return [
        # the headline: one long document per step, learned V compression
        dict(_train(WIDE, 1, 65536, 65536), name="train_64k"),
        # pre-training on packed documents of medium length; the data loader has the lengths on the host
        dict(_train(WIDE, 8, 4096, 8192, host_lens=True), name="train_packed_8"),
        # the smallest training step of the reference's tables, through the module that runs one autograd node per
        # stage
        dict(_train(NARROW, 1, 4096, 4096, core="staged", cmp_v="mean"), name="train_4k_staged"),
        # fine-tuning a small model on many short, ragged samples, learned compression of K and V
        dict(_train(SMALL, 40, 17, 1200, cmp_k="linear", cmp_v="swiglu", host_lens=True), name="train_short_samples"),
        # scoring / evaluation without gradients, an odd length, 192 q/k channels
        dict(_forward(QK192, 1, 16381, 16381), name="forward_16k_qk192"),
        # serving: a chunk of a chunked prefill of 16 requests, prefixes already in the cache
        dict(_prefill(WIDE, 16, 0, 16384, 2048, 2048), name="prefill_chunks"),
        # serving: a few short prompts, nothing cached, K/V written by the same call
        dict(_prefill(WIDE, 3, 0, 0, 60, 700, store=True), name="prefill_short_prompts"),
        # serving: the benchmark's decode batch
        dict(_decode(WIDE, 64, 4096, 32768), name="decode_64_ragged"),
        # one chat with a long context, called eagerly: latency and launches count
        dict(_decode(WIDE, 1, 32768, 32768, graph=False), name="decode_1_32k_eager"),
        # throughput serving: many short contexts
        dict(_decode(WIDE, 512, 4096, 4096), name="decode_512_4k"),
        # few, very long contexts
        dict(_decode(WIDE, 16, 131072, 131072), name="decode_16_128k"),
        # a small ragged batch with 192 q/k channels, the newest token's K/V written by the same call
        dict(_decode(QK192, 8, 700, 16384, store=True), name="decode_8_qk192"),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng: random.Random):
    kind = rng.choice(("train", "train", "forward", "prefill", "decode", "decode"))
    shape = rng.choice((WIDE, WIDE, NARROW, QK192, SMALL))
    seed = rng.randrange(1, 1 << 16)
    if kind in ("train", "forward"):
        total = _log(rng, 1024, 49152)
        seqs = min(rng.choice((1, 1, _log(rng, 2, 40))), max(1, total // 400))
        hi = max(total // seqs, 17)
        lo = hi if seqs == 1 else rng.randint(17, hi)
        if kind == "forward":
            return _forward(shape, seqs, lo, hi, rng.choice(("staged", "fused")), "mean",
                            rng.choice(("mean", "sigmoid-mul")), seed)
        methods = rng.choice((("mean", "mean"), ("mean", "sigmoid-mul"), ("linear", "swiglu")))
        return _train(shape, seqs, lo, hi, rng.choice(("fused", "fused", "staged")), *methods,
                      host_lens=rng.random() < 0.5, len_seed=seed)
    page = rng.choice((64, 128, 256, 256))
    if kind == "prefill":
        seqs = _log(rng, 1, 16)
        hi = _log(rng, 40, 2048 * 16 // seqs)
        lo = rng.randint(max(1, hi // 8), hi)
        prefix = rng.choice((0, _log(rng, 64, 16384)))
        return _prefill(shape, seqs, prefix // 4, prefix, lo, hi, page, rng.random() < 0.5, seed)
    seqs = _log(rng, 1, 512)
    hi = min(_log(rng, 512, 131072), (2 << 20) // seqs)
    lo = rng.randint(max(1, hi // 8), hi)
    return _decode(shape, seqs, lo, hi, page, rng.random() < 0.4, rng.random() < 0.7, seed)


# ------------------------------------------------------------------------------------------------ sizes of a case
def _lens(case, lo="lo", hi="hi", salt=0):
    """Lengths per sequence: a property of the case, so that its work does not depend on the inputs' seed."""
    r = random.Random(case["len_seed"] * 1000003 + salt)
    return [r.randint(case[lo], case[hi]) for _ in range(case["seqs"])]


def _cmp_len(n):
    return max((n - KERNEL) // STRIDE + 1, 0)


def _branch_pairs(first, last):
    """Visible (query, key) pairs per q-head of the compressed, selected and window branch for tokens first..last-1."""
    t = np.arange(first, last, dtype=np.int64)
    nc = np.maximum((t - (KERNEL - 1)) // STRIDE + 1, 0).sum()
    ns = (BLOCK * np.minimum(TOP_N, t // BLOCK + 1)).sum()
    nw = np.minimum(t + 1, WINDOW + 1).sum()
    return int(nc), int(ns), int(nw)


def work(case):
    QH, KH, D, VD = case["q_heads"], case["kv_heads"], case["qk_dim"], case["v_dim"]
    kv_row = KH * (D + VD) * 2
    if case["kind"] == "decode":
        nbytes = flops = 0
        for n in _lens(case):
            nc, ns, nw = _branch_pairs(n - 1, n)
            ns = min(ns, n)
            nbytes += (_cmp_len(n) + ns + nw) * kv_row + QH * (D + VD + 3) * 2 + (2 * kv_row if case["store"] else 0)
            flops += QH * (2 * (D + VD) * (nc + ns + nw) + 2 * D * nc)
        return dict(bytes=nbytes, flops=flops)
    if case["kind"] == "prefill":
        nbytes = flops = 0
        for new, prefix in zip(_lens(case), _lens(case, "prefix_lo", "prefix_hi", 1)):
            nc, ns, nw = _branch_pairs(prefix, prefix + new)
            rows = min(prefix + new, new * TOP_N * BLOCK + WINDOW)
            nbytes += new * QH * (D + VD + 3) * 2 + (rows + _cmp_len(prefix + new)) * kv_row
            nbytes += new * kv_row if case["store"] else 0
            flops += QH * (2 * (D + VD) * (nc + ns + nw) + 2 * D * nc)
        return dict(bytes=nbytes, flops=flops)
    lens = _lens(case)
    T, Y = sum(lens), sum(_cmp_len(n) for n in lens)
    nc, ns, nw = (sum(p) for p in zip(*(_branch_pairs(0, n) for n in lens)))
    flops = QH * (2 * (D + VD) * (nc + ns + nw) + 2 * D * nc)
    nbytes = T * (QH * (D + VD + 3) * 2 + kv_row)
    for method, dim in ((case["cmp_k"], D), (case["cmp_v"], VD)):
        if method != "mean":  # the projection of the learned compression, once forward and twice backward
            out = dim if method == "linear" else 2 * dim
            gemm = 2 * Y * KH * KERNEL * dim * out
            flops += gemm * (3 if case["kind"] == "train" else 1)
    if case["kind"] == "train":
        flops += QH * 5 * (D + VD) * (nc + ns + nw)
        nbytes += T * (QH * (D + VD + 3) * 2 + kv_row) + T * QH * (D + VD) * 2
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    # bf16 inputs, outputs and matrix operands with fp32 accumulation; a few tokens may take another block where the
    # scores of two blocks tie to within rounding
    return {"rel": 1e-2}


# ------------------------------------------------------------------------------------------------ inputs
def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.bfloat16)


def _prepare_packed(case, g):
    QH, KH, D, VD = case["q_heads"], case["kv_heads"], case["qk_dim"], case["v_dim"]
    cu = np.concatenate([[0], np.cumsum(_lens(case))]).astype(np.int32)
    T = int(cu[-1])
    cfg = NSAConfig(head_dim=VD, qk_head_dim=D, v_head_dim=VD, num_heads=QH, num_kv_heads=KH,
                    cmp_k_method=case["cmp_k"], cmp_v_method=case["cmp_v"])
    core = (NSACore if case["core"] == "fused" else HFNSACore)(cfg).to(device="cuda", dtype=torch.bfloat16)
    for p in core.parameters():
        with torch.no_grad():
            p.normal_(std=p.size(-1) ** -0.5, generator=g)
    leaves = dict(q=_randn(g, T, QH, D), k=_randn(g, T, KH, D), v=_randn(g, T, KH, VD), w=_randn(g, T, QH, 3))
    args = (torch.from_numpy(cu).cuda(),) + ((cu,) if case["core"] == "fused" and case["host_lens"] else ())
    state = dict(kind=case["kind"], core=core, leaves=leaves, args=args)
    if case["kind"] == "train":
        for t in leaves.values():
            t.requires_grad_()
        state["do"] = _randn(g, T, QH, VD)
        state["params"] = dict(core.named_parameters())
    return state


def _pages(case, total, seed):
    """Pools filled with random rows, page tables (pages handed out in random order) and the flat pool row of every
    raw and every compressed row of requests of the given total lengths."""
    KH, D, VD, page = case["kv_heads"], case["qk_dim"], case["v_dim"], case["page"]
    r = np.random.RandomState(seed % (1 << 31))
    ys = [_cmp_len(n) for n in total]
    n_raw, n_cmp = [-(-n // page) for n in total], [max(-(-y // page), 1) for y in ys]
    perm = r.permutation(sum(n_raw) + sum(n_cmp)).astype(np.int32)
    bt, cbt = np.full((len(total), max(n_raw)), -1, np.int32), np.full((len(total), max(n_cmp)), -1, np.int32)
    pos, rows, cmp_rows = 0, [], []
    for b, (n, y) in enumerate(zip(total, ys)):
        bt[b, :n_raw[b]] = perm[pos:pos + n_raw[b]]
        pos += n_raw[b]
        cbt[b, :n_cmp[b]] = perm[pos:pos + n_cmp[b]]
        pos += n_cmp[b]
        i = np.arange(max(n, y))
        rows.append((bt[b, i[:n] // page] * page + i[:n] % page).astype(np.int32))
        cmp_rows.append((cbt[b, i[:y] // page] * page + i[:y] % page).astype(np.int32))
    (k, v), = allocate_kv_pools(len(perm), page, KH, D, VD)
    return k, v, bt, cbt, rows, cmp_rows


def _gpu(x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.int32)).cuda()


def _cu(lens):
    return _gpu(np.concatenate([[0], np.cumsum(lens)]))


def _pool_rows(k, v, bt, upto, cmp_rows):
    """The compressed rows that earlier steps left in the cache: those inside the first upto[b] tokens."""
    ys = [_cmp_len(n) for n in upto]
    if max(ys) > 0:
        slots = _gpu(np.concatenate([c[:y] for c, y in zip(cmp_rows, ys)]))
        for cache in (k, v):
            mean_pooling_prefill(cache, _cu(ys), max(ys), bt, slots)


def _prepare_prefill(case, g, seed):
    QH, KH, D, VD = case["q_heads"], case["kv_heads"], case["qk_dim"], case["v_dim"]
    new, prefix = _lens(case), _lens(case, "prefix_lo", "prefix_hi", 1)
    total = [n + p for n, p in zip(new, prefix)]
    k, v, bt, cbt, rows, cmp_rows = _pages(case, total, seed)
    k.normal_(generator=g)
    v.normal_(generator=g)
    bt, cbt = _gpu(bt), _gpu(cbt)
    _pool_rows(k, v, bt, prefix, cmp_rows)
    ys = [_cmp_len(n) for n in total]
    slots = [np.where(np.arange(y) < _cmp_len(p), -1, c) for y, p, c in zip(ys, prefix, cmp_rows)]
    t = sum(new)
    args = (_randn(g, t, QH, D), k, v, _randn(g, t, QH, 3), _cu(new), _cu(ys), max(new), max(ys), _gpu(total), bt,
            _gpu(np.concatenate(slots)), cbt)
    kw = {}
    if case["store"]:
        kw = dict(new_k=_randn(g, t, KH, D), new_v=_randn(g, t, KH, VD),
                  slot_mapping=_gpu(np.concatenate([r[p:] for r, p in zip(rows, prefix)])))
    return dict(kind="prefill", args=args, kw=kw)


def _prepare_decode(case, g, seed):
    QH, KH, D, VD = case["q_heads"], case["kv_heads"], case["qk_dim"], case["v_dim"]
    lens = _lens(case)
    k, v, bt, cbt, rows, cmp_rows = _pages(case, lens, seed)
    k.normal_(generator=g)
    v.normal_(generator=g)
    bt, cbt = _gpu(bt), _gpu(cbt)
    _pool_rows(k, v, bt, [n - 1 for n in lens], cmp_rows)
    slots = [c[-1] if len(c) > _cmp_len(n - 1) else -1 for n, c in zip(lens, cmp_rows)]
    B = len(lens)
    args = (_randn(g, B, QH, D), k, v, _randn(g, B, QH, 3), _gpu(lens), bt, _gpu(slots), cbt)
    # an engine fixes its capacities once, from the longest context that it admits
    kw = dict(fixed_y_maxlen=max(2048, -(-case["hi"] // STRIDE // 256) * 256),
              fixed_num_slc_blocks=max(512, -(-case["hi"] // BLOCK)))
    if case["store"]:
        kw.update(new_k=_randn(g, B, KH, D), new_v=_randn(g, B, KH, VD), slot_mapping=_gpu([r[-1] for r in rows]))
    state = dict(kind="decode", args=args, kw=kw)
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            nsa_decode(*args, **kw)
        torch.cuda.current_stream().wait_stream(side)
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["o"] = nsa_decode(*args, **kw)
    return state


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] == "prefill":
        return _prepare_prefill(case, g, seed)
    if case["kind"] == "decode":
        return _prepare_decode(case, g, seed)
    return _prepare_packed(case, g)


# ------------------------------------------------------------------------------------------------ one pass
def run(state):
    if state["kind"] == "decode":
        if "graph" in state:
            state["graph"].replay()
            o = state["o"]
        else:
            o = nsa_decode(*state["args"], **state["kw"])
        return dict(o=o, k=state["args"][1], v=state["args"][2])
    if state["kind"] == "prefill":
        o = nsa_prefill(*state["args"], **state["kw"])
        return dict(o=o, k=state["args"][1], v=state["args"][2])
    x = state["leaves"]
    if state["kind"] == "forward":
        with torch.no_grad():
            return state["core"](x["q"], x["k"], x["v"], x["w"], *state["args"])
    grads = dict(x, **state["params"])
    for t in grads.values():
        t.grad = None
    o = state["core"](x["q"], x["k"], x["v"], x["w"], *state["args"])
    o.backward(state["do"])
    return dict({"d" + n: t.grad for n, t in grads.items()}, o=o.detach())
