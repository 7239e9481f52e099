"""GPU parity of the paged-KV prefill and decode entry points against the CPU oracle, and the invariants the
upstream notebook checks (inference.ipynb cells 9/11/16/19/26/34/43/50): pooled rows bit-equal to the contiguous
pooling, decode == last row of the training forward, chunked prefill == one-shot prefill, graph replay == eager."""
import pytest
import torch

from oracle import nsa_oracle as O
from gpu_util import randn_bf16, assert_close, make_cu
from paged_util import build_pool, prepool, prefill_slot_mapping, decode_slot_mapping

pytestmark = pytest.mark.gpu


def to_dev(case, device):
    return {k: (v.to(device) if isinstance(v, torch.Tensor) else v) for k, v in case.items()}


@pytest.mark.parametrize("QH,KH,D", [(16, 1, 128), (8, 2, 128), (64, 2, 64)])
def test_prefill_with_cached_prefix(device, QH, KH, D):
    from flash_nsa import nsa_prefill
    cached = [0, 37, 512, 1000, 130]
    new = [300, 200, 64, 17, 1]
    ctx = [c + n for c, n in zip(cached, new)]
    case = build_pool(ctx, KH, D, D, page=128, seed=3)
    prepool(case, cached)
    slots, ycu = prefill_slot_mapping(case, cached)
    xcu = make_cu(new)
    t = int(xcu[-1])
    q, w = randn_bf16(t, QH, D, seed=5), randn_bf16(t, QH, 3, seed=6)
    top_n = 6
    kw = dict(top_n=top_n, window_size=100)
    d = to_dev(case, device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    o = nsa_prefill(q.to(device), d["k"], d["v"], w.to(device), xcu.to(device), ycu.to(device), max(new),
                    max(case["ys"]), ctx_t.to(device), d["bt"], slots.to(device), d["cbt"], fixed_y_maxlen=256,
                    fixed_num_slc_blocks=32, **kw)
    # pooled rows: identical to pooling on the host (fp32 mean, same summation order, rounded to bf16)
    ref_case = {k: (v.clone() if isinstance(v, torch.Tensor) else v) for k, v in case.items()}
    O.paged_pool_prefill(ref_case["k"], ycu, ctx_t, case["bt"], slots)
    O.paged_pool_prefill(ref_case["v"], ycu, ctx_t, case["bt"], slots)
    assert_close(d["k"], ref_case["k"], "pooled K rows", atol=0, rtol=8e-3)
    assert_close(d["v"], ref_case["v"], "pooled V rows", atol=0, rtol=8e-3)
    # oracle on the device's pool (compressed rows as the device wrote them) and the device's indices
    from flash_nsa.inference import cmp_attn_prefill, topk_prefill
    _, lse = cmp_attn_prefill(q.to(device), d["k"], d["v"], xcu.to(device), max(new), d["cbt"], ctx_t.to(device))
    topk = topk_prefill(q.to(device), d["k"], lse, xcu.to(device), max(new), max(case["ys"]), d["cbt"],
                        ctx_t.to(device), 256, 32, top_n=top_n)
    cfg = O.OracleConfig(**kw)
    kc, vc = d["k"].float().cpu(), d["v"].float().cpu()
    ro, parts = O.nsa_paged_forward(q.float(), kc, vc, w.float(), xcu, ctx_t, case["bt"], case["cbt"], cfg,
                                    topk=topk.cpu(), round_dtype=torch.bfloat16, return_parts=True)
    assert_close(o, ro, "prefill o")
    # selection parity (oracle's own selection vs device's), ties excused within 1e-3
    own = torch.cat([p["topk"] for p in parts], 1)  # these are the device's (fed in); recompute the oracle's own
    ro2, parts2 = O.nsa_paged_forward(q.float(), kc, vc, w.float(), xcu, ctx_t, case["bt"], case["cbt"], cfg,
                                      return_parts=True)
    rt = torch.cat([p["topk"] for p in parts2], 1)
    n_rows, n_diff, n_bad = O.topk_mismatch_report(topk.cpu(), rt, [p["imp"] for p in parts2], xcu, 64, top_n,
                                                   tie_tol=1e-3, t_offsets=cached)
    assert n_bad == 0 and n_diff <= max(1, n_rows // 200), (n_rows, n_diff, n_bad)


def test_chunked_prefill_equals_one_shot(device):
    from flash_nsa import nsa_prefill
    QH, KH, D = 16, 1, 128
    ctx = [5000, 777]
    kw = dict(top_n=6, window_size=100, fixed_y_maxlen=512, fixed_num_slc_blocks=128)
    q_all = [randn_bf16(L, QH, D, seed=10 + i) for i, L in enumerate(ctx)]
    w_all = [randn_bf16(L, QH, 3, seed=20 + i) for i, L in enumerate(ctx)]

    def run(chunks):
        case = build_pool(ctx, KH, D, D, page=128, seed=4)
        d = to_dev(case, device)
        outs = [[] for _ in ctx]
        done = [0, 0]
        for step in range(chunks):
            new = [(L * (step + 1)) // chunks - (L * step) // chunks for L in ctx]
            cur = [dn + n for dn, n in zip(done, new)]
            sub = dict(case)
            sub["ctx"] = cur
            sub["ys"] = [max((L - 32) // 16 + 1, 0) for L in cur]
            slots, ycu = prefill_slot_mapping(sub, done)
            xcu = make_cu(new)
            q = torch.cat([q_all[b][done[b]:cur[b]] for b in range(len(ctx))])
            w = torch.cat([w_all[b][done[b]:cur[b]] for b in range(len(ctx))])
            o = nsa_prefill(q.to(device), d["k"], d["v"], w.to(device), xcu.to(device), ycu.to(device), max(new),
                            max(sub["ys"]), torch.tensor(cur, dtype=torch.int32, device=device), d["bt"],
                            slots.to(device), d["cbt"], **kw)
            for b in range(len(ctx)):
                outs[b].append(o[int(xcu[b]):int(xcu[b + 1])].cpu())
            done = cur
        return [torch.cat(x) for x in outs], d

    one, d1 = run(1)
    four, d4 = run(4)
    for b in range(len(ctx)):
        assert torch.equal(one[b], four[b]), f"request {b}: chunked prefill differs from one-shot"
    assert torch.equal(d1["k"], d4["k"]) and torch.equal(d1["v"], d4["v"]), "pooled cache rows differ"
    # the paged block selector working segment by segment (as it does for contexts whose score rows do not fit LDS)
    from flash_nsa import _lib
    _lib.call("nsa_set_tuning", b"topk_seg_blocks", 32)
    try:
        seg, _ = run(4)
    finally:
        _lib.call("nsa_reset_tuning")
    for b in range(len(ctx)):
        assert torch.equal(one[b], seg[b]), f"request {b}: segmented block selection changed the prefill"


@pytest.mark.parametrize("hp", [
    dict(kernel_size=32, stride=16, block_size=64, top_n=16, window_size=512),
    dict(kernel_size=64, stride=32, block_size=128, top_n=4, window_size=256),
    dict(kernel_size=32, stride=8, block_size=64, top_n=16, window_size=512),
    dict(kernel_size=16, stride=16, block_size=64, top_n=3, window_size=1, num_init_blocks=0, num_local_blocks=1),
    dict(kernel_size=32, stride=16, block_size=32, top_n=12, window_size=64),
    dict(kernel_size=64, stride=16, block_size=256, top_n=3, window_size=128),
    dict(kernel_size=32, stride=16, block_size=96, top_n=5, window_size=64),
])
def test_prefill_with_cached_prefix_equals_training_rows(device, hp):
    """Prefill of new tokens behind a cached prefix, default and other compression / block / top-n / window settings:
    the output rows are bit-equal to the same rows of the training forward on the gathered sequence."""
    _prefill_equals_training_rows(device, 16, 2, 128, 128, [0, 37, 512, 1000, 130, 64], [300, 200, 64, 17, 1, 700], hp)


@pytest.mark.parametrize("QH,KH,D,page", [(16, 2, 128, 64), (16, 2, 128, 512), (6, 2, 128, 128), (5, 1, 128, 128),
                                          (7, 7, 128, 128), (64, 2, 128, 128), (8, 2, 64, 256)])
def test_prefill_head_groups_and_page_sizes_equal_training_rows(device, QH, KH, D, page):
    """The same for pages of 64 / 256 / 512 rows (prefixes and chunks on and around page boundaries) and for groups of
    1, 3, 5 and 32 q-heads per kv head."""
    _prefill_equals_training_rows(device, QH, KH, D, page, [0, 37, 512, 1000, 130, 64, page, page - 1, 3 * page + 5],
                                  [300, 200, 64, 17, 1, 700, page, page + 1, 2 * page], {})


def _prefill_equals_training_rows(device, QH, KH, D, page, cached, new, hp):
    from flash_nsa import nsa_prefill, NSAConfig, NSACore, NSAHelper
    ctx = [c + n for c, n in zip(cached, new)]
    ks, st = hp.get("kernel_size", 32), hp.get("stride", 16)
    case = build_pool(ctx, KH, D, D, page=page, seed=3, kernel=ks, stride=st)
    prepool(case, cached, kernel=ks, stride=st)
    slots, ycu = prefill_slot_mapping(case, cached, kernel=ks, stride=st)
    xcu = make_cu(new)
    d = to_dev(case, device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    qs = [randn_bf16(L, QH, D, seed=100 + b) for b, L in enumerate(ctx)]
    ws = [randn_bf16(L, QH, 3, seed=200 + b) for b, L in enumerate(ctx)]
    q = torch.cat([qs[b][cached[b]:] for b in range(len(ctx))])
    w = torch.cat([ws[b][cached[b]:] for b in range(len(ctx))])
    try:
        o = nsa_prefill(q.to(device), d["k"], d["v"], w.to(device), xcu.to(device), ycu.to(device), max(new),
                        max(case["ys"]), ctx_t.to(device), d["bt"], slots.to(device), d["cbt"], fixed_y_maxlen=512,
                        fixed_num_slc_blocks=128, **hp)
        core = NSACore(NSAConfig(head_dim=D, num_heads=QH, num_kv_heads=KH, **hp))
        for b, L in enumerate(ctx):
            ks_ = O.gather_rows(case["k"], case["bt"][b], L).to(device)
            vs_ = O.gather_rows(case["v"], case["bt"][b], L).to(device)
            with torch.no_grad():
                full = core(qs[b].to(device), ks_, vs_, ws[b].to(device),
                            torch.tensor([0, L], dtype=torch.int32, device=device))
            a, e = int(xcu[b]), int(xcu[b + 1])
            assert torch.equal(o[a:e], full[cached[b]:]), f"request {b} (cached {cached[b]}, new {new[b]})"
    finally:
        NSAHelper.set_hyperparameters()


@pytest.mark.parametrize("store", [False, True])
def test_prefill_chunk_that_completes_no_compressed_row(device, store):
    """A chunk that ends before its next compressed row: no row has a destination, so the pooling may be told of none
    (y_maxlen 0) as well as of all of them with slots of -1.  y_maxlen says nothing about the length of the context."""
    from flash_nsa import nsa_prefill
    QH, KH, D, page = 16, 1, 128, 64
    cached, new = [1600, 3200], [13, 9]
    ctx = [c + n for c, n in zip(cached, new)]
    case = build_pool(ctx, KH, D, D, page=page, seed=5)
    prepool(case, ctx)
    assert case["ys"] == [max((c - 32) // 16 + 1, 0) for c in cached]
    slots, ycu = prefill_slot_mapping(case, ctx)
    assert int(slots.max()) == -1
    xcu = make_cu(new).to(device)
    d = to_dev(case, device)
    t = sum(new)
    q, w = randn_bf16(t, QH, D, seed=6).to(device), randn_bf16(t, QH, 3, seed=7).to(device)
    kw = dict(fixed_y_maxlen=512, fixed_num_slc_blocks=128)
    if store:
        at = torch.cat([torch.tensor([int(case["bt"][b, i // page]) * page + i % page for i in range(c, c + n)])
                        for b, (c, n) in enumerate(zip(cached, new))])
        kw.update(new_k=case["k"].view(-1, KH, D)[at].to(device), new_v=case["v"].view(-1, KH, D)[at].to(device),
                  slot_mapping=at.to(torch.int32).to(device))

    def run(ycu, y_maxlen):
        poison = [torch.full((t, QH, D), float("nan"), device=device, dtype=torch.bfloat16) for _ in range(4)]
        del poison  # rows that no kernel writes are not finite
        return nsa_prefill(q, d["k"], d["v"], w, xcu, ycu.to(device), max(new), y_maxlen,
                           torch.tensor(ctx, dtype=torch.int32, device=device), d["bt"], slots.to(device), d["cbt"], **kw)

    none = run(torch.zeros_like(ycu), 0)
    assert torch.isfinite(none).all()
    assert torch.equal(none, run(ycu, max(case["ys"])))


@pytest.mark.parametrize("hp", [
    dict(kernel_size=64, stride=32, block_size=128, top_n=4, window_size=256),
    dict(kernel_size=64, stride=16, block_size=64, top_n=5, window_size=100),
    dict(kernel_size=32, stride=8, block_size=64, top_n=16, window_size=512),
    dict(kernel_size=16, stride=16, block_size=64, top_n=3, window_size=1, num_init_blocks=0, num_local_blocks=1),
    dict(kernel_size=32, stride=16, block_size=32, top_n=12, window_size=64),
    dict(kernel_size=64, stride=16, block_size=256, top_n=3, window_size=128),
    dict(kernel_size=32, stride=16, block_size=96, top_n=5, window_size=64),
])
def test_decode_other_hyperparameters_equals_training_row(device, hp):
    """Decode with compression, block, top-n, forced-block and window settings other than the defaults: every
    request's output is the last row of the training forward on its gathered sequence, and the one-launch path agrees
    with the stage-by-stage one."""
    from flash_nsa import nsa_decode, NSAConfig, NSACore, NSAHelper
    from flash_nsa.inference import nsa_decode_staged
    QH, KH, D = 16, 2, 128
    ctx = [1024, 333, 130, 64, 65, 1, 777, 2000, 640]
    ks, st = hp["kernel_size"], hp["stride"]
    case = build_pool(ctx, KH, D, D, page=128, seed=7, kernel=ks, stride=st)
    prepool(case, [L - 1 for L in ctx], kernel=ks, stride=st)
    slots = decode_slot_mapping(case, kernel=ks, stride=st)
    B = len(ctx)
    q, w = randn_bf16(B, QH, D, seed=8), randn_bf16(B, QH, 3, seed=9)
    d = to_dev(case, device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32).to(device)
    nb_cap = max(32, -(-max(ctx) // hp["block_size"]))  # capacity: at least the blocks of the longest context
    try:
        o = nsa_decode(q.to(device), d["k"], d["v"], w.to(device), ctx_t, d["bt"], slots.to(device), d["cbt"],
                       fixed_y_maxlen=256, fixed_num_slc_blocks=nb_cap, **hp)
        o2 = nsa_decode_staged(q.to(device), d["k"], d["v"], w.to(device), ctx_t, d["bt"], d["cbt"],
                               fixed_y_maxlen=256, fixed_num_slc_blocks=nb_cap, **hp)
        assert_close(o, o2, "one-launch vs stage-by-stage decode", atol=1e-2, rtol=1e-2)
        core = NSACore(NSAConfig(head_dim=D, num_heads=QH, num_kv_heads=KH, **hp))
        for b in range(B):
            L = ctx[b]
            ks_ = O.gather_rows(case["k"], case["bt"][b], L).to(device)
            vs_ = O.gather_rows(case["v"], case["bt"][b], L).to(device)
            qs = randn_bf16(L, QH, D, seed=100 + b)
            qs[-1] = q[b]
            ws = randn_bf16(L, QH, 3, seed=200 + b)
            ws[-1] = w[b]
            with torch.no_grad():
                full = core(qs.to(device), ks_, vs_, ws.to(device),
                            torch.tensor([0, L], dtype=torch.int32, device=device))
            assert_close(o[b], full[-1], f"decode vs training row (request {b})", atol=1e-2, rtol=1e-2)
    finally:
        NSAHelper.set_hyperparameters()


@pytest.mark.parametrize("QH,KH,page", [(6, 2, 128), (5, 1, 128), (24, 2, 128), (7, 7, 128), (16, 2, 64), (16, 2, 512)])
def test_decode_head_groups_and_page_sizes_equal_training_row(device, QH, KH, page):
    """Groups of 3, 5, 12 and 1 q-heads per kv head and pages of 64 / 512 rows, contexts on and around page and
    block boundaries plus a padded request: every output is the last row of the training forward on the gathered
    sequence (padded rows are zero).  The stage-by-stage decode (fp32 block scores) must agree everywhere; the
    one-launch kernel keeps its probabilities as fp16 between its phases, so a kv head whose block scores tie within
    2e-4 at the selection cut (the parity bar excuses 1e-3) may pick the other block and is left out of its
    comparison."""
    from flash_nsa import nsa_decode, NSAConfig, NSACore, NSAHelper
    from flash_nsa.inference import nsa_decode_staged
    from flash_nsa.ops.compress_kv import mean_pooling_fwd
    from flash_nsa.ops.compress_attn import cmp_attn_fwd
    from flash_nsa.ops.topk import slc_topk_indices
    D, G = 128, QH // KH
    ctx = [1024, 333, 130, 64, 65, 1, 777, 2000, 640, 0, 4097, page, page + 1, page - 1, 2 * page]
    case = build_pool(ctx, KH, D, D, page=page, seed=7)
    prepool(case, [max(L - 1, 0) for L in ctx])
    slots = decode_slot_mapping(case)
    B = len(ctx)
    q, w = randn_bf16(B, QH, D, seed=8), randn_bf16(B, QH, 3, seed=9)
    d = to_dev(case, device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32).to(device)
    kw = dict(fixed_y_maxlen=512, fixed_num_slc_blocks=128)
    o = nsa_decode(q.to(device), d["k"], d["v"], w.to(device), ctx_t, d["bt"], slots.to(device), d["cbt"], **kw)
    staged = nsa_decode_staged(q.to(device), d["k"], d["v"], w.to(device), ctx_t, d["bt"], d["cbt"], **kw)
    core = NSACore(NSAConfig(head_dim=D, num_heads=QH, num_kv_heads=KH))
    n_ties = 0
    for b, L in enumerate(ctx):
        if L == 0:
            assert float(o[b].float().abs().max()) == 0.0 and float(staged[b].float().abs().max()) == 0.0
            continue
        ks = O.gather_rows(case["k"], case["bt"][b], L).to(device)
        vs = O.gather_rows(case["v"], case["bt"][b], L).to(device)
        qs = randn_bf16(L, QH, D, seed=100 + b)
        qs[-1] = q[b]
        ws = randn_bf16(L, QH, 3, seed=200 + b)
        ws[-1] = w[b]
        cu1 = torch.tensor([0, L], dtype=torch.int32, device=device)
        with torch.no_grad():
            full = core(qs.to(device), ks, vs, ws.to(device), cu1)
            _, lse = cmp_attn_fwd(qs.to(device), mean_pooling_fwd(ks), mean_pooling_fwd(vs))
            _, scores = slc_topk_indices(qs.to(device), mean_pooling_fwd(ks), lse, return_slc_prob=True)
        assert_close(staged[b], full[-1], f"stage-by-stage decode vs training row (request {b}, context {L})",
                     atol=1e-2, rtol=1e-2)
        nb = (L - 1) // 64 + 1
        keep = torch.ones(QH, dtype=torch.bool)
        for kh in range(KH):
            free = scores[kh, -1, 1:max(nb - 2, 1)].float().sort(descending=True).values  # not forced: 1 .. nb-3
            if free.numel() > 13 and float(free[12] - free[13]) < 2e-4:
                keep[kh * G:(kh + 1) * G] = False
                n_ties += 1
        if keep.any():
            assert_close(o[b][keep.to(device)], full[-1][keep.to(device)],
                         f"one-launch decode vs training row (request {b}, context {L})", atol=1e-2, rtol=1e-2)
    NSAHelper.set_hyperparameters()
    assert n_ties <= 2 * KH, f"{n_ties} (request, kv head) pairs excused as ties"


@pytest.mark.parametrize("QH,KH,D", [(16, 1, 128), (64, 4, 128)])
def test_decode_vs_oracle_and_training_forward(device, QH, KH, D):
    from flash_nsa import nsa_decode, NSAConfig, NSACore
    ctx = [1024, 333, 48, 31, 1, 777, 2000, 640]
    case = build_pool(ctx, KH, D, D, page=128, seed=7)
    prepool(case, [L - 1 for L in ctx])           # everything that was complete before the newest token
    slots = decode_slot_mapping(case)
    B = len(ctx)
    q, w = randn_bf16(B, QH, D, seed=8), randn_bf16(B, QH, 3, seed=9)
    kw = dict(top_n=6, window_size=100)
    d = to_dev(case, device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    o = nsa_decode(q.to(device), d["k"], d["v"], w.to(device), ctx_t.to(device), d["bt"], slots.to(device), d["cbt"],
                   fixed_y_maxlen=256, fixed_num_slc_blocks=32, **kw)
    ref_case = {k: (v.clone() if isinstance(v, torch.Tensor) else v) for k, v in case.items()}
    O.paged_pool_decode(ref_case["k"], ctx_t, case["bt"], slots)
    O.paged_pool_decode(ref_case["v"], ctx_t, case["bt"], slots)
    assert_close(d["k"], ref_case["k"], "decode pooled K", atol=0, rtol=8e-3)
    from flash_nsa.inference import cmp_attn_decode, topk_decode
    _, lse = cmp_attn_decode(q.to(device), d["k"], d["v"], d["cbt"], ctx_t.to(device))
    topk = topk_decode(q.to(device), d["k"], lse, d["cbt"], ctx_t.to(device), 256, 32, top_n=6)
    xcu = torch.arange(B + 1, dtype=torch.int32)
    cfg = O.OracleConfig(**kw)
    kc, vc = d["k"].float().cpu(), d["v"].float().cpu()
    ro = O.nsa_paged_forward(q.float(), kc, vc, w.float(), xcu, ctx_t, case["bt"], case["cbt"], cfg, topk=topk.cpu(),
                             round_dtype=torch.bfloat16)
    assert_close(o, ro, "decode o")
    # decode == last row of the training forward on the same (contiguous) sequence
    cfgm = NSAConfig(head_dim=D, num_heads=QH, num_kv_heads=KH, **kw)
    core = NSACore(cfgm)
    for b in (0, 5):
        L = ctx[b]
        ks = O.gather_rows(case["k"], case["bt"][b], L).to(device)
        vs = O.gather_rows(case["v"], case["bt"][b], L).to(device)
        qs = randn_bf16(L, QH, D, seed=100 + b)
        qs[-1] = q[b]
        ws = randn_bf16(L, QH, 3, seed=200 + b)
        ws[-1] = w[b]
        with torch.no_grad():
            full = core(qs.to(device), ks, vs, ws.to(device), torch.tensor([0, L], dtype=torch.int32, device=device))
        assert_close(o[b], full[-1], f"decode vs training row (request {b})", atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("page,hp", [
    (128, dict(block_size=64, top_n=16)),
    (256, dict(block_size=64, top_n=16)),
    (128, dict(block_size=32, top_n=12)),
    (256, dict(block_size=96, top_n=5)),
])
def test_decode_selectors_return_the_oracle_selection(device, page, hp):
    """Every decode selector (the staged topk_decode, the one-launch kernel, the split path) against the oracle's own
    selection from the oracle's own scores on the same pool: index sets identical, differences excused only between
    blocks whose scores lie within 1e-3 of each other (none of the outputs feeds the oracle here)."""
    from flash_nsa.inference import (cmp_attn_decode, topk_decode, decode_one_launch, decode_split,
                                     decode_one_launch_fits, decode_split_fits)
    QH, KH, D = 64, 4, 128
    ctx = [1, 31, 32, 64, 65, 4097, 333, 2999, 640, 1024, 127, 129, 4096, 1777]
    case = build_pool(ctx, KH, D, D, page=page, seed=91)
    prepool(case, ctx)                               # every compressed row pooled on the CPU: one pool for both sides
    B = len(ctx)
    d = to_dev(case, device)
    q, w = randn_bf16(B, QH, D, seed=92), randn_bf16(B, QH, 3, seed=93)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    Bs, top_n = hp["block_size"], hp["top_n"]
    y_cap, nb_cap = 512, (4608 // Bs)
    kw = dict(fixed_y_maxlen=y_cap, fixed_num_slc_blocks=nb_cap, block_size=Bs, top_n=top_n)
    cfg = O.OracleConfig(block_size=Bs, top_n=top_n)
    xcu = torch.arange(B + 1, dtype=torch.int32)
    _, parts = O.nsa_paged_forward(q.float(), case["k"].float(), case["v"].float(), w.float(), xcu, ctx_t, case["bt"],
                                   case["cbt"], cfg, return_parts=True)
    own = torch.cat([p["topk"] for p in parts], 1)
    imps = [p["imp"] for p in parts]
    qd, wd, cd = q.to(device), w.to(device), ctx_t.to(device)
    got = {}
    _, lse = cmp_attn_decode(qd, d["k"], d["v"], d["cbt"], cd)
    got["topk_decode"] = topk_decode(qd, d["k"], lse, d["cbt"], cd, **kw)
    assert decode_one_launch_fits(qd, d["k"], d["v"], d["bt"], y_cap, nb_cap)
    got["decode_one_launch"] = decode_one_launch(qd, d["k"], d["v"], wd, d["bt"], d["cbt"], cd, return_parts=True,
                                                 **kw)[4]
    assert decode_split_fits(qd, d["k"], d["v"], d["bt"], y_cap, nb_cap)
    for nsplit in (2, 8):
        got[f"decode_split[{nsplit}]"] = decode_split(qd, d["k"], d["v"], wd, d["bt"], d["cbt"], cd, nsplit=nsplit,
                                                      return_parts=True, **kw)[4]
    for name, tk in got.items():
        tk = tk.cpu()
        assert tk.shape == own.shape and tk.dtype == torch.int32, name
        n_rows, n_diff, n_bad = O.topk_mismatch_report(tk, own, imps, xcu, Bs, top_n, tie_tol=1e-3,
                                                       t_offsets=[L - 1 for L in ctx])
        assert n_rows == B * KH and n_bad == 0 and n_diff <= 1, (name, n_rows, n_diff, n_bad)
        # unused slots carry the inference ignore value, used ones are distinct
        for b, L in enumerate(ctx):
            nv = min(top_n, (L - 1) // Bs + 1)
            for kh in range(KH):
                row = tk[kh, b].tolist()
                assert len(set(row[:nv])) == nv and all(x == -1 for x in row[nv:]), (name, b, kh, row)


def test_decode_graph_replay_equals_eager(device):
    from flash_nsa import nsa_decode
    QH, KH, D = 64, 4, 128
    ctx = [512, 1000, 0, 333]                     # a zero-length row: graph padding
    case = build_pool([max(c, 1) for c in ctx], KH, D, D, page=128, seed=11)
    case["ctx"] = ctx
    case["ys"] = [max((L - 32) // 16 + 1, 0) for L in ctx]
    prepool(case, [max(L - 1, 0) for L in ctx])
    slots = decode_slot_mapping(case)
    B = len(ctx)
    d = to_dev(case, device)
    q = randn_bf16(B, QH, D, seed=12).to(device)
    w = randn_bf16(B, QH, 3, seed=13).to(device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=device)
    sl = slots.to(device)
    args = (q, d["k"], d["v"], w, ctx_t, d["bt"], sl, d["cbt"])
    kw = dict(fixed_y_maxlen=256, fixed_num_slc_blocks=32)
    eager = nsa_decode(*args, **kw).clone()
    assert torch.isfinite(eager).all() and (eager[2] == 0).all()
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        nsa_decode(*args, **kw)
    torch.cuda.current_stream().wait_stream(side)
    with torch.cuda.graph(graph):
        out = nsa_decode(*args, **kw)
    for it in range(4):
        out.zero_()
        junk = torch.randn(1 << 20, device=device).sum()  # the program's own eager work between replays
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {it} differs from eager"
    # new inputs through the same static buffers
    q.copy_(randn_bf16(B, QH, D, seed=14).to(device))
    eager2 = nsa_decode(*args, **kw).clone()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, eager2)


@pytest.mark.parametrize("QH,KH,D", [(64, 4, 128), (16, 1, 128), (12, 2, 64)])
def test_fused_decode_matches_staged_decode(device, QH, KH, D):
    """The two-launch fused decode against the stage-by-stage path (a second, independent set of kernels):
    same block selection, branch outputs and final output."""
    from flash_nsa.inference import (nsa_decode_staged, decode_cmp_topk, decode_slc_swa_combine, cmp_attn_decode,
                                     topk_decode, fused_slc_swa_attn_decode)
    ctx = [4096, 333, 48, 31, 1, 777, 2999, 640, 1024, 65]
    case = build_pool(ctx, KH, D, D, page=128, seed=21)
    prepool(case, ctx)
    B = len(ctx)
    d = to_dev(case, device)
    q = randn_bf16(B, QH, D, seed=22).to(device)
    w = randn_bf16(B, QH, 3, seed=23).to(device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=device)
    kw = dict(top_n=8, window_size=200)
    cmp_o, topk, lse = decode_cmp_topk(q, d["k"], d["v"], d["cbt"], ctx_t, 512, 64, top_n=8, return_lse=True)
    out, slc_o, swa_o = decode_slc_swa_combine(q, d["k"], d["v"], w, topk, cmp_o, d["bt"], ctx_t, return_branches=True,
                                               **kw)
    r_cmp, r_lse = cmp_attn_decode(q, d["k"], d["v"], d["cbt"], ctx_t)
    r_topk = topk_decode(q, d["k"], r_lse, d["cbt"], ctx_t, 512, 64, top_n=8)
    r_slc, r_swa = fused_slc_swa_attn_decode(q, d["k"], d["v"], topk, d["bt"], ctx_t, **kw)
    assert_close(cmp_o, r_cmp, "cmp_o", atol=4e-3, rtol=1e-2)
    assert_close(lse, r_lse, "cmp lse", atol=1e-3, rtol=1e-4)
    nv = torch.clamp((ctx_t - 1) // 64 + 1, max=8).cpu()
    a, r = topk.cpu(), r_topk.cpu()
    for b in range(B):
        for kh in range(KH):
            assert sorted(a[kh, b, :nv[b]].tolist()) == sorted(r[kh, b, :nv[b]].tolist()), (b, kh)
    assert_close(slc_o, r_slc, "slc_o", atol=4e-3, rtol=1e-2)
    assert_close(swa_o, r_swa, "swa_o", atol=4e-3, rtol=1e-2)
    ref = nsa_decode_staged(q, d["k"], d["v"], w, ctx_t, d["bt"], d["cbt"], fixed_y_maxlen=512,
                            fixed_num_slc_blocks=64, **kw)
    assert_close(out, ref, "decode o", atol=8e-3, rtol=1e-2)
    # split compressed branch + in-kernel selection (the path nsa_decode takes)
    from flash_nsa.inference import decode_cmp_split
    for nsplit in (1, 3, 4):
        cmp2, pg, lse2 = decode_cmp_split(q, d["k"], d["v"], d["cbt"], ctx_t, nsplit=nsplit, fixed_y_maxlen=512,
                                          return_lse=True)
        assert_close(cmp2, r_cmp, f"split{nsplit} cmp_o", atol=4e-3, rtol=1e-2)
        assert_close(lse2, r_lse, f"split{nsplit} lse", atol=1e-3, rtol=1e-4)
        out2, topk2 = decode_slc_swa_combine(q, d["k"], d["v"], w, None, cmp2, d["bt"], ctx_t, pg=pg,
                                             fixed_num_slc_blocks=64, **kw)
        t2 = topk2.cpu()
        for b in range(B):
            for kh in range(KH):
                assert sorted(t2[kh, b, :nv[b]].tolist()) == sorted(r[kh, b, :nv[b]].tolist()), (nsplit, b, kh)
        assert_close(out2, ref, f"split{nsplit} decode o", atol=8e-3, rtol=1e-2)


@pytest.mark.parametrize("QH,KH,D", [(64, 4, 128), (16, 1, 128), (12, 2, 64)])
def test_one_launch_decode_matches_two_launch_and_staged(device, QH, KH, D):
    """The one-launch decode kernel (what nsa_decode runs when its tables fit in LDS) against the two-launch path
    and the stage-by-stage kernels: branch outputs, lse, selection and the final output."""
    from flash_nsa.inference import (nsa_decode_staged, decode_cmp_topk, decode_slc_swa_combine, decode_one_launch,
                                     decode_one_launch_fits)
    ctx = [4096, 333, 48, 31, 1, 777, 2999, 640, 1024, 65, 0, 513, 514]
    case = build_pool([max(c, 1) for c in ctx], KH, D, D, page=128, seed=31)
    prepool(case, [max(c, 1) for c in ctx])
    B = len(ctx)
    d = to_dev(case, device)
    q = randn_bf16(B, QH, D, seed=32).to(device)
    w = randn_bf16(B, QH, 3, seed=33).to(device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=device)
    assert decode_one_launch_fits(q, d["k"], d["v"], d["bt"], 512, 64)
    assert not decode_one_launch_fits(q, d["k"], d["v"], d["bt"], 8192, 2048)
    kw = dict(top_n=8, window_size=200)
    out, cmp_o, slc_o, swa_o, topk, lse = decode_one_launch(q, d["k"], d["v"], w, d["bt"], d["cbt"], ctx_t, 512, 64,
                                                            return_parts=True, **kw)
    r_cmp, r_topk, r_lse = decode_cmp_topk(q, d["k"], d["v"], d["cbt"], ctx_t, 512, 64, top_n=8, return_lse=True)
    r_out, r_slc, r_swa = decode_slc_swa_combine(q, d["k"], d["v"], w, r_topk, r_cmp, d["bt"], ctx_t,
                                                 return_branches=True, **kw)
    live = ctx_t > 0
    assert torch.equal(cmp_o[live], r_cmp[live]) and torch.equal(lse[live], r_lse[live])
    assert torch.equal(topk[:, live], r_topk[:, live])
    assert_close(slc_o[live], r_slc[live], "slc_o", atol=4e-3, rtol=1e-2)
    assert_close(swa_o[live], r_swa[live], "swa_o", atol=4e-3, rtol=1e-2)
    assert_close(out[live], r_out[live], "o", atol=8e-3, rtol=1e-2)
    assert float(out[~live].abs().max()) == 0.0, "a padded request (context 0) must give zeros"
    ref = nsa_decode_staged(q[live], d["k"], d["v"], w[live], ctx_t[live], d["bt"][live], d["cbt"][live],
                            fixed_y_maxlen=512, fixed_num_slc_blocks=64, **kw)
    assert_close(out[live], ref, "o vs staged", atol=8e-3, rtol=1e-2)
    out2 = decode_one_launch(q, d["k"], d["v"], w, d["bt"], d["cbt"], ctx_t, 512, 64, **kw)
    assert torch.equal(out, out2), "optional outputs must not change the result"


@pytest.mark.parametrize("QH,KH,D", [(64, 4, 128), (16, 1, 128), (12, 2, 64)])
@pytest.mark.parametrize("nsplit", [1, 3, 4])
def test_split_decode_matches_one_launch(device, QH, KH, D, nsplit):
    """The two-launch decode for small batches of long contexts (compressed branch in `nsplit` parts with spilled
    fp16 probabilities, then merge + selection + selected/window attention + combine) against the one-launch kernel:
    same lse and selection (both fold the same fp16 probabilities), branch outputs and output to bf16 rounding."""
    from flash_nsa.inference import decode_one_launch, decode_split, decode_split_fits
    ctx = [4096, 333, 48, 31, 1, 777, 2999, 640, 1024, 65, 0, 513, 514]
    case = build_pool([max(c, 1) for c in ctx], KH, D, D, page=128, seed=51)
    prepool(case, [max(c, 1) for c in ctx])
    B = len(ctx)
    d = to_dev(case, device)
    q = randn_bf16(B, QH, D, seed=52).to(device)
    w = randn_bf16(B, QH, 3, seed=53).to(device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=device)
    assert decode_split_fits(q, d["k"], d["v"], d["bt"], 512, 64)
    assert not decode_split_fits(q, d["k"], d["v"], d["bt"], 32768, 8192)
    kw = dict(top_n=8, window_size=200)
    r_out, r_cmp, r_slc, r_swa, r_topk, r_lse = decode_one_launch(q, d["k"], d["v"], w, d["bt"], d["cbt"], ctx_t, 512,
                                                                  64, return_parts=True, **kw)
    out, cmp_o, slc_o, swa_o, topk, lse = decode_split(q, d["k"], d["v"], w, d["bt"], d["cbt"], ctx_t, nsplit=nsplit,
                                                       fixed_y_maxlen=512, fixed_num_slc_blocks=64,
                                                       return_parts=True, **kw)
    live = ctx_t > 0
    assert_close(lse[live], r_lse[live], "lse", atol=1e-4, rtol=1e-5)
    assert_close(cmp_o[live], r_cmp[live], "cmp_o", atol=4e-3, rtol=1e-2)
    # the parts change the order of the fp32 sums behind the scores: selections may differ only at score ties
    nv = torch.clamp((ctx_t - 1) // 64 + 1, max=8).cpu()
    a, r = topk.cpu(), r_topk.cpu()
    same = [(b, kh) for b in range(B) if ctx[b] > 0 for kh in range(KH)
            if sorted(a[kh, b, :nv[b]].tolist()) == sorted(r[kh, b, :nv[b]].tolist())]
    n_pairs = sum(1 for c in ctx if c > 0) * KH
    assert len(same) >= n_pairs - max(1, n_pairs // 50), f"{n_pairs - len(same)} of {n_pairs} selections differ"
    G = QH // KH
    for b, kh in same:
        hs = slice(kh * G, (kh + 1) * G)
        assert_close(slc_o[b, hs], r_slc[b, hs], "slc_o", atol=4e-3, rtol=1e-2)
        assert_close(swa_o[b, hs], r_swa[b, hs], "swa_o", atol=4e-3, rtol=1e-2)
        assert_close(out[b, hs], r_out[b, hs], "o", atol=8e-3, rtol=1e-2)
    assert float(out[~live].abs().max()) == 0.0, "a padded request (context 0) must give zeros"
    out2 = decode_split(q, d["k"], d["v"], w, d["bt"], d["cbt"], ctx_t, nsplit=nsplit, fixed_y_maxlen=512,
                        fixed_num_slc_blocks=64, **kw)
    assert torch.equal(out, out2), "optional outputs must not change the result"


@pytest.mark.parametrize("QH,KH,D", [(64, 4, 128), (12, 2, 64)])
@pytest.mark.parametrize("slc_nsplit", [2, 3, 4])
def test_split_decode_with_window_and_selected_blocks_in_parts(device, QH, KH, D, slc_nsplit):
    """slc_nsplit workgroups per (request, kv head) share the window units and the selected blocks and a third
    launch merges them: the selection and lse are those of the uncut second launch bit for bit (the prologue is the
    same code on the same data), the branch outputs and the output agree to bf16 rounding (the merge sums the same
    partial results in another order)."""
    from flash_nsa.inference import decode_split
    ctx = [4096, 333, 48, 31, 1, 777, 2999, 640, 1024, 65, 0, 513, 514]
    case = build_pool([max(c, 1) for c in ctx], KH, D, D, page=128, seed=61)
    prepool(case, [max(c, 1) for c in ctx])
    B = len(ctx)
    d = to_dev(case, device)
    q = randn_bf16(B, QH, D, seed=62).to(device)
    w = randn_bf16(B, QH, 3, seed=63).to(device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=device)
    kw = dict(nsplit=3, fixed_y_maxlen=512, fixed_num_slc_blocks=64, top_n=8, window_size=200)
    ref = decode_split(q, d["k"], d["v"], w, d["bt"], d["cbt"], ctx_t, return_parts=True, **kw)
    got = decode_split(q, d["k"], d["v"], w, d["bt"], d["cbt"], ctx_t, return_parts=True, slc_nsplit=slc_nsplit, **kw)
    live = ctx_t > 0
    assert torch.equal(got[4][:, live], ref[4][:, live]), "selection"
    assert torch.equal(got[5][live], ref[5][live]), "lse"
    assert torch.equal(got[1][live], ref[1][live]), "cmp_o"
    assert_close(got[2][live], ref[2][live], "slc_o", atol=4e-3, rtol=1e-2)
    assert_close(got[3][live], ref[3][live], "swa_o", atol=4e-3, rtol=1e-2)
    assert_close(got[0][live], ref[0][live], "o", atol=8e-3, rtol=1e-2)
    assert float(got[0][~live].abs().max()) == 0.0, "a padded request (context 0) must give zeros"
    out2 = decode_split(q, d["k"], d["v"], w, d["bt"], d["cbt"], ctx_t, slc_nsplit=slc_nsplit, **kw)
    assert torch.equal(got[0], out2), "optional outputs must not change the result"


@pytest.mark.parametrize("window,num_init,num_local,top_n", [(0, 1, 2, 16), (31, 0, 0, 4), (513, 2, 5, 7), (3000, 1, 2, 8)])
@pytest.mark.parametrize("QH,KH,D,VD", [(64, 4, 128, 128), (12, 2, 64, 64), (16, 2, 192, 128)])
def test_split_decode_attends_the_window_in_the_first_launch(device, monkeypatch, QH, KH, D, VD, window, num_init,
                                                             num_local, top_n):
    """win_parts 1..4 against 0 (window in the second launch): selection, lse and compressed branch bit for bit; the
    other branches sum the same partial results in another order (one bf16 rounding of either side apart).  Windows that
    end with a unit and that do not, shorter and longer than the context, all or none of the selection forced."""
    from flash_nsa import _lib
    from flash_nsa.inference import decode_split
    ctx = [4096, 333, 48, 31, 1, 777, 2999, 65, 0, 513, 514]
    case = build_pool([max(c, 1) for c in ctx], KH, D, VD, page=64, seed=71)
    prepool(case, [max(c, 1) for c in ctx])
    d = to_dev(case, device)
    q, w = randn_bf16(len(ctx), QH, D, seed=72).to(device), randn_bf16(len(ctx), QH, 3, seed=73).to(device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=device)
    live = ctx_t > 0
    value = _lib.value

    def run(parts):
        monkeypatch.setattr(_lib, "value", lambda name, *a: parts if name == "nsa_decode_split_window_parts" else value(name, *a))
        return decode_split(q, d["k"], d["v"], w, d["bt"], d["cbt"], ctx_t, return_parts=True, nsplit=3, fixed_y_maxlen=512,
                            fixed_num_slc_blocks=64, top_n=top_n, window_size=window, num_inital=num_init,
                            num_local=num_local)

    ref = run(0)
    for parts in (1, 2, 3, 4):
        got = run(parts)
        for i in (4, 5, 1):
            a, b = (got[i][:, live], ref[i][:, live]) if i == 4 else (got[i][live], ref[i][live])
            assert torch.equal(a, b), (parts, i)
        assert_close(got[2][live], ref[2][live], "slc_o", atol=4e-3, rtol=1e-2)
        assert_close(got[3][live], ref[3][live], "swa_o", atol=4e-3, rtol=1e-2)
        assert_close(got[0][live], ref[0][live], "o", atol=8e-3, rtol=1e-2)
        assert float(got[0][~live].abs().max()) == 0.0


@pytest.mark.parametrize("kernel_size,stride,block", [(128, 64, 128), (32, 16, 64), (16, 16, 32)])
def test_decode_kernels_pool_like_the_pooling_kernel(device, kernel_size, stride, block):
    """The row that the decode kernels pool themselves, for windows longer than a page, inside one, across two and shorter
    than a batch of fetched rows: the pools equal those of the pooling launch bit for bit."""
    from flash_nsa.inference import decode_one_launch, decode_split, kv_mean_pooling_decode
    QH, KH, D, page = 16, 1, 128, 64
    ctx = [n * stride + kernel_size for n in (0, 1, 3, 9, 30)]
    case = build_pool(ctx, KH, D, D, page=page, seed=81)
    slots = torch.tensor([int(case["cbt"][b, 0]) * page + 5 for b in range(len(ctx))], dtype=torch.int32, device=device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=device)
    q, w = randn_bf16(len(ctx), QH, D, seed=82).to(device), randn_bf16(len(ctx), QH, 3, seed=83).to(device)
    d = [to_dev(case, device) for _ in range(3)]
    for x in d:
        x["k"], x["v"] = x["k"].clone(), x["v"].clone()
    sizes = dict(kernel_size=kernel_size, stride=stride)
    kw = dict(fixed_y_maxlen=512, fixed_num_slc_blocks=64, block_size=block, cmp_slot_mapping=slots, **sizes)
    kv_mean_pooling_decode(d[0]["k"], d[0]["v"], block_table=d[0]["bt"], slot_mapping=slots, context_lens=ctx_t, **sizes)
    decode_split(q, d[1]["k"], d[1]["v"], w, d[1]["bt"], d[1]["cbt"], ctx_t, nsplit=2, **kw)
    decode_one_launch(q, d[2]["k"], d[2]["v"], w, d[2]["bt"], d[2]["cbt"], ctx_t, **kw)
    for x in d[1:]:
        assert torch.equal(d[0]["k"], x["k"]) and torch.equal(d[0]["v"], x["v"])


def test_one_launch_decode_pools_the_new_row_itself(device):
    """nsa_decode's one-launch kernel with a slot mapping == pooling kernel followed by the same kernel without:
    the pools end bit-identical and so do the outputs."""
    from flash_nsa.inference import decode_one_launch, kv_mean_pooling_decode
    QH, KH, D = 64, 4, 128
    ctx = [1024, 48, 32, 31, 2001, 656, 645, 4099]       # four of them complete a compressed row at this step
    case = build_pool(ctx, KH, D, D, page=128, seed=41)
    prepool(case, [L - 1 for L in ctx])
    slots = decode_slot_mapping(case)
    assert int((slots >= 0).sum()) == 4
    B = len(ctx)
    q, w = randn_bf16(B, QH, D, seed=42).to(device), randn_bf16(B, QH, 3, seed=43).to(device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=device)
    d1, d2 = to_dev(case, device), to_dev(case, device)
    d2["k"], d2["v"] = d2["k"].clone(), d2["v"].clone()
    kv_mean_pooling_decode(d1["k"], d1["v"], block_table=d1["bt"], slot_mapping=slots.to(device), context_lens=ctx_t)
    o1 = decode_one_launch(q, d1["k"], d1["v"], w, d1["bt"], d1["cbt"], ctx_t, 512, 64)
    o2 = decode_one_launch(q, d2["k"], d2["v"], w, d2["bt"], d2["cbt"], ctx_t, 512, 64,
                           cmp_slot_mapping=slots.to(device))
    assert torch.equal(d1["k"], d2["k"]) and torch.equal(d1["v"], d2["v"])
    assert torch.equal(o1, o2)


@pytest.mark.parametrize("B", [3, 9])
def test_split_decode_graph_replay_equals_eager(device, B):
    """The two-launch path (with the pooling as a launch of its own for 3 requests, inside the first launch for 9)
    captured in a HIP graph: every replay, with eager work and synchronisations in between, equals the eager result,
    also after the static inputs change."""
    from flash_nsa import nsa_decode
    QH, KH, D = 64, 4, 128
    ctx = [2064, 1000, 0, 333, 4128, 640, 2049, 48, 1][:B]
    case = build_pool([max(c, 1) for c in ctx], KH, D, D, page=128, seed=11)
    case["ctx"] = ctx
    case["ys"] = [max((L - 32) // 16 + 1, 0) for L in ctx]
    prepool(case, [max(L - 1, 0) for L in ctx])
    slots = decode_slot_mapping(case)
    d = to_dev(case, device)
    q = randn_bf16(B, QH, D, seed=12).to(device)
    w = randn_bf16(B, QH, 3, seed=13).to(device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=device)
    args = (q, d["k"], d["v"], w, ctx_t, d["bt"], slots.to(device), d["cbt"])
    kw = dict(fixed_y_maxlen=512, fixed_num_slc_blocks=128, cmp_num_splits=4)
    eager = nsa_decode(*args, **kw).clone()
    assert torch.isfinite(eager).all() and (eager[2] == 0).all()
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        nsa_decode(*args, **kw)
    torch.cuda.current_stream().wait_stream(side)
    with torch.cuda.graph(graph):
        out = nsa_decode(*args, **kw)
    for it in range(4):
        out.zero_()
        junk = torch.randn(1 << 20, device=device).sum()  # the program's own eager work between replays
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {it} differs from eager"
    q.copy_(randn_bf16(B, QH, D, seed=14).to(device))
    eager2 = nsa_decode(*args, **kw).clone()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, eager2)


@pytest.mark.parametrize("nsplit", [2, 8])
def test_split_decode_pools_the_new_row_itself(device, nsplit):
    """The two-launch decode with a slot mapping == pooling kernel followed by the same path without: the pools end
    bit-identical and so do the outputs (the part that owns the last unit pools the row before it attends it), and
    nsa_decode takes that route when asked for parts."""
    from flash_nsa import nsa_decode
    from flash_nsa.inference import decode_split, kv_mean_pooling_decode
    QH, KH, D = 64, 4, 128
    ctx = [1024, 48, 32, 31, 2001, 656, 645, 4099, 4128, 2064]   # six of them complete a compressed row at this step
    case = build_pool(ctx, KH, D, D, page=128, seed=41)
    prepool(case, [L - 1 for L in ctx])
    slots = decode_slot_mapping(case)
    assert int((slots >= 0).sum()) == 6
    B = len(ctx)
    q, w = randn_bf16(B, QH, D, seed=42).to(device), randn_bf16(B, QH, 3, seed=43).to(device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=device)
    d1, d2, d3 = to_dev(case, device), to_dev(case, device), to_dev(case, device)
    for d in (d2, d3):
        d["k"], d["v"] = d["k"].clone(), d["v"].clone()
    kw = dict(fixed_y_maxlen=512, fixed_num_slc_blocks=128)
    kv_mean_pooling_decode(d1["k"], d1["v"], block_table=d1["bt"], slot_mapping=slots.to(device), context_lens=ctx_t)
    o1 = decode_split(q, d1["k"], d1["v"], w, d1["bt"], d1["cbt"], ctx_t, nsplit=nsplit, **kw)
    o2 = decode_split(q, d2["k"], d2["v"], w, d2["bt"], d2["cbt"], ctx_t, nsplit=nsplit,
                      cmp_slot_mapping=slots.to(device), **kw)
    assert torch.equal(d1["k"], d2["k"]) and torch.equal(d1["v"], d2["v"])
    assert torch.equal(o1, o2)
    o3 = nsa_decode(q, d3["k"], d3["v"], w, ctx_t, d3["bt"], slots.to(device), d3["cbt"], cmp_num_splits=nsplit, **kw)
    assert torch.equal(d1["k"], d3["k"]) and torch.equal(d1["v"], d3["v"])
    assert torch.equal(o1, o3)


@pytest.mark.parametrize("D,VD", [(192, 128), (32, 32), (256, 256)])
def test_decode_qk192_v128_equals_training_last_row(device, D, VD):
    """Dqk = 192, Dv = 128, 2 kv heads (the head shape of upstream's inference notebook, cell 43), and head dims of 32
    and 256, which decode stage by stage (192: the fused kernels): the output equals the last row of the training forward
    on the gathered contiguous sequence."""
    from flash_nsa import nsa_decode, NSAConfig, NSACore
    QH, KH = 16, 2
    ctx = [1000, 333, 64, 2049]
    case = build_pool(ctx, KH, D, VD, page=128, seed=51)
    prepool(case, [L - 1 for L in ctx])
    slots = decode_slot_mapping(case)
    B = len(ctx)
    q, w = randn_bf16(B, QH, D, seed=52), randn_bf16(B, QH, 3, seed=53)
    d = to_dev(case, device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=device)
    o = nsa_decode(q.to(device), d["k"], d["v"], w.to(device), ctx_t, d["bt"], slots.to(device), d["cbt"],
                   fixed_y_maxlen=256, fixed_num_slc_blocks=64)
    assert o.shape == (B, QH, VD) and torch.isfinite(o).all()
    core = NSACore(NSAConfig(qk_head_dim=D, v_head_dim=VD, num_heads=QH, num_kv_heads=KH))
    for b in range(B):
        L = ctx[b]
        ks = O.gather_rows(case["k"], case["bt"][b], L).to(device)
        vs = O.gather_rows(case["v"], case["bt"][b], L).to(device)
        qs, ws = randn_bf16(L, QH, D, seed=300 + b), randn_bf16(L, QH, 3, seed=400 + b)
        qs[-1], ws[-1] = q[b], w[b]
        with torch.no_grad():
            full = core(qs.to(device), ks, vs, ws.to(device), torch.tensor([0, L], dtype=torch.int32, device=device))
        assert_close(o[b], full[-1], f"decode vs training row (request {b})", atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("B,cap,blocks,columns,splits", [(33, 16384, 4096, None, 0), (2, 16384, 4096, None, 1),
                                                         (2, 512, 64, 24000, 1), (2, 512, 64, 24000, 2)])
def test_decode_qk192_beyond_the_lds_of_the_fused_kernels(device, B, cap, blocks, columns, splits):
    """Capacities and page tables that no fused kernel holds at 192 channels are served stage by stage: bit for bit what
    the stages give."""
    from flash_nsa import nsa_decode
    from flash_nsa.inference import kv_mean_pooling_decode, nsa_decode_staged
    QH, KH, D, VD = 64, 4, 192, 128
    ctx = [(517 * i) % 1500 + 16 * (i % 3) for i in range(B)]
    ctx[0] = 1024
    case = build_pool([max(c, 1) for c in ctx], KH, D, VD, page=64, seed=61)
    prepool(case, [max(c - 1, 0) for c in ctx])
    slots = decode_slot_mapping(case).to(device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=device)
    q, w = randn_bf16(B, QH, D, seed=62).to(device), randn_bf16(B, QH, 3, seed=63).to(device)
    d = to_dev(case, device)
    bt = d["bt"]
    if columns:
        bt = torch.full((B, columns), -1, dtype=torch.int32, device=device)
        bt[:, :d["bt"].size(1)] = d["bt"]
    kw = dict(fixed_y_maxlen=cap, fixed_num_slc_blocks=blocks, cmp_num_splits=splits)
    k, v = d["k"].clone(), d["v"].clone()
    out = nsa_decode(q, d["k"], d["v"], w, ctx_t, bt, slots, d["cbt"], **kw)
    kv_mean_pooling_decode(k, v, block_table=bt, slot_mapping=slots, context_lens=ctx_t)
    assert torch.equal(k, d["k"]) and torch.equal(v, d["v"])
    assert torch.equal(out, nsa_decode_staged(q, k, v, w, ctx_t, bt, d["cbt"], **kw))


@pytest.mark.parametrize("D,VD", [(128, 128), (192, 128)])
@pytest.mark.parametrize("splits", [1, 2])
def test_decode_refuses_operands_that_its_kernels_would_misread(device, D, VD, splits):
    """The fused kernels read the gates and the newest rows as bf16 with contiguous channels and a slot per request, as
    the stage-by-stage functions check."""
    from flash_nsa import nsa_decode
    QH, KH, ctx = 16, 2, [100, 64]
    case = build_pool(ctx, KH, D, VD, page=64, seed=65)
    prepool(case, ctx)
    d = to_dev(case, device)
    q, w = randn_bf16(2, QH, D, seed=66).to(device), randn_bf16(2, QH, 3, seed=67).to(device)
    nk, nv = randn_bf16(2, KH, D, seed=68).to(device), randn_bf16(2, KH, VD, seed=69).to(device)
    at = torch.tensor([int(d["bt"][0, 1]) * 64 + 35, int(d["bt"][1, 0]) * 64 + 63], dtype=torch.int32, device=device)

    def run(w=w, **kw):
        return nsa_decode(q, d["k"], d["v"], w, torch.tensor(ctx, dtype=torch.int32, device=device), d["bt"],
                          torch.full((2,), -1, dtype=torch.int32, device=device), d["cbt"], cmp_num_splits=splits,
                          fixed_y_maxlen=512, fixed_num_slc_blocks=64, **kw)

    run(new_k=nk, new_v=nv, slot_mapping=at)
    for bad in (dict(w=w.float()), dict(w=w.transpose(1, 2).contiguous().transpose(1, 2)), dict(w=w[:, :8]),
                dict(new_k=nk.float(), new_v=nv, slot_mapping=at), dict(new_k=nk, new_v=nv.float(), slot_mapping=at),
                dict(new_k=nk, new_v=nv, slot_mapping=at[:1])):
        with pytest.raises(AssertionError):
            run(**bad)


@pytest.mark.parametrize("D,VD", [(128, 128), (192, 128)])
def test_decode_takes_more_parts_than_it_can_merge_as_64(device, D, VD):
    """cmp_num_splits is a hint: the stage-by-stage path has no use for it, the kernels with parts merge up to 64."""
    from flash_nsa import nsa_decode
    QH, KH, ctx = 16, 2, [4099, 64]
    case = build_pool(ctx, KH, D, VD, page=64, seed=75)
    prepool(case, ctx)
    d = to_dev(case, device)
    q, w = randn_bf16(2, QH, D, seed=76).to(device), randn_bf16(2, QH, 3, seed=77).to(device)
    run = lambda n: nsa_decode(q, d["k"], d["v"], w, torch.tensor(ctx, dtype=torch.int32, device=device), d["bt"],
                               torch.full((2,), -1, dtype=torch.int32, device=device), d["cbt"], cmp_num_splits=n,
                               fixed_y_maxlen=512, fixed_num_slc_blocks=128)
    assert torch.equal(run(100), run(64))


def test_decode_small_batch_long_context_takes_the_split_path(device):
    """nsa_decode with its defaults on 2 requests of 40K tokens (fixed_y_maxlen 4096): the compressed branch is cut
    into parts by itself; the result equals the two-launch path without parts up to ties of the selection, and head
    dims the split kernels are not built for (192/128) are not routed there."""
    from flash_nsa import nsa_decode
    from flash_nsa.inference import auto_cmp_splits, decode_cmp_topk, decode_slc_swa_combine
    assert auto_cmp_splits(2, 4, 4096) == 8 and auto_cmp_splits(64, 4, 4096) == 1 and auto_cmp_splits(2, 4, 512) == 1
    QH, KH, D = 64, 4, 128
    ctx = [40000, 33333]
    case = build_pool(ctx, KH, D, D, page=256, seed=61)
    prepool(case, ctx)
    d = to_dev(case, device)
    q, w = randn_bf16(2, QH, D, seed=62).to(device), randn_bf16(2, QH, 3, seed=63).to(device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32, device=device)
    none = torch.full((2,), -1, dtype=torch.int32, device=device)
    kw = dict(fixed_y_maxlen=4096, fixed_num_slc_blocks=1024)
    o = nsa_decode(q, d["k"], d["v"], w, ctx_t, d["bt"], none, d["cbt"], **kw)
    cmp_o, topk = decode_cmp_topk(q, d["k"], d["v"], d["cbt"], ctx_t, **kw)
    ref = decode_slc_swa_combine(q, d["k"], d["v"], w, topk, cmp_o, d["bt"], ctx_t)
    err = (o.float() - ref.float()).abs().view(2, KH, -1).amax(-1)           # per (request, kv head)
    assert int((err > 1e-2).sum()) <= 1, err
    o1 = nsa_decode(q, d["k"], d["v"], w, ctx_t, d["bt"], none, d["cbt"], cmp_num_splits=1, **kw)
    assert_close(o1, ref, "no parts", atol=8e-3, rtol=1e-2)


def test_decode_more_workgroups_than_compute_units(device):
    """320 requests x 2 kv heads = 640 workgroups of the one-launch kernel on 256 CUs (several rounds per CU), contexts
    of 40-1000 tokens (at most 16 selection blocks, so every block is selected and no tie can change the result):
    equal to the stage-by-stage decode, and identical when the same batch is run again."""
    from flash_nsa import nsa_decode
    from flash_nsa.inference import nsa_decode_staged
    from synthetic_decode import build_decode_case, pool_all_rows
    c = build_decode_case(device, B=320, QH=32, KH=2, D=128, page=64, lo=40, hi=1000, seed=11)
    pool_all_rows(c, device)
    kw = dict(fixed_y_maxlen=128, fixed_num_slc_blocks=32)
    args = (c["q"], c["k"], c["v"], c["w"], c["ctx"], c["bt"])
    fused = nsa_decode(*args, c["slots"], c["cbt"], **kw)
    staged = nsa_decode_staged(*args, c["cbt"], **kw)
    assert torch.isfinite(fused).all()
    assert_close(fused, staged, "one-launch vs staged decode, 640 workgroups", atol=8e-3, rtol=1e-2)
    again = nsa_decode(*args, torch.full_like(c["slots"], -1), c["cbt"], **kw)
    assert torch.equal(fused, again)


@pytest.mark.parametrize("QH,KH,D,VD", [(32, 2, 128, 128), (12, 2, 64, 64), (24, 2, 192, 128)])
@pytest.mark.parametrize("cap", [300, 2048])
def test_one_launch_decode_with_four_waves(device, QH, KH, D, VD, cap):
    """The one-launch decode kernel with two workgroups of four waves per CU, capacities that keep every probability in
    LDS and that spill some to scratch memory, and the 192-channel kernel (all of them spilled, fp32): contexts around
    the unit, block and spill boundaries.  The kept probabilities are those of eight waves, so the selection is the same
    up to fp32 rounding; 192 channels are compared with the stage-by-stage kernels.  Outputs are rounded to bf16 from
    differently ordered fp32 sums of bf16-rounded P: 2^-7 relative and 2^-7 absolute (N(0,1) values)."""
    from flash_nsa import _lib
    from flash_nsa.inference import decode_one_launch, nsa_decode_staged
    ctx = [4800, 1, 31, 32, 33, 0, 1055, 1056, 1057, 4799] + ([32768, 16431, 28000] if cap == 2048 else [])
    case = build_pool(ctx, KH, D, VD, page=128, seed=21)
    prepool(case, ctx)
    B = len(ctx)
    q, w = randn_bf16(B, QH, D, seed=22).to(device), randn_bf16(B, QH, 3, seed=23).to(device)
    d = to_dev(case, device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32).to(device)
    kw = dict(fixed_y_maxlen=cap, fixed_num_slc_blocks=512)
    runs = {}
    try:
        for waves in (4, 8):
            _lib.call("nsa_set_tuning", b"decode_waves", waves)
            runs[waves] = decode_one_launch(q, d["k"], d["v"], w, d["bt"], d["cbt"], ctx_t, return_parts=True, **kw)
    finally:
        _lib.call("nsa_reset_tuning")
    if D > 128:
        ref = nsa_decode_staged(q, d["k"], d["v"], w, ctx_t, d["bt"], d["cbt"], **kw)
    else:
        ref = runs[8][0]
        same = (runs[4][4] == runs[8][4]).all(-1)
        assert int((~same).sum()) <= 1, "selections differ"   # one fp32 near-tie at the cut is excused
    bad = (runs[4][0].float() - ref.float()).abs() > 2 ** -7 + 2 ** -7 * ref.float().abs()
    assert int(bad.flatten(1).any(1).sum()) <= 1              # the request of that tie


@pytest.mark.parametrize("QH,KH,D,page,cached,new", [
    (16, 2, 64, 64, [0, 130, 0, 900], [700, 17, 1, 124]),    # whole prompts, chunks behind prefixes, the longest context that fits
    (6, 2, 128, 128, [37, 0], [300, 5]),                     # groups of 3 q-heads
    (64, 4, 128, 256, [0, 0, 200], [498, 345, 56]),
])
def test_prefill_of_short_contexts_in_one_launch_equals_two(device, QH, KH, D, page, cached, new):
    """Contexts of at most top_n * block_size tokens: every branch and the gated sum in one launch are the bits of the compressed
    branch's launch and the window's."""
    from flash_nsa.inference import stages as S
    ctx = [c + n for c, n in zip(cached, new)]
    case = build_pool(ctx, KH, D, D, page=page, seed=9)
    prepool(case, ctx)
    d = to_dev(case, device)
    xcu, t = make_cu(new).to(device), sum(new)
    q, w = randn_bf16(t, QH, D, seed=10).to(device), randn_bf16(t, QH, 3, seed=11).to(device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32).to(device)
    got = S.short_prefill(q, d["k"], d["v"], w, xcu, max(new), d["bt"], d["cbt"], ctx_t, 1024)
    cmp_o, _ = S.cmp_attn_prefill(q, d["k"], d["v"], xcu, max(new), d["cbt"], ctx_t)
    want = S.swa_combine_prefill(q, d["k"], d["v"], cmp_o, torch.empty_like(cmp_o), w, xcu, max(new), d["bt"], ctx_t, all_below=1024)
    assert torch.equal(got, want)


@pytest.mark.parametrize("QH,KH,D,VD,all_below", [(16, 1, 128, 128, 2560), (6, 2, 64, 64, 3072), (8, 2, 192, 128, 1024), (4, 1, 256, 256, 2560)])
def test_short_prefill_of_a_request_does_not_depend_on_the_others(device, QH, KH, D, VD, all_below):
    """All orders in which a launch takes its rows (by the longest context that selects everything): each request has the bits that it has
    alone."""
    from flash_nsa.inference import stages as S
    cached, new = ([0, 130, 1500, 1, 0], [2560, 700, 33, 129, 1]) if all_below > 1024 else ([0, 130, 900, 1, 0], [1024, 700, 33, 129, 1])
    ctx = [c + n for c, n in zip(cached, new)]
    case = build_pool(ctx, KH, D, VD, page=64, seed=12)
    prepool(case, ctx)
    d = to_dev(case, device)
    t = sum(new)
    q, w = randn_bf16(t, QH, D, seed=13).to(device), randn_bf16(t, QH, 3, seed=14).to(device)
    ctx_t = torch.tensor(ctx, dtype=torch.int32).to(device)
    got = S.short_prefill(q, d["k"], d["v"], w, make_cu(new).to(device), max(new), d["bt"], d["cbt"], ctx_t, all_below)
    assert bool(torch.isfinite(got).all())
    at = 0
    for b, n in enumerate(new):
        alone = S.short_prefill(q[at:at + n], d["k"], d["v"], w[at:at + n], make_cu([n]).to(device), n, d["bt"][b:b + 1], d["cbt"][b:b + 1],
                                ctx_t[b:b + 1], all_below)
        assert torch.equal(got[at:at + n], alone), b
        at += n
