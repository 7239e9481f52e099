"""Decode cut into parts: the launch that writes the newest token's row attends it from registers; the block selection by
counting, at the numbers of blocks and candidates where its list overflows."""
import pytest
import torch

from gpu_util import randn_bf16
from paged_util import build_pool, cmp_row_slot, prepool

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,VD,KH,G", [(128, 128, 2, 16), (192, 128, 2, 16), (64, 64, 2, 8)])
@pytest.mark.parametrize("page,window", [(64, 512), (256, 100), (128, 0)])
def test_newest_row_written_by_the_first_launch(device, D, VD, KH, G, page, window):
    """Same outputs and caches, bit for bit, as with the row stored beforehand: the row first / last in a unit and a page,
    with and without a compressed row that it completes, one token of context, padding, a slot that is not the block
    table's (the table's row is then the one attended)."""
    from flash_nsa.inference import store_kvcache
    from flash_nsa.inference.stages import decode_split
    ctx = [1, 31, 32, 33, 64, 65, 256, 257, 800, 801, 1024, 4096, 0, 640, 128]
    B = len(ctx)
    case = build_pool(ctx, KH, D, VD, page=page, seed=3)
    prepool(case, [max(n - 1, 0) for n in ctx])
    slots, cmp_slots = [], []
    for b, n in enumerate(ctx):
        slots.append(int(case["bt"][b, (n - 1) // page]) * page + (n - 1) % page if n else -1)
        done = n >= 32 and (n - 32) % 16 == 0
        cmp_slots.append(cmp_row_slot(case, b, (n - 32) // 16) if done else -1)
    spare = next(i for i in range(case["k"].size(0)) if not (case["bt"] == i).any() and not (case["cbt"] == i).any())
    slots[-2], slots[-1] = spare * page + 5, -1
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=device)
    q, w = randn_bf16(B, KH * G, D, seed=5).to(device), randn_bf16(B, KH * G, 3, seed=6).to(device)
    new_k, new_v = randn_bf16(B, KH, D, seed=7).to(device), randn_bf16(B, KH, VD, seed=8).to(device)
    kw = dict(fixed_y_maxlen=512, fixed_num_slc_blocks=64, window_size=window, cmp_slot_mapping=i32(cmp_slots), top_n=8)
    results = []
    for stored in (True, False):
        for nsplit in (2, 16):
            k, v = case["k"].to(device).clone(), case["v"].to(device).clone()
            new = dict(new_k=new_k, new_v=new_v, slot_mapping=i32(slots))
            if stored:
                store_kvcache(new_k, new_v, k, v, new.pop("slot_mapping"))
                new = {}
            o = decode_split(q, k, v, w, case["bt"].to(device), case["cbt"].to(device), i32(ctx), nsplit=nsplit, **new, **kw)
            results.append((o, k, v))
    for a, b in zip(results[:2], results[2:]):
        for x, y in zip(a, b):
            assert torch.equal(x, y)


@pytest.mark.parametrize("D,VD,KH,G", [(128, 128, 2, 16), (192, 128, 2, 16), (64, 64, 2, 8)])
@pytest.mark.parametrize("page,window", [(64, 512), (256, 100), (128, 0)])
def test_newest_row_into_a_slot_never_written(device, D, VD, KH, G, page, window):
    """As above, bit for bit, where every pool row that holds no token yet, the newest's own slot among them, is NaN (a new
    pool is uninitialised memory): the newest row first, in the middle and last in a unit, and the only one of its window."""
    from flash_nsa.inference import store_kvcache
    from flash_nsa.inference.stages import decode_split
    ctx = [1, 2, 31, 32, 33, 48, 64, 65, 257, 800, 1024, 1025, 4096]
    B = len(ctx)
    case = build_pool(ctx, KH, D, VD, page=page, seed=4)
    prepool(case, [n - 1 for n in ctx])
    slots, cmp_slots, written = [], [], []
    for b, n in enumerate(ctx):
        rows = [int(case["bt"][b, i // page]) * page + i % page for i in range(n)]
        written += rows[:-1]
        slots.append(rows[-1])
        y = max((n - 1 - 32) // 16 + 1, 0)
        written += [cmp_row_slot(case, b, i) for i in range(y)]
        cmp_slots.append(cmp_row_slot(case, b, y) if case["ys"][b] > y else -1)
    for name in ("k", "v"):
        flat = case[name].view(-1, *case[name].shape[2:])
        empty = torch.ones(len(flat), dtype=torch.bool)
        empty[written] = False
        flat[empty] = float("nan")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=device)
    q, w = randn_bf16(B, KH * G, D, seed=15).to(device), randn_bf16(B, KH * G, 3, seed=16).to(device)
    new_k, new_v = randn_bf16(B, KH, D, seed=17).to(device), randn_bf16(B, KH, VD, seed=18).to(device)
    kw = dict(fixed_y_maxlen=512, fixed_num_slc_blocks=64, window_size=window, cmp_slot_mapping=i32(cmp_slots), top_n=8)
    for nsplit in (2, 16):
        results = []
        for new in ({}, dict(new_k=new_k, new_v=new_v, slot_mapping=i32(slots))):
            k, v = case["k"].to(device), case["v"].to(device)
            if not new:
                store_kvcache(new_k, new_v, k, v, i32(slots))
            o = decode_split(q, k, v, w, case["bt"].to(device), case["cbt"].to(device), i32(ctx), nsplit=nsplit, **new, **kw)
            results.append((o, k, v))
        assert torch.isfinite(results[0][0]).all()
        for x, y in zip(*results):
            assert torch.equal(x.view(torch.int16), y.view(torch.int16))


@pytest.mark.parametrize("blocks", [20, 64, 65, 512, 513, 2048])
@pytest.mark.parametrize("values", [1, 3, 40, 100000])
def test_selection_by_counting(device, blocks, values):
    """Decode's own selection against a stable sort of the same scores.  Scores from few different values: ties go to the
    lower block, and more scores at the bound than the short list holds take the register form."""
    from flash_nsa.inference.stages import decode_slc_swa_combine
    KH, G, D, top_n, page = 2, 8, 64, 16, 128
    n = blocks * 64
    case = build_pool([n], KH, D, D, page=page, seed=11)
    y = (n - 32) // 16 + 1
    g = torch.Generator().manual_seed(blocks * 1000 + values)
    score = torch.randint(1, values + 1, (KH, blocks), generator=g).float() / 1024  # exact in every sum of four
    pg = torch.zeros(1, KH, (y + 3) // 4 * 4)
    for j in range(blocks):  # one compressed key inside every block carries its score: no overlap with its neighbours
        pg[0, :, min(4 * j + 1, y - 1)] = score[:, j]
    q, w = randn_bf16(1, KH * G, D, seed=12).to(device), randn_bf16(1, KH * G, 3, seed=13).to(device)
    cmp_o = torch.zeros(1, KH * G, D, dtype=torch.bfloat16, device=device)
    _, topk = decode_slc_swa_combine(q, case["k"].to(device), case["v"].to(device), w, None, cmp_o, case["bt"].to(device),
                                     torch.tensor([n], dtype=torch.int32, device=device), top_n=top_n, pg=pg.to(device),
                                     fixed_num_slc_blocks=blocks)
    for kh in range(KH):
        forced = [0, blocks - 1, blocks - 2]
        rest = [j for j in range(1, blocks - 2)]
        ref = forced + sorted(rest, key=lambda j: (-float(score[kh, j]), j))[:top_n - 3]
        assert topk[kh, 0].tolist() == ref


@pytest.mark.parametrize("QH,KH,D", [(16, 2, 64), (32, 2, 128)])
@pytest.mark.parametrize("blocks", [72, 600])
def test_one_launch_selection_is_the_oracles(device, QH, KH, D, blocks):
    """The one-launch kernel's picks against the oracle's, which may differ only between blocks whose scores lie within 1e-3 of
    each other; capacities of fewer and of more blocks than its smallest selector holds."""
    from flash_nsa.inference import decode_one_launch
    from oracle import nsa_oracle as O
    ctx = [1, 640, 1025, 1777, 4097]
    case = build_pool(ctx, KH, D, D, seed=21)
    prepool(case, ctx)
    q, w = randn_bf16(len(ctx), QH, D, seed=22), randn_bf16(len(ctx), QH, 3, seed=23)
    lens, cu = torch.tensor(ctx, dtype=torch.int32), torch.arange(len(ctx) + 1, dtype=torch.int32)
    _, parts = O.nsa_paged_forward(q.float(), case["k"].float(), case["v"].float(), w.float(), cu, lens, case["bt"], case["cbt"],
                                   O.OracleConfig(block_size=64, top_n=16), return_parts=True)
    own = torch.cat([p["topk"] for p in parts], 1)
    topk = decode_one_launch(*[t.to(device) for t in (q, case["k"], case["v"], w, case["bt"], case["cbt"], lens)],
                             fixed_y_maxlen=512, fixed_num_slc_blocks=blocks, block_size=64, top_n=16, return_parts=True)[4].cpu()
    _, differ, wrong = O.topk_mismatch_report(topk, own, [p["imp"] for p in parts], cu, 64, 16, tie_tol=1e-3,
                                              t_offsets=[n - 1 for n in ctx])
    assert wrong == 0 and differ <= 1
