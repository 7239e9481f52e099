"""dq of the compressed and the window branch from the dS that their dk / dv kernels store, against the kernels that compute S
and dP again (what the deterministic mode runs), over the shapes, sizes and ranges of tokens that the path takes."""
import pytest
import torch

from gpu_util import assert_close, make_cu, make_qkvw, randn_bf16

pytestmark = pytest.mark.gpu


def _grads(core, ts, cu, do, device):
    ts = [t.to(device).detach().requires_grad_() for t in ts]
    out = core(*ts, cu)
    out.backward(do)
    return [out.detach()] + [t.grad for t in ts]


# ends of tiles of 64 rows (8 .. 1 tokens), of units of 32 keys, of groups of 128 positions, and sequences without a
# compressed row; mb: a scratch limit in MB that needs several ranges; whole: ranges of the whole batch, as where a helper does not
# have the lengths on the host, else of parts of it
CASES = [
    # QH, KH, D, VD, lens, mb, whole, settings
    (8, 1, 128, 128, [1, 31, 32, 33, 700], 0, False, {}),
    (16, 1, 128, 128, [1024, 1025, 47, 1279], 0, False, dict(top_n=4)),
    (32, 1, 128, 128, [0, 515, 0, 640], 0, False, dict(window_size=100, top_n=3)),
    (64, 1, 128, 128, [513, 1, 129], 0, False, dict(window_size=0, top_n=3)),
    (64, 4, 128, 128, [4700], 300, False, {}),
    (64, 1, 128, 128, [2047, 300, 2500, 5], 200, True, dict(top_n=6)),
    (64, 1, 128, 128, [2047, 300, 2500, 5], 200, False, dict(top_n=6)),
    (64, 4, 192, 128, [130, 4300], 190, True, dict(window_size=300)),
    (64, 4, 192, 128, [130, 4300], 165, False, dict(window_size=300)),
    (32, 2, 192, 128, [900, 64, 333], 0, False, dict(block_size=96, kernel_size=64, stride=32, top_n=5)),
    (16, 2, 128, 128, [1500, 200], 0, False, dict(window_size=2000)),
    (16, 1, 192, 128, [777], 0, False, dict(kernel_size=16, stride=8, block_size=32, top_n=40)),
    # chunks of 256 queries, cut from the first row of a share in the middle of a sequence
    (32, 2, 128, 128, [3063, 9859], 200, True, {}),
    # the keys before the window in places taken in turn
    (64, 1, 128, 128, [1100, 1024, 1300, 1111, 1029], 500, True, dict(window_size=100)),
    # ranges of an eighth of the tokens that fill the GPU
    (64, 4, 128, 128, [4700], 80, False, {}),
    (8, 1, 128, 128, [9001], 28, False, {}),
    (64, 1, 128, 128, [2047, 300, 2500, 5], 80, True, dict(top_n=6)),
    (64, 4, 192, 128, [130, 4300], 150, True, dict(window_size=300)),
    # a long sequence between many short ones
    (64, 4, 128, 128, [40, 0, 350, 5, 350, 350, 4500, 33, 350, 350, 0, 350, 31], 300, False, {}),
]


def _wide(t):
    """t in rows twice as long"""
    return torch.cat([t, t], -1)[..., :t.size(-1)]


@pytest.mark.parametrize("QH,KH,D,VD,lens,mb,whole,settings", CASES)
def test_dq_from_stored_ds_is_the_recomputed_one(device, QH, KH, D, VD, lens, mb, whole, settings):
    from flash_nsa import NSAConfig, NSACore, _lib
    from flash_nsa.ops import bwd_ds
    from flash_nsa.utils import NSAHelper as H
    T = sum(lens)
    cu = make_cu(lens).to(device)
    ts = make_qkvw(T, QH, KH, D, VD, seed=300)
    do = randn_bf16(T, QH, VD, seed=301).to(device)
    if mb:
        ts, do = [*map(_wide, ts[:3]), ts[3]], _wide(do)
    core = NSACore(NSAConfig(qk_head_dim=D, v_head_dim=VD, num_heads=QH, num_kv_heads=KH, **settings))
    core = core.to(device=device, dtype=torch.bfloat16)
    made, init = [], bwd_ds.DenseDs.__init__

    def recorded(self, *a, **k):
        host, H._host_cu = H._host_cu, None if whole else H._host_cu
        init(self, *a, **k)
        H._host_cu = host
        made.append(self)

    bwd_ds.DenseDs.__init__ = recorded
    if mb:
        _lib.call("nsa_set_tuning", b"dense_ds_mb", mb)
    try:
        got = _grads(core, ts, cu, do, device)
        H.set_deterministic(True)
        want = _grads(core, ts, cu, do, device)
    finally:
        H.set_deterministic(False)
        _lib.call("nsa_reset_tuning")
        bwd_ds.DenseDs.__init__ = init
    assert len(made) == 1 and (len(made[0].ranges) > 1) == (mb > 0)
    assert len({id(p) for p, *_ in made[0].ranges}) == 1 or not whole
    assert torch.equal(got[0], want[0])
    # the same products of bf16 operands whose last bit may differ (P from differently rounded exponents): the bar that both
    # are held to against the oracle
    for a, b, name in zip(got[1:], want[1:], ("dq", "dk", "dv", "dw")):
        assert_close(a, b, name, row_scale=name in ("dk", "dv"))
        d = (a.double() - b.double()).norm() / b.double().norm()
        assert d < 4e-3, (name, float(d))  # 2^-8


@pytest.mark.parametrize("QH,KH,lens,cmp_mb,swa_mb", [(16, 1, [12000, 8200], 200, 200), (64, 4, [2600, 2500], 80, 200)])
def test_branch_backward_ranges_give_the_same_bits(device, QH, KH, lens, cmp_mb, swa_mb):
    """The two branches by themselves: whole and in ranges of tokens, dq bit for bit; into bf16, stored fp32 and added to fp32."""
    from flash_nsa import _lib
    from flash_nsa.ops import bwd_ds
    from flash_nsa.ops._common import delta_of
    from flash_nsa.ops.compress_attn import cmp_attn_bwd, cmp_attn_fwd
    from flash_nsa.ops.compress_kv import mean_pooling_fwd
    from flash_nsa.ops.sliding_window_attention import swa_bwd, swa_fwd
    from flash_nsa.utils import NSAHelper as H
    T = sum(lens)
    H.set_hyperparameters()
    H.init_cu_seqlens(make_cu(lens).to(device))
    q, k, v, _ = [t.to(device) for t in make_qkvw(T, QH, KH, 128, 128, seed=310)]
    do = randn_bf16(T, QH, 128, seed=311).to(device)
    ck, cv = mean_pooling_fwd(k), mean_pooling_fwd(v)
    for fwd, bwd, args, small in ((cmp_attn_fwd, cmp_attn_bwd, (q, ck, cv), cmp_mb), (swa_fwd, swa_bwd, (q, k, v), swa_mb)):
        o, lse = fwd(*args)
        delta = delta_of(o, do)
        runs = []
        for mb in (4096, small):
            _lib.call("nsa_set_tuning", b"dense_ds_mb", mb)
            try:
                ranges = bwd_ds.DenseDs(q, k, with_cmp=bwd is cmp_attn_bwd, with_swa=bwd is swa_bwd).ranges
                assert len(ranges) == 1 if mb == 4096 else len(ranges) > 1
                runs.append(bwd(*args, o, lse, do, delta=delta))
                base = torch.randn(T, QH, 128, device=device)
                added = bwd(*args, o, lse, do, dq=base.clone(), delta=delta)[0]
            finally:
                _lib.call("nsa_reset_tuning")
            assert_close((added - base).to(torch.bfloat16), runs[-1][0], "added dq", atol=1e-3)
        assert torch.equal(runs[0][0], runs[1][0])
        for a, b, name in zip(runs[0][1:], runs[1][1:], ("dk", "dv")):
            assert_close(a, b, name, atol=2e-3, rtol=8e-3, row_scale=True)


def test_scratch_that_does_not_fit_is_not_taken(device):
    """Where the limit does not hold the least range, dq is computed apart: the bits of the deterministic mode's dq."""
    from flash_nsa import _lib
    from flash_nsa.ops._common import delta_of
    from flash_nsa.ops.compress_attn import cmp_attn_bwd, cmp_attn_fwd
    from flash_nsa.ops.compress_kv import mean_pooling_fwd
    from flash_nsa.ops.sliding_window_attention import swa_bwd, swa_fwd
    from flash_nsa.utils import NSAHelper as H
    QH, KH, lens = 16, 1, [700, 90]
    T = sum(lens)
    H.set_hyperparameters()
    H.init_cu_seqlens(make_cu(lens).to(device))
    q, k, v, _ = [t.to(device) for t in make_qkvw(T, QH, KH, 128, 128, seed=320)]
    do = randn_bf16(T, QH, 128, seed=321).to(device)
    ck, cv = mean_pooling_fwd(k), mean_pooling_fwd(v)
    for fwd, bwd, args in ((cmp_attn_fwd, cmp_attn_bwd, (q, ck, cv)), (swa_fwd, swa_bwd, (q, k, v))):
        o, lse = fwd(*args)
        delta, got = delta_of(o, do), []
        for mb, deterministic in ((0, False), (4096, True)):
            _lib.call("nsa_set_tuning", b"dense_ds_mb", mb)
            H.set_deterministic(deterministic)
            try:
                got.append(bwd(*args, o, lse, do, delta=delta)[0])
            finally:
                H.set_deterministic(False)
                _lib.call("nsa_reset_tuning")
        assert torch.equal(*got)
