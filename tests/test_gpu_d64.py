"""Head dim 64 on the MFMA kernel: 16-bit caches, both V layouts, pages of one
and of several 16-token blocks, groups at the edges of its q-head blocks,
context lengths around page, block and wave boundaries. The fp32 output
carries no rounding of its own, so the bound is the arithmetic's: p in full
(24 bits in bf16 parts, fp32 over an fp16 cache) and fp32 sums of up to 3000
terms, a few 1e-7 of the row."""
import numpy as np
import pytest
import torch

import oracle
import sched_pd
import workloads
from sched_rt import SchedPlane

pytestmark = pytest.mark.gpu

CTX = [1, 15, 16, 17, 63, 64, 65, 128, 257, 1000, 2999, 0]


@pytest.mark.parametrize("kv", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", ["tokmajor", "dmajor"])
@pytest.mark.parametrize("ps", [16, 32, 256])
@pytest.mark.parametrize("G", [4, 7, 16])
def test_d64_matches_the_oracle(kv, layout, ps, G):
    hkv = 2
    b = workloads.make_batch(np.asarray(CTX), num_q_heads=G * hkv, num_kv_heads=hkv, head_dim=64,
                             page_size=ps, kv_dtype=kv, q_dtype=kv, seed=G + ps, device="cuda")
    v = b["v_pool"]
    if layout == "tokmajor":
        v = v.permute(0, 1, 3, 2).contiguous()
    out = torch.full((len(CTX), G * hkv, 64), 7.0, device="cuda")
    args = sched_pd.build_args(b["q"], b["k_pool"], v, b["block_table"], b["ctx_lens"], out=out,
                               v_layout=layout)
    assert sched_pd.kernel_kind(args) == "mfma"
    assert sched_pd.prefetch_range(args) == (0, 0)
    sched_pd.launch(args)
    torch.cuda.synchronize()
    ref = np.asarray(oracle.decode(b["q"], b["k_pool"], v, b["block_table"], b["ctx_lens"],
                                   v_layout=layout), np.float64)
    got = out.cpu().double().numpy()
    assert np.isnan(got[-1]).all()                  # an empty context: 0/0
    err = np.linalg.norm(got[:-1] - ref[:-1], axis=-1) / np.linalg.norm(ref[:-1], axis=-1)
    assert err.max() <= 4e-6, err.max()


@pytest.mark.parametrize("kv", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", ["tokmajor", "dmajor"])
@pytest.mark.parametrize("ps", [16, 64])
@pytest.mark.parametrize("shed", [False, True])
def test_d64_reads_nothing_from_masked_slots(kv, layout, ps, shed):
    """A pool the caller never cleared: NaN and infinities past every context
    (and past every shed budget, whose pages are loaded and masked) leave the
    output of a zeroed one, bit for bit."""
    hkv, G = 2, 4
    b = workloads.make_batch(np.asarray(CTX), num_q_heads=G * hkv, num_kv_heads=hkv, head_dim=64,
                             page_size=ps, kv_dtype=kv, q_dtype=kv, seed=ps, device="cuda")
    ctx = np.asarray(CTX)
    seen = np.maximum(1, ctx // 2 + 1) if shed else ctx
    kw = {}
    if shed:
        plane = SchedPlane(max_tasks=ctx.size * hkv)
        plane.set_rows(tau=np.repeat(seen, hkv), n=ctx.size * hkv)
        plane.push()
        kw["plane"] = plane
    live = torch.zeros(b["k_pool"].shape[0], ps, dtype=torch.bool, device="cuda")
    bt = b["block_table"].cpu().numpy()
    for r, n in enumerate(np.minimum(ctx, seen)):
        for p in range(-(-int(n) // ps)):
            live[int(bt[r, p]), :min(ps, int(n) - p * ps)] = True
    outs = []
    for bad in (0.0, float("nan"), float("inf")):
        k = torch.where(live[:, None, :, None], b["k_pool"], bad)
        v = torch.where(live[:, None, None, :], b["v_pool"], bad)
        if layout == "tokmajor":
            v = v.permute(0, 1, 3, 2).contiguous()
        out = torch.full((len(CTX), G * hkv, 64), 7.0, device="cuda")
        args = sched_pd.build_args(b["q"], k, v, b["block_table"], b["ctx_lens"], out=out,
                                   v_layout=layout, **kw)
        assert sched_pd.kernel_kind(args) == "mfma"
        sched_pd.launch(args)
        torch.cuda.synchronize()
        outs.append(out[:-1].cpu())              # the last context is empty: 0/0
    assert outs[0].isfinite().all()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("kv", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", ["tokmajor", "dmajor"])
def test_d64_keeps_the_tail_of_a_peaked_row(kv, layout):
    """A token in each of the first four pages (one for each wave of a task)
    scores 18 above 4093 others, whose p = e^-18 = 2^-26 is far below a 16-bit
    float's smallest step and whose V is 256 times larger: an output that drops
    them is 0.4% off."""
    n, ps = 4097, 16
    b = workloads.make_batch(np.asarray([n]), num_q_heads=4, num_kv_heads=1, head_dim=64,
                             page_size=ps, kv_dtype=kv, q_dtype=kv, seed=3, device="cuda")
    q, k = torch.zeros_like(b["q"]), torch.zeros_like(b["k_pool"])
    v = torch.full_like(b["v_pool"], 256.0)
    first = b["block_table"][0, :4].long()
    q[..., 0] = 12.0                             # 12 * 12 / sqrt(64) = 18
    k[first, 0, 0, 0] = 12.0
    v[first, 0, :, 0] = 1.0
    if layout == "tokmajor":
        v = v.permute(0, 1, 3, 2).contiguous()
    out = torch.empty(1, 4, 64, device="cuda")
    args = sched_pd.build_args(q, k, v, b["block_table"], b["ctx_lens"], out=out, v_layout=layout)
    assert sched_pd.kernel_kind(args) == "mfma"
    sched_pd.launch(args)
    p = np.exp(-18.0)
    want = (4.0 + 4093 * p * 256.0) / (4.0 + 4093 * p)
    # a wave's fp32 sum adds 1024 tokens, fp32 MFMAs one at a time, and each add
    # of this input may round by 2^-24 the same way: 6.1e-5
    err = (out.double() / want - 1.0).abs().max().item()
    assert err <= 6.1e-5
