"""Launches without lever tables run the MFMA kernel's lever-free form (three
waves per SIMD, K lines read whole): the same bits as the lever form, which a
launch with a timer row runs, and the oracle's values within 16-bit output
rounding (2^-8 of a row's largest element). Contexts at page, block, wave and
ring boundaries and on both sides of the long-item line (256 pages)."""
import numpy as np
import pytest
import torch

import oracle
import sched_abi as abi
import sched_pd
import workloads
from sched_rt import SchedPlane

pytestmark = pytest.mark.gpu

CTX = [1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 257, 1000, 4096, 4097, 4500]


@pytest.mark.parametrize("kv,q", [(torch.bfloat16, torch.bfloat16),
                                  (torch.float16, torch.float16),
                                  (torch.float8_e4m3fn, torch.bfloat16)])
@pytest.mark.parametrize("layout", ["tokmajor", "dmajor"])
@pytest.mark.parametrize("ps", [16, 64])
@pytest.mark.parametrize("form", ["softmax", "linear", "tiles"])
def test_stock_and_lever_forms_agree(schedlib, kv, q, layout, ps, form):
    if form == "linear" and kv == torch.float16:
        pytest.skip("no MFMA linear mode over fp16")
    hkv, G, d = 2, 5, 128
    b = workloads.make_batch(np.asarray(CTX), num_q_heads=G * hkv, num_kv_heads=hkv, head_dim=d,
                             page_size=ps, kv_dtype=kv, q_dtype=q, seed=ps, device="cuda")
    v = b["v_pool"]
    if layout == "tokmajor":
        v = v.permute(0, 1, 3, 2).contiguous()
    kw = dict(v_layout=layout, k_scale=b.get("k_scale"), v_scale=b.get("v_scale"))
    rows = G * hkv
    if form == "linear":
        g = torch.Generator(device="cuda").manual_seed(ps)
        kw.update(mode=abi.LINEAR, lin_w=torch.rand(max(CTX), device="cuda", generator=g))
        rows = hkv
    if form == "tiles":
        tp = 256 // ps
        kw.update(tiles=sched_pd.plan_tiles_host(np.asarray(CTX), ps, tp, hkv), tile_pages=tp)
    outs = []
    for plane in (None, SchedPlane(max_tasks=len(CTX) * hkv)):
        out = torch.full((len(CTX), rows, d), 7.0, device="cuda")
        a = sched_pd.build_args(b["q"], b["k_pool"], v, b["block_table"], b["ctx_lens"], out=out,
                                plane=plane, **kw)
        assert sched_pd.kernel_kind(a) == "mfma"
        sched_pd.launch(a)
        torch.cuda.synchronize()
        outs.append(out.cpu())
    assert torch.equal(outs[0], outs[1])
    for k in ("tiles", "tile_pages"):
        kw.pop(k, None)
    ref = np.asarray(oracle.decode(b["q"], b["k_pool"], v, b["block_table"], b["ctx_lens"], **kw),
                     np.float64)
    err = np.abs(outs[0].double().numpy() - ref).max(-1) / np.abs(ref).max(-1)
    assert err.max() <= 2 ** -8, err.max()


@pytest.mark.parametrize("ctx", [CTX * 10, [c for c in CTX if c <= 1024], [1024] * 3, [1025] * 3])
def test_fp8_token_major_forms_agree(schedlib, ctx):
    """fp8 token-major V of 16-token pages runs the lever-free form once there
    are more than 256 items, or none longer than 64 pages: on both sides of both
    lines the lever form's bits and the oracle's values."""
    b = workloads.make_batch(np.asarray(ctx), num_q_heads=10, num_kv_heads=2, head_dim=128,
                             page_size=16, kv_dtype=torch.float8_e4m3fn, q_dtype=torch.bfloat16,
                             seed=7, device="cuda")
    v = b["v_pool"].permute(0, 1, 3, 2).contiguous()
    kw = dict(v_layout="tokmajor", k_scale=b.get("k_scale"), v_scale=b.get("v_scale"))
    outs = []
    for plane in (None, SchedPlane(max_tasks=len(ctx) * 2)):
        out = torch.full((len(ctx), 10, 128), 7.0, device="cuda")
        sched_pd.launch(sched_pd.build_args(b["q"], b["k_pool"], v, b["block_table"],
                                            b["ctx_lens"], out=out, plane=plane, **kw))
        torch.cuda.synchronize()
        outs.append(out.cpu())
    assert torch.equal(outs[0], outs[1])
    ref = np.asarray(oracle.decode(b["q"], b["k_pool"], v, b["block_table"], b["ctx_lens"], **kw),
                     np.float64)
    err = np.abs(outs[0].double().numpy() - ref).max(-1) / np.abs(ref).max(-1)
    assert err.max() <= 2 ** -8, err.max()


@pytest.mark.parametrize("kv,q,d", [(torch.bfloat16, torch.bfloat16, 128),
                                    (torch.float16, torch.float16, 64),
                                    (torch.float8_e4m3fn, torch.bfloat16, 128),
                                    (torch.float32, torch.float32, 64)])
def test_occupancy_is_the_lever_forms_before_any_table_is_armed(schedlib, kv, q, d):
    """A queue's worker count is asked of arguments that name no tables yet."""
    b = workloads.make_batch(np.asarray(CTX), num_q_heads=8, num_kv_heads=2, head_dim=d,
                             page_size=16, kv_dtype=kv, q_dtype=q, seed=1, device="cuda")
    got = []
    for plane in (None, SchedPlane(max_tasks=len(CTX) * 2)):
        out = torch.empty(len(CTX), 8, d, device="cuda")
        got.append(sched_pd.occupancy(sched_pd.build_args(
            b["q"], b["k_pool"], b["v_pool"], b["block_table"], b["ctx_lens"], out=out,
            plane=plane, k_scale=b.get("k_scale"), v_scale=b.get("v_scale"))))
    assert got[0] == got[1] > 0
