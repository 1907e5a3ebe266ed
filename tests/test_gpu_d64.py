"""Head dim 64 on the MFMA kernel: 16-bit caches, both V layouts, pages of one
and of several 16-token blocks, groups at the edges of its q-head blocks,
context lengths around page, block and wave boundaries. The fp32 output
carries no rounding of its own, so the bound is the arithmetic's: p in full
(24 bits in bf16 parts, 22 in fp16 ones) and fp32 sums of up to 3000 terms,
a few 1e-7 of the row."""
import numpy as np
import pytest
import torch

import oracle
import sched_pd
import workloads

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
