"""Launches without a plan whose tasks the library cuts on the device
(sched_paged_decode_auto_split): contexts at chunk boundaries, empty ones and
ones far past the mean, on the three kernels, against the oracle; and the same
bits under pi, the queue, the timer, a shed budget loaded or skipped, a CSR
page table and graph replays. Bounds: an output rounded to 16 bits moves by
2^-9 of itself (bf16 p in two halves adds 2^-16), an fp32 one carries the fp32
sums of up to 4097 terms, a few 1e-7 of the row; fp16 p rounds at 2^-12, so its
row norm moves by at most that; the linear mode's weights carry 16 bits."""
import numpy as np
import pytest
import torch

import oracle
import sched_abi as abi
import sched_pd
import workloads
from sched_rt import SchedPlane

pytestmark = pytest.mark.gpu

CTX = [4097, 1, 511, 512, 513, 0, 2048, 64, 65, 3000]

KINDS = {
    # name: kv, q, layout, page, hq, hkv, d, linear, kernel, tolerance
    "bf16": (torch.bfloat16, torch.bfloat16, "tokmajor", 16, 10, 2, 128, False, "mfma", 2e-5),
    "bf16_blocks": (torch.bfloat16, torch.bfloat16, "dmajor", 64, 4, 2, 128, False, "mfma", 2e-5),
    "fp8": (torch.float8_e4m3fn, torch.bfloat16, "dmajor", 16, 7, 1, 128, False, "mfma", 2e-5),
    "fp16": (torch.float16, torch.float16, "tokmajor", 32, 8, 1, 128, False, "mfma", 2.5e-4),
    "d64": (torch.bfloat16, torch.bfloat16, "tokmajor", 16, 8, 2, 64, False, "mfma", 4e-6),
    "linear": (torch.bfloat16, torch.bfloat16, "dmajor", 16, 2, 2, 128, True, "mfma", 2e-5),
    "wave": (torch.float32, torch.float32, "tokmajor", 16, 2, 2, 64, False, "wave", 4e-6),
    "wave_page48": (torch.bfloat16, torch.bfloat16, "tokmajor", 48, 4, 2, 128, False, "wave",
                    4e-6),
    "valu": (torch.float32, torch.float32, "dmajor", 16, 4, 2, 64, False, "valu", 4e-6),
}


def make(kind):
    kv, q, layout, ps, hq, hkv, d, linear, kernel, tol = KINDS[kind]
    b = workloads.make_batch(np.asarray(CTX), num_q_heads=hq, num_kv_heads=hkv, head_dim=d,
                             page_size=ps, kv_dtype=kv, q_dtype=q, seed=ps + d, device="cuda")
    v = b["v_pool"]
    if layout == "tokmajor":
        v = v.permute(0, 1, 3, 2).contiguous()
    kw = dict(v_layout=layout, k_scale=b.get("k_scale"), v_scale=b.get("v_scale"))
    if linear:
        g = torch.Generator(device="cuda").manual_seed(ps)
        kw.update(mode=abi.LINEAR, lin_w=torch.rand(max(CTX), device="cuda", generator=g))
    pos = (b["q"], b["k_pool"], v, b["block_table"], b["ctx_lens"])
    a = sched_pd.build_args(*pos, out=torch.empty(len(CTX), hkv if linear else hq, d,
                                                  device="cuda"), **kw)
    assert sched_pd.kernel_kind(a) == kernel
    need = abi.load_library().sched_paged_decode_auto_split(a, b["block_table"].shape[1], 0)
    assert need > 0 and a.num_tiles >= 2 * len(CTX) * hkv      # this shape is split
    return pos, kw, hkv, tol


def run(pos, kw, **more):
    out = sched_pd.paged_decode(*pos, out_dtype=torch.float32, **kw, **more)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("kind", list(KINDS))
def test_matches_the_oracle_under_every_lever(schedlib, kind):
    pos, kw, hkv, tol = make(kind)
    base = run(pos, kw)
    ref = np.asarray(oracle.decode(*pos, **kw), np.float64)
    live = np.asarray(CTX) > 0
    got = base.cpu().double().numpy()
    err = np.linalg.norm(got - ref, axis=-1)[live] / np.linalg.norm(ref, axis=-1)[live]
    assert err.max() <= tol, err.max()
    if kw.get("mode") != abi.LINEAR:
        assert np.isnan(got[~live]).all()
    n = len(CTX) * hkv
    order = np.random.default_rng(3).permutation(n)
    for workers in (0, 3, 64):
        plane = SchedPlane(max_tasks=n)
        plane.install_order(torch.from_numpy(order.astype(np.int32)), n)
        plane.set_num_tasks(n)
        plane.push()
        for _ in range(2):          # the ticket counter is left for the next launch
            got = run(pos, kw, plane=plane, workers=workers)
            assert torch.equal(got.nan_to_num(9.0), base.nan_to_num(9.0)), workers


@pytest.mark.parametrize("kind", list(KINDS))
def test_shed_budgets_loaded_or_skipped(schedlib, kind):
    pos, kw, hkv, tol = make(kind)
    n = len(CTX) * hkv
    tau = np.minimum(np.random.default_rng(5).integers(1, 4097, n), 65535)
    outs = []
    for flags in (0, abi.FLAG_SHED_LOADS):
        plane = SchedPlane(max_tasks=n)
        plane.set_rows(tau=tau, n=n)
        plane.push()
        outs.append(run(pos, kw, plane=plane, flags=flags).nan_to_num(9.0))
    assert torch.equal(outs[0], outs[1])
    live = np.asarray(CTX) > 0
    ref = np.asarray(oracle.decode(*pos, ctrl=bytes(plane._ctrl_host), max_tasks=n, **kw),
                     np.float64)[live]
    got = outs[0].cpu().double().numpy()[live]
    err = np.linalg.norm(got - ref, axis=-1) / np.linalg.norm(ref, axis=-1)
    assert err.max() <= tol, err.max()
    assert not torch.equal(outs[0], run(pos, kw).nan_to_num(9.0))


@pytest.mark.parametrize("kind", ["bf16", "wave", "valu"])
def test_an_order_naming_a_task_twice_leaves_nothing_behind(schedlib, kind):
    """A permitted order (an entry out of range falls back to its own position)
    that runs a task twice and another not at all: the launch's other rows are
    the plain ones, its workspace's arrival words end at zero, and the plain
    launches after it, of other queries and of shorter contexts (fewer chunks),
    equal the oracle."""
    pos, kw, hkv, tol = make(kind)
    base = run(pos, kw).nan_to_num(9.0)
    n, rows = len(CTX) * hkv, base.shape[1] // hkv
    order = np.arange(n, dtype=np.int32)
    order[1] = 0                    # task 0 (4097 tokens) twice, task 1 never
    order[-1] = n + 7               # falls back to its position
    for workers in (0, 3):
        plane = SchedPlane(max_tasks=n)
        plane.install_order(torch.from_numpy(order), 0)
        plane.set_num_tasks(n)
        plane.push()
        out = torch.full_like(base, 5.0)
        sched_pd.paged_decode(*pos, out=out, plane=plane, workers=workers, **kw)
        torch.cuda.synchronize()
        out = out.nan_to_num(9.0).view(n, rows, -1)
        want = base.view(n, rows, -1).clone()
        want[1] = 5.0
        assert torch.equal(out, want), workers
        for ws, zeroed in sched_pd._SPLIT_WS.streams.values():
            words = ws[sched_pd.WS_COUNTERS_OFF:sched_pd.WS_COUNTERS_OFF + 4 * n]
            assert not words.any(), workers
        for shorter in (0, 2000, 3400):
            ctx = torch.clamp(pos[4] - shorter, min=1).int()
            q = torch.randn(pos[0].shape, device="cuda",
                            generator=torch.Generator(device="cuda").manual_seed(shorter))
            again = (q.to(pos[0].dtype), *pos[1:4], ctx)
            got = torch.full_like(base, 5.0)
            sched_pd.paged_decode(*again, out=got, **kw)
            torch.cuda.synchronize()
            got = got.cpu().double().numpy()
            ref = np.asarray(oracle.decode(*again, **kw), np.float64)
            err = np.linalg.norm(got - ref, axis=-1) / np.linalg.norm(ref, axis=-1)
            assert err.max() <= tol, (workers, shorter, err.max())


@pytest.mark.parametrize("kind", ["bf16", "fp8", "wave", "valu"])
def test_a_wider_table_leaves_the_bits(schedlib, kind):
    pos, kw, hkv, _ = make(kind)
    base = run(pos, kw).nan_to_num(9.0)
    for times in (4, 16):
        wide = torch.zeros(len(CTX), pos[3].shape[1] * times, dtype=torch.int32, device="cuda")
        wide[:, :pos[3].shape[1]] = pos[3]
        assert torch.equal(run((*pos[:3], wide, pos[4]), kw).nan_to_num(9.0), base), times


def test_csr_table_and_graph_replays(schedlib):
    pos, kw, hkv, tol = make("bf16")
    base = run(pos, kw).nan_to_num(9.0)
    ps = pos[1].shape[2]
    npg = -(-np.asarray(CTX) // ps)
    bt = pos[3].cpu().numpy()
    ids = np.concatenate([bt[r, :k] for r, k in enumerate(npg)]).astype(np.int32)
    ind = np.concatenate([[0], np.cumsum(npg)]).astype(np.int32)
    csr = run((*pos[:3], torch.from_numpy(ids).cuda(), pos[4]), kw,
              page_indptr=torch.from_numpy(ind).cuda()).nan_to_num(9.0)
    # the known mean may set another chunk size: equal values, not bits
    assert ((csr - base).norm(dim=-1) <= 2 * tol * base.norm(dim=-1)).all()
    out = torch.empty_like(base)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        sched_pd.paged_decode(*pos, out=out, **kw)
    for _ in range(4):
        out.fill_(3.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.nan_to_num(9.0), base)
        assert torch.equal(run(pos, kw).nan_to_num(9.0), base)


def test_raw_stream_capture_holds_no_freed_memory(schedlib):
    """A capture that torch does not manage keeps no pool for what is allocated
    under it: such a launch is captured whole, with no workspace (one node, the
    decode's), and its replays leave tensors allocated later alone."""
    import ctypes
    hip = ctypes.CDLL("libamdhip64.so")
    pos, kw, hkv, tol = make("bf16")
    base = run(pos, kw).nan_to_num(9.0)
    out = torch.empty_like(base)
    side = torch.cuda.Stream()
    graph, exe, nodes = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_size_t()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        h = ctypes.c_void_p(side.cuda_stream)
        assert hip.hipStreamBeginCapture(h, 1) == 0         # thread-local mode
        sched_pd.paged_decode(*pos, out=out, **kw)
        assert hip.hipStreamEndCapture(h, ctypes.byref(graph)) == 0
        assert hip.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0
        assert nodes.value == 1
        assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None,
                                       ctypes.c_size_t(0)) == 0
        fillers = [torch.full((1 << 18,), 3, dtype=torch.uint8, device="cuda") for _ in range(64)]
        for _ in range(3):
            out.fill_(7.0)
            assert hip.hipGraphLaunch(exe, h) == 0
            side.synchronize()
            got = out.nan_to_num(9.0)
            assert ((got - base).norm(dim=-1) <= 2 * tol * base.norm(dim=-1)).all()
        assert all((f == 3).all().item() for f in fillers)
        assert hip.hipGraphExecDestroy(exe) == 0 and hip.hipGraphDestroy(graph) == 0


def test_threads_on_one_stream(schedlib):
    """Launches of several threads' shapes interleave on the default stream: each
    thread's workspace keeps its counters."""
    import threading
    cases = [make(k)[:2] for k in ("bf16", "wave", "valu")]
    want = [run(pos, kw).nan_to_num(9.0) for pos, kw in cases]
    bad = []

    def work(i):
        pos, kw = cases[i]
        for _ in range(60):
            out = sched_pd.paged_decode(*pos, out_dtype=torch.float32, **kw)
            if not torch.equal(out.nan_to_num(9.0), want[i]):
                bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
