"""Benchmark of the CSR message-passing hot path on one MI355X.

Default workload (the headline metric): GAT additive
edge attention, fp32, 1,000,000 nodes, in-degree ~ Poisson(16) + one
self-loop per row, h [N, 8, 32], forward + backward (dh, da_src, da_dst).
A step = one forward + one backward over the whole graph, inputs resident in
HBM.  Prints ONE JSON line (rank 0): edges/s, ms/step, the dominant kernel's
roofline (algorithmic bytes / its live HIP-event duration) and the
reference's CPU path timed on a bounded sample of the same workload.

  python bench.py [--steps K] [--warmup W]
                  [--config all|c1..c5|dense|dense-causal|dense-pruned|nn|refcases]
                  [--no-cpu] [--no-cold] [--no-graph]

By default (--config all) the line is C2's and carries C1, C3, C4 and C5 as
sub-lines under "configs" (step time, throughput, per-kernel averages, the
roofline of each one's dominant kernel and its CPU baseline), all measured in
this run, plus one summary each of the other shapes.  The line is kept to a
few KB; --detail PATH writes the full record (per-kernel tables, every case).
c1-c5 are BASELINE.json's configurations; dense* are the reference's dense
attention benchmark shapes (N=4096, H=16, D=64, fp16, forward); nn is the
reference's nn-scored GAT training step (131072 nodes, net 19-16-1);
refcases are the reference's archived sum and segmented-softmax GPU cases
(131072 nodes), each beside the figure the reference publishes for it.
"""

from __future__ import annotations

import argparse
import json
import os
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
for p in (str(ROOT / "tiga-lang_amd"), str(ROOT)):
    if p not in sys.path:
        sys.path.insert(0, p)

HBM_PEAK_GBS = 8000.0
BF16_PEAK_TFLOPS = 2500.0   # MI355X dense bf16 (and fp16) MFMA


def measured_traffic(config, kernel):
    """L2-to-memory bytes per step of `kernel` (or the sum over a
    "+"-joined list of kernels that run once per step each) measured by
    rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE (scaled by the copy calibration)
    and recorded in profiles/traffic.json; None when any is unrecorded.
    These are L2-miss bytes: they include Infinity-Cache (MALL) hits, so
    they bound HBM traffic from above rather than equal it."""
    path = ROOT / "profiles" / "traffic.json"
    try:
        table = json.loads(path.read_text())[config]
        recs = [table[k] for k in kernel.split("+")]
    except (OSError, KeyError, ValueError):
        return None, None
    return sum(r["fetch_bytes"] + r["write_bytes"] for r in recs), recs[0]["source"]


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--config", default="all",
                    choices=["all", "c1", "c2", "c3", "c4", "c5", "dense", "dense-causal",
                             "dense-pruned", "nn", "refcases"],
                    help="all (default): C2 as the headline line with C1, C3, C4, C5, "
                         "nn and the dense attention shapes under its 'configs' key")
    ap.add_argument("--nodes", type=int, default=None, help="override node count (testing)")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--no-graph", action="store_true",
                    help="skip the HIP-graph replay measurement (c1, c2)")
    ap.add_argument("--no-cold", action="store_true",
                    help="skip the cold-cache samples (kernel traces then hold only the "
                         "warmup and timed launches)")
    ap.add_argument("--cpu-rows", type=int, default=None)
    ap.add_argument("--seed", type=int, default=20260821)
    ap.add_argument("--detail", default=None, metavar="PATH",
                    help="also write the full record (per-kernel tables, every case) as JSON "
                         "to PATH; stdout keeps the compact line")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="run only a 1 GiB device copy (PMC byte-counter calibration)")
    return ap.parse_args()


def calibrate_copy():
    """A plain copy of known size: reads and writes exactly 1 GiB.  Run under
    rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE, it gives the factor between the
    counters and real bytes."""
    import torch

    n = (1 << 30) // 4
    x = torch.randn(n, device="cuda")
    y = torch.empty_like(x)
    for _ in range(3):
        y.copy_(x)
    torch.cuda.synchronize()
    print(json.dumps({"calibration": "copy", "bytes_read": 4 * n, "bytes_written": 4 * n}))


# ---------------------------------------------------------------------------
# Synthetic inputs (seeded, generated on the GPU)

def poisson_self_loop_csr(n, mean, seed, device):
    """Uniform-random sources, in-degree ~ Poisson(mean), plus a self-loop per
    row; neighbour lists sorted.  int64 row_ptr/col (as the reference's graphs)."""
    import torch

    g = torch.Generator(device=device).manual_seed(seed)
    deg = torch.poisson(torch.full((n,), float(mean), device=device), generator=g).to(torch.int64)
    e_rand = int(deg.sum().item())
    rows = torch.repeat_interleave(torch.arange(n, device=device), deg)
    cols = torch.randint(0, n, (e_rand,), device=device, generator=g)
    ar = torch.arange(n, device=device)
    keys = torch.cat([rows * n + cols, ar * n + ar])
    keys, _ = torch.sort(keys)
    col = keys % n
    row_ptr = torch.zeros(n + 1, dtype=torch.int64, device=device)
    row_ptr[1:] = torch.cumsum(deg + 1, 0)
    return row_ptr, col


def fixed_degree_csr(n_dst, n_src, degree, seed, device):
    """Each row gets exactly `degree` sources drawn with replacement, sorted."""
    import torch

    g = torch.Generator(device=device).manual_seed(seed)
    col = torch.randint(0, n_src, (n_dst, degree), device=device, generator=g)
    col, _ = torch.sort(col, dim=1)
    row_ptr = torch.arange(n_dst + 1, dtype=torch.int64, device=device) * degree
    return row_ptr, col.reshape(-1)


def rmat_csr(scale, edge_factor, probs, seed, device):
    """R-MAT (Chakrabarti et al. 2004) on the GPU: edge_factor * 2**scale tuples,
    one quadrant draw per level, duplicates removed, first coordinate = the
    destination row; returns an int64 dst-row CSR with sorted columns."""
    import torch

    g = torch.Generator(device=device).manual_seed(seed)
    n = 1 << scale
    m = edge_factor * n
    a, b, c, _ = probs
    row = torch.zeros(m, dtype=torch.int64, device=device)
    col = torch.zeros(m, dtype=torch.int64, device=device)
    for level in range(scale):
        r = torch.rand(m, device=device, generator=g)
        down = r >= a + b
        right = ((r >= a) & (r < a + b)) | (r >= a + b + c)
        row |= down.to(torch.int64) << level
        col |= right.to(torch.int64) << level
    keys = torch.unique(row * n + col)
    row, col = keys // n, keys % n
    row_ptr = torch.zeros(n + 1, dtype=torch.int64, device=device)
    row_ptr[1:] = torch.cumsum(torch.bincount(row, minlength=n), 0)
    return row_ptr, col


# ---------------------------------------------------------------------------
# Algorithmic bytes per launch (no-reuse model: every edge reads its index
# (4 B) and its gathered rows once; every per-node array is read or written
# once per pass).

def gat_kernel_bytes(N, E, H, D):
    """The folded backward the Torch front end runs: the forward also writes
    pos (a row per node); the node pass reads dout, out and pos; the source
    pass gathers dout and the destination node state per edge (no per-edge
    output) and reads its source's sdz_dst; the da pass reads h once."""
    row = H * D * 4
    ns = H * 16
    return {
        "gat_fwd_kernel": E * (4 + row) + N * (4 + 3 * row + ns),
        "gat_delta_kernel": N * (3 * row + 2 * H * 4),
        "gat_bwd_src_kernel": E * (4 + row + ns) + N * (4 + 2 * row + 2 * H * 4),
        "gat_da_nodes_kernel": N * (row + 2 * H * 4),
    }


def dot_kernel_bytes(N, E, H, D):
    """The stored-ds backward the Torch front end runs: the source pass also
    writes each edge's ds (transposed order); the destination pass reads it
    through inv_perm, gathers the k row and writes dbias (C4 has a bias)."""
    row = H * D * 2
    return {
        "dot_fwd_kernel": E * (4 + 2 * row + H * 4) + N * (4 + 2 * row + H * 8),
        "dot_delta_kernel": N * (2 * row + H * 4),
        "dot_bwd_dst_kernel": E * (4 + 4 + row + 2 * H * 4) + N * (4 + row),
        "dot_bwd_src_kernel": E * (4 + 4 + 2 * row + H * 4 + H * 8 + H * 4) + N * (4 + 4 * row),
    }


def sum_kernel_bytes(N_dst, N_src, E, F):
    return {
        "csr_sum_fwd": E * (4 + 4 + F * 4) + N_dst * (4 + F * 4),
        "csr_sum_bwd": E * (4 + 4 + 4 + F * 4 + 4) + N_src * (4 + 2 * F * 4),
    }


# ---------------------------------------------------------------------------

def cpu_cores():
    try:
        return len(os.sched_getaffinity(0))
    except AttributeError:
        return os.cpu_count() or 1


def cpu_baseline_gat(row_ptr, col, h, a_src, a_dst, slope, rows):
    """The reference's eager Torch CPU path on the first `rows` destination
    rows (their edges gather from the full source table)."""
    import torch

    from oracle import eager_torch

    threads = cpu_cores()
    torch.set_num_threads(threads)
    rp = row_ptr[: rows + 1].cpu()
    e = int(rp[-1])
    c = col[:e].cpu()
    hc = h.detach().cpu()
    dout = torch.randn(rows, *h.shape[1:], generator=torch.Generator().manual_seed(1))
    eager_torch.gat_step(rp, c, hc, a_src.detach().cpu(), a_dst.detach().cpu(), slope, dout)
    reps, t = 0, 0.0
    while reps < 3 and (reps == 0 or t < 10.0):
        t0 = time.perf_counter()
        eager_torch.gat_step(rp, c, hc, a_src.detach().cpu(), a_dst.detach().cpu(), slope, dout)
        t += time.perf_counter() - t0
        reps += 1
    return {"value": e * reps / t, "unit": "edges/s", "cores": threads, "kind": "port",
            "sample": f"reference eager Torch CPU path (gather, scatter_reduce amax, exp, "
                      f"index_add, autograd), fwd+bwd on the first {rows} destination rows "
                      f"({e} edges) gathering from the full 1M-node table, {reps} reps"}


def timed_steps(step, steps):
    """(seconds for `steps` steps, per-kernel totals).  The steps are timed
    twice, back to back: first as they run for a user, bracketed by device
    synchronisations (this gives `value` and `ms_per_step`); then again with
    the library's HIP-event timer around every launch (tgx_profile_*), whose
    per-kernel averages give the roofline.  The events cost host time per
    launch (about 10 us each), which would inflate host-bound steps like C1's
    if both came from one region; the kernels' own durations do not change."""
    import torch

    from tiga import _native

    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        step()
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    with _native.KernelTimer() as timer:
        t1 = time.perf_counter()
        for _ in range(steps):
            step()
        torch.cuda.synchronize()
        profiled = time.perf_counter() - t1
    return elapsed, profiled, dict(timer.totals)


def cold_step_ms(step, samples=5):
    """Median step time with L2 and the 256 MB MALL flushed before each
    sample (a 1 GiB fill), HIP events on Torch's current stream, which is
    where every kernel of the step runs.  None with --no-cold."""
    import torch

    if ARGS.no_cold:
        return None

    flush = torch.empty(1 << 28, dtype=torch.float32, device="cuda")
    times = []
    for _ in range(samples):
        flush.fill_(1.0)
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        step()
        end.record()
        torch.cuda.synchronize()
        times.append(start.elapsed_time(end))
    del flush
    return sorted(times)[len(times) // 2]


def graph_step_ms(leaves, capture_step, replays=20):
    """Mean time of one step replayed from a HIP graph
    (torch.cuda.graph): warm-up on a side stream (per-graph plans and the
    transposed CSR are built there, with their host synchronisations), one
    capture of `capture_step` (forward + backward into the leaves' .grad),
    `replays` timed replays between HIP events on the current stream.  The
    last replay's gradients are checked bit for bit against an eager step.
    Returns None with --no-graph."""
    import torch

    if ARGS.no_graph:
        return None
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            for t in leaves:
                t.grad = None
            capture_step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    for t in leaves:
        t.grad = None
    with torch.cuda.graph(g):
        capture_step()
    g.replay()
    torch.cuda.synchronize()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    start.record()
    for _ in range(replays):
        g.replay()
    end.record()
    torch.cuda.synchronize()
    ms = start.elapsed_time(end) / replays
    got = [t.grad.clone() for t in leaves]
    for t in leaves:
        t.grad = None
    capture_step()
    torch.cuda.synchronize()
    for a, b in zip(got, leaves):
        assert torch.equal(a, b.grad), "graph replay differs from the eager step"
    del g
    return ms


def _timed_reps(fn, budget_s=10.0, max_reps=3):
    fn()
    reps, t = 0, 0.0
    while reps < max_reps and (reps == 0 or t < budget_s):
        t0 = time.perf_counter()
        fn()
        t += time.perf_counter() - t0
        reps += 1
    return reps, t


def cpu_baseline_sum(row_ptr, col, x, w):
    """C1 on the host: the reference's native CPU runtime loop
    (oracle/cpu_native.c, forward; T = min(32, cores) threads as its default
    pool, and T = cores) and the Torch CPU path the reference dispatches for
    Torch tensors (torch.sparse.mm forward + autograd backward), whole graph."""
    import numpy as np
    import torch

    from oracle import eager_torch, native

    threads = cpu_cores()
    torch.set_num_threads(threads)
    rp, c = row_ptr.cpu(), col.cpu()
    xc, wc = x.detach().cpu(), w.detach().cpu().reshape(-1)
    E = c.numel()
    dout = torch.ones(rp.numel() - 1, xc.shape[1])
    reps, t = _timed_reps(lambda: eager_torch.sum_step(rp, c, xc, wc, dout))
    rp_np, c_np, x_np, w_np = rp.numpy(), c.numpy(), xc.numpy(), wc.numpy()
    out = np.empty((rp_np.size - 1, x_np.shape[1]), dtype=np.float32)
    native_fwd = {}
    for t_native in sorted({min(32, threads), threads}):
        r, tn = _timed_reps(lambda: native.csr_sum_fwd(rp_np, c_np, x_np, w_np, t_native, out),
                            budget_s=5.0, max_reps=10)
        native_fwd[f"threads_{t_native}"] = E * r / tn
    # The native runtime's lowered backward costs E * F * (N_dst + N_src)
    # select/scan steps: timed on a small graph of the same shape and
    # extrapolated to the whole graph by that count.
    n_s, deg = 1000, (E + (rp.numel() - 2)) // (rp.numel() - 1)
    g_s = np.random.default_rng(0)
    rp_s = np.arange(n_s + 1, dtype=np.int64) * deg
    c_s = np.sort(g_s.integers(0, n_s, (n_s, deg)), axis=1).reshape(-1)
    F = x_np.shape[1]
    x_s = g_s.standard_normal((n_s, F)).astype(np.float32)
    w_s = g_s.random(c_s.size).astype(np.float32)
    d_s = np.ones((n_s, F), dtype=np.float32)
    t0 = time.perf_counter()
    native.csr_sum_bwd_lowered(rp_s, c_s, x_s, w_s, d_s)
    t_s = time.perf_counter() - t0
    n_full = rp.numel() - 1
    scale = (E * F * 2 * n_full) / (c_s.size * F * 2 * n_s)
    return {"value": E * reps / t, "unit": "edges/s", "cores": threads, "kind": "port",
            "sample": f"whole C1 graph ({E} edges), fwd+bwd, reference's Torch CPU path "
                      f"(torch.sparse.mm + autograd), {reps} reps",
            "native_runtime_fwd_edges_per_s": native_fwd,
            "native_runtime_bwd": {
                "sample": f"the reference runtime's lowered backward (oracle/cpu_native.c) on "
                          f"{n_s} rows x {deg} neighbours, F={F}, 1 thread",
                "sample_seconds": t_s,
                "extrapolated_c1_seconds": t_s * scale,
                "extrapolated_c1_edges_per_s": E / (t_s * scale)}}


def cpu_baseline_dot(row_ptr, col, q, k, v, bias, scale, dout, edges=1_000_000):
    """C3/C4 on the host: the reference's eager Torch CPU path (gather,
    scatter_reduce amax, exp, index_add, autograd) on the leading destination
    rows holding about `edges` edges, gathering from the full tables.
    Returns forward edges/s and backward edges/s (fwd+bwd minus fwd)."""
    import torch

    from oracle import eager_torch

    threads = cpu_cores()
    torch.set_num_threads(threads)
    rpc = row_ptr.cpu()
    rows = max(1, int(torch.searchsorted(rpc, edges, right=True)) - 1)
    rp = rpc[: rows + 1]
    e = int(rp[-1])
    c = col[:e].cpu()
    qc, kc, vc = (t.detach().cpu() for t in (q, k, v))
    bc = bias.detach()[:e].cpu()
    dc = dout[:rows].cpu()
    qs = qc[:rows]
    r_f, t_f = _timed_reps(lambda: eager_torch.dot_step(rp, c, qs, kc, vc, bc, scale))
    r_s, t_s = _timed_reps(lambda: eager_torch.dot_step(rp, c, qs, kc, vc, bc, scale, dc))
    fwd_s, step_s = t_f / r_f, t_s / r_s
    sample = (f"reference eager Torch CPU path, bf16 inputs with fp32 accumulate, on the "
              f"first {rows} destination rows ({e} edges) gathering from the full tables")
    return e / fwd_s, e / max(step_s - fwd_s, 1e-9), threads, sample


def cpu_baseline_varlen(lengths, q, k, v, dout, scale, pairs_target=120_000):
    """C5 on the host: the reference's eager CPU path materializes every
    causal pair (about 400 GB per gathered tensor at C5), so it runs on a
    row chunk of the first sequence's materialized CSR (the last rows, about
    `pairs_target` pairs), fwd + bwd; TFLOP/s uses the same FLOP convention
    as the GPU figure (fwd 4*H*D per pair, bwd 2.5x)."""
    import torch

    from oracle import eager_torch

    threads = cpu_cores()
    torch.set_num_threads(threads)
    L = int(lengths[0])
    H, D = q.shape[1], q.shape[2]
    r1 = L
    r0 = r1
    while r0 > 0 and (r1 * (r1 + 1) - r0 * (r0 + 1)) // 2 < pairs_target:
        r0 -= 1
    deg = torch.arange(r0 + 1, r1 + 1)
    rp = torch.zeros(r1 - r0 + 1, dtype=torch.int64)
    rp[1:] = torch.cumsum(deg, 0)
    c = torch.cat([torch.arange(i + 1) for i in range(r0, r1)])
    pairs = int(rp[-1])
    qc, kc, vc = (t.detach()[:L].cpu() for t in (q, k, v))
    dc = dout[r0:r1].cpu()
    bias = torch.zeros(pairs, H)
    reps, t = _timed_reps(lambda: eager_torch.dot_step(rp, c, qc[r0:r1], kc, vc, bias, scale,
                                                       dc))
    flops = 3.5 * 4.0 * H * D * pairs
    return {"value": flops * reps / t / 1e12, "unit": "TFLOP/s", "cores": threads,
            "kind": "port",
            "sample": f"reference eager Torch CPU path (gathered pairs, scatter softmax, "
                      f"autograd), fwd+bwd on query rows {r0}..{r1 - 1} of sequence 0 "
                      f"(length {L}, {pairs} causal pairs), bf16 inputs, {reps} reps"}


def cpu_baseline_nn(row_ptr, col, x, disp, net, rows):
    """The nn step on the reference's eager Torch CPU path, on the first
    `rows` destination rows gathering from the full node table."""
    import copy

    import torch

    from oracle import eager_torch

    threads = cpu_cores()
    torch.set_num_threads(threads)
    rp = row_ptr[: rows + 1].cpu()
    e = int(rp[-1])
    c = col[:e].cpu()
    xc, dc = x.detach().cpu(), disp.detach()[:e].cpu()
    net_c = copy.deepcopy(net).cpu()
    dout = torch.randn(rows, xc.shape[1], generator=torch.Generator().manual_seed(1))
    reps, t = _timed_reps(lambda: eager_torch.nn_gat_step(rp, c, xc, dc, net_c, dout))
    return {"value": e * reps / t, "unit": "edges/s", "cores": threads, "kind": "port",
            "sample": f"reference eager Torch CPU path (gathered inputs, the same nn.Sequential, "
                      f"scatter softmax, autograd), fwd+bwd on the first {rows} destination rows "
                      f"({e} edges), {reps} reps"}


def run_c2(args):
    import torch
    import torch.nn.functional as F

    import tiga as tg
    from tiga import _native

    dev = torch.device("cuda")
    N = args.nodes or 1_000_000
    H, D, slope = 8, 32, 0.2
    row_ptr, col = poisson_self_loop_csr(N, 16.0, args.seed, dev)
    E = col.numel()
    g = torch.Generator(device=dev).manual_seed(args.seed + 1)
    h = torch.randn(N, H, D, device=dev, generator=g).requires_grad_(True)
    a_src = (0.1 * torch.randn(H, D, device=dev, generator=g)).requires_grad_(True)
    a_dst = (0.1 * torch.randn(H, D, device=dev, generator=g)).requires_grad_(True)
    dout = torch.randn(N, H, D, device=dev, generator=g)
    graph = tg.Graph.from_csr(row_ptr, col, num_src=N)
    tg.config.strict = True

    class GAT(tg.MessagePassing):
        reducer = tg.online_softmax()

        def edge(self, src, dst, edge):
            s = F.leaky_relu((src.h * a_src).sum(-1) + (dst.h * a_dst).sum(-1), slope)
            return self.reducer(s, src.h)

    kernel = GAT()

    def step():
        h.grad = a_src.grad = a_dst.grad = None
        out = kernel(graph=graph, src={"h": h}, dst={"h": h})
        out.backward(dout)

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    assert kernel.last_variant.backend == "hip"
    elapsed, profiled, per_kernel = timed_steps(step, args.steps)
    cold_ms = cold_step_ms(step)
    graph_ms = graph_step_ms(
        [h, a_src, a_dst],
        lambda: kernel(graph=graph, src={"h": h}, dst={"h": h}).backward(dout))
    bytes_per = gat_kernel_bytes(N, E, H, D)
    step_bytes = sum(bytes_per.values())
    dominant = max((k for k in per_kernel if k in bytes_per), key=lambda k: per_kernel[k][1])
    # Per step, as the bytes are: the gather passes of a table this size are two
    # launches, one per half of the heads.
    avg_ms = per_kernel[dominant][1] / args.steps
    achieved = bytes_per[dominant] / (avg_ms * 1e-3) / 1e9
    ms_per_step = elapsed * 1e3 / args.steps
    result = {
        "metric": "edge-attention fwd+bwd edges/s and % of HBM peak, 1M-node deg-16 graph, 1xMI355X",
        "value": E * args.steps / elapsed,
        "unit": "edges/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp32",
        "data": "synthetic (seeded Poisson(16)+self-loop CSR, h~N(0,1), a~N(0,0.1))",
        "config": {"workload": "c2-gat-additive-fwd-bwd", "nodes": N, "edges": E,
                   "heads": H, "head_dim": D, "index_dtype": "int64"},
        "hbm_frac_step": step_bytes / (ms_per_step * 1e-3) / 1e9 / HBM_PEAK_GBS,
        "cold_ms_per_step": cold_ms,
        "graph_ms_per_step": graph_ms,
        "roofline": {"kernel": dominant, "bound": "hbm", "achieved": achieved,
                     "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS,
                     "traffic": measured_traffic("c2", dominant)[0],
                     "traffic_source": measured_traffic("c2", dominant)[1], "avg_ms": avg_ms,
                     "algorithmic_bytes": bytes_per[dominant]},
        "kernels": {k: {"launches": n, "avg_ms": ms / args.steps,
                        "gbs": (bytes_per[k] / (ms / args.steps * 1e-3) / 1e9)
                               if k in bytes_per else None}
                    for k, (n, ms) in sorted(per_kernel.items())},
    }
    result["profiled_ms_per_step"] = profiled * 1e3 / args.steps
    if not args.no_cpu:
        rows = args.cpu_rows or min(N, 65536)
        result["cpu_baseline"] = cpu_baseline_gat(row_ptr, col, h, a_src, a_dst, slope, rows)
    return result


def run_c1(args):
    import torch

    import tiga as tg
    from tiga import _native

    dev = torch.device("cuda")
    N = args.nodes or 100_000
    F_, deg = 64, 16
    row_ptr, col = fixed_degree_csr(N, N, deg, args.seed, dev)
    E = col.numel()
    g = torch.Generator(device=dev).manual_seed(args.seed + 1)
    x = torch.randn(N, F_, device=dev, generator=g).requires_grad_(True)
    w = torch.rand(E, 1, device=dev, generator=g).requires_grad_(True)
    graph = tg.Graph.from_csr(row_ptr, col, num_src=N)
    tg.config.strict = True

    class WeightedSum(tg.MessagePassing):
        reducer = tg.sum()

        def edge(self, src, dst, edge):
            return edge.weight * src.x

    kernel = WeightedSum()

    def step():
        x.grad = w.grad = None
        kernel(graph=graph, src={"x": x}, dst={}, edge={"weight": w}).sum().backward()

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    elapsed, profiled, totals = timed_steps(step, args.steps)
    cold_ms = cold_step_ms(step)
    graph_ms = graph_step_ms(
        [x, w],
        lambda: kernel(graph=graph, src={"x": x}, dst={}, edge={"weight": w}).sum().backward())
    bytes_per = sum_kernel_bytes(N, N, E, F_)
    dominant = max((k for k in totals if k in bytes_per), key=lambda k: totals[k][1])
    n_launch, total_ms = totals[dominant]
    achieved = bytes_per[dominant] / (total_ms / n_launch * 1e-3) / 1e9
    result = {
        "metric": "weighted-sum fwd+bwd edges/s, 100k x deg-16, F=64, 1xMI355X",
        "value": E * args.steps / elapsed, "unit": "edges/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": elapsed * 1e3 / args.steps,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "fp32",
        "data": "synthetic", "config": {"workload": "c1-weighted-sum-fwd-bwd", "nodes": N,
                                        "edges": E, "features": F_},
        "hbm_frac_step": sum(bytes_per.values()) / (elapsed / args.steps) / 1e9 / HBM_PEAK_GBS,
        "cold_ms_per_step": cold_ms,
        "graph_ms_per_step": graph_ms,
        "roofline": {"kernel": dominant, "bound": "hbm", "achieved": achieved,
                     "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS,
                     "traffic": measured_traffic("c1", dominant)[0],
                     "traffic_source": measured_traffic("c1", dominant)[1],
                     "avg_ms": total_ms / n_launch, "algorithmic_bytes": bytes_per[dominant]},
        "kernels": {k: {"launches": n, "avg_ms": ms / n} for k, (n, ms) in totals.items()},
        "profiled_ms_per_step": profiled * 1e3 / args.steps,
    }
    if not args.no_cpu:
        result["cpu_baseline"] = cpu_baseline_sum(row_ptr, col, x, w)
    return result


def run_dot(args, phases=("c3", "c4")):
    """C3: dot-product attention forward, bf16, on R-MAT scale 21; C4: its
    fused backward (transposed CSR built once, untimed).  One graph and one
    set of inputs serve both phases; returns {phase: result line}."""
    import torch

    import tiga as tg
    from tiga import _native

    dev = torch.device("cuda")
    scale_log2 = 21 if args.nodes is None else max(4, int(args.nodes).bit_length() - 1)
    row_ptr, col = rmat_csr(scale_log2, 16, (0.57, 0.19, 0.19, 0.05), args.seed, dev)
    N = row_ptr.numel() - 1
    E = col.numel()
    H, D = 4, 64
    g = torch.Generator(device=dev).manual_seed(args.seed + 1)
    q = torch.randn(N, H, D, device=dev, generator=g).to(torch.bfloat16).requires_grad_(True)
    k = torch.randn(N, H, D, device=dev, generator=g).to(torch.bfloat16).requires_grad_(True)
    v = torch.randn(N, H, D, device=dev, generator=g).to(torch.bfloat16).requires_grad_(True)
    bias = torch.randn(E, H, device=dev, generator=g).requires_grad_(True)
    dout = torch.randn(N, H, D, device=dev, generator=g).to(torch.bfloat16)
    graph = tg.Graph.from_csr(row_ptr, col, num_src=N)
    tg.config.strict = True

    class DotAttention(tg.MessagePassing):
        reducer = tg.online_softmax()

        def edge(self, src, dst, edge, scale):
            return self.reducer((src.k * dst.q).sum(dim=-1) * scale + edge.bias, src.v)

    kernel = DotAttention()

    def fwd():
        return kernel(graph=graph, src={"k": k, "v": v}, dst={"q": q}, edge={"bias": bias},
                      scale=1.0 / 8.0)

    out = fwd()
    out.backward(dout, retain_graph=True)
    graph._transposed()
    setup = setup_times(graph, N)
    deg = (row_ptr[1:] - row_ptr[:-1])
    stats = {"max_in_degree": int(deg.max()), "empty_rows": int((deg == 0).sum())}
    bytes_per = dot_kernel_bytes(N, E, H, D)
    cpu = None
    if not args.no_cpu:
        cpu = cpu_baseline_dot(row_ptr, col, q, k, v, bias, 1.0 / 8.0, dout)

    def forward_step():
        with torch.no_grad():
            fwd()

    def backward_step():
        q.grad = k.grad = v.grad = bias.grad = None
        out.backward(dout, retain_graph=True)

    results = {}
    for phase in phases:
        step = forward_step if phase == "c3" else backward_step
        for _ in range(args.warmup):
            step()
        torch.cuda.synchronize()
        assert kernel.last_variant.backend == "hip"
        elapsed, profiled, totals = timed_steps(step, args.steps)
        cold_ms = cold_step_ms(step)
        names = ["dot_fwd_kernel"] if phase == "c3" else [
            "dot_delta_kernel", "dot_bwd_dst_kernel", "dot_bwd_src_kernel"]
        step_bytes = sum(bytes_per[n] for n in names)
        dominant = max((n for n in names if n in totals), key=lambda n: totals[n][1])
        n_launch, total_ms = totals[dominant]
        avg_ms = total_ms / n_launch
        achieved = bytes_per[dominant] / (avg_ms * 1e-3) / 1e9
        ms = elapsed * 1e3 / args.steps
        what = "forward" if phase == "c3" else "fused backward"
        traffic, source = measured_traffic(phase, dominant)
        result = {
            "metric": f"dot-product edge attention {what} edges/s, R-MAT scale 21, bf16, "
                      "1xMI355X",
            "value": E * args.steps / elapsed, "unit": "edges/s", "n_gpus": 1,
            "steps": args.steps, "warmup": args.warmup, "ms_per_step": ms,
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "bf16",
            "data": "synthetic (seeded R-MAT a=.57 b=.19 c=.19 d=.05, dedup; q,k,v,bias "
                    "~N(0,1))",
            "config": {"workload": f"{phase}-dot-attention-{'fwd' if phase == 'c3' else 'bwd'}",
                       "nodes": N, "edges": E, "heads": H, "head_dim": D, **stats},
            "hbm_frac_step": step_bytes / (ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
            "cold_ms_per_step": cold_ms,
            "roofline": {"kernel": dominant, "bound": "hbm", "achieved": achieved,
                         "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS,
                         "traffic": traffic, "traffic_source": source, "avg_ms": avg_ms,
                         "algorithmic_bytes": bytes_per[dominant]},
            "kernels": {kk: {"launches": n, "avg_ms": t / n,
                             "gbs": (bytes_per[kk] / (t / n * 1e-3) / 1e9)
                             if kk in bytes_per else None}
                        for kk, (n, t) in sorted(totals.items())},
            "profiled_ms_per_step": profiled * 1e3 / args.steps,
            "setup_ms": setup,
        }
        if cpu is not None:
            fwd_rate, bwd_rate, threads, sample = cpu
            result["cpu_baseline"] = {
                "value": fwd_rate if phase == "c3" else bwd_rate, "unit": "edges/s",
                "cores": threads, "kind": "port",
                "sample": sample + (", forward" if phase == "c3" else
                                    ", backward = (fwd+bwd) - fwd")}
        results[phase] = result
    return results


def setup_times(graph, N, reps=3):
    """One-off per-graph work, timed apart from the steps: building the CSR
    from edge lists on the device (this library vs the Torch ops the
    reference's Graph.from_coo runs, interop/torch/graph.py:219-227), the
    stable transpose, and the degree-binned row plan."""
    import torch

    from tiga.graph import build_coo_csr, build_row_plan, build_transpose

    row_ptr, col = graph._kernel_csr()
    dst = graph.destination_index()

    def torch_coo():
        order = torch.argsort(dst, stable=True)
        c = col[order]
        counts = torch.bincount(dst, minlength=N)
        rp = torch.empty(N + 1, dtype=dst.dtype, device=dst.device)
        rp[0] = 0
        torch.cumsum(counts, dim=0, out=rp[1:])
        return rp, c

    def timed(fn):
        fn()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(reps):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) * 1e3 / reps

    rp_n, col_n = build_coo_csr(col, dst, N)
    rp_t, col_t = torch_coo()
    assert torch.equal(rp_n.cpu(), rp_t.cpu()) and torch.equal(col_n.cpu(), col_t.cpu())
    return {"from_coo_device": timed(lambda: build_coo_csr(col, dst, N)),
            "from_coo_torch_ops": timed(torch_coo),
            "transpose": timed(lambda: build_transpose(row_ptr, col, N, N)),
            "row_plan": timed(lambda: build_row_plan(row_ptr, N))}


def run_c5(args):
    """C5: varlen causal attention, 32 sequences of U[512, 4096] tokens,
    H=16, D=128, bf16, forward + backward on MFMA."""
    import numpy as np
    import torch

    import tiga as tg
    from tiga import _native

    dev = torch.device("cuda")
    rng = np.random.default_rng(args.seed)
    lengths = rng.integers(512, 4097, size=32)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lengths)]), dtype=torch.int64, device=dev)
    T, H, D = int(lengths.sum()), 16, 128
    g = torch.Generator(device=dev).manual_seed(args.seed + 1)
    mk = lambda: torch.randn(T, H, D, device=dev, generator=g).to(torch.bfloat16)
    q, k, v = (mk().requires_grad_(True) for _ in range(3))
    dout = mk()
    graph = tg.Graph.cu_seqlens(cu, causal=True)
    tg.config.strict = True

    class VarlenAttention(tg.MessagePassing):
        reducer = tg.online_softmax()

        def edge(self, src, dst, edge, scale):
            return self.reducer((src.key * dst.query).sum(dim=-1) * scale, src.value)

    kernel = VarlenAttention()

    def step():
        q.grad = k.grad = v.grad = None
        out = kernel(graph=graph, src={"key": k, "value": v}, dst={"query": q}, scale=D ** -0.5)
        out.backward(dout)

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    assert kernel.last_variant.backend == "hip"
    elapsed, profiled, totals = timed_steps(step, args.steps)
    cold_ms = cold_step_ms(step)
    pairs = int((lengths * (lengths + 1) // 2).sum())
    fwd_flops = 4.0 * H * D * pairs
    step_flops = 3.5 * fwd_flops              # FA2 convention: bwd = 2.5 x fwd
    ms = elapsed * 1e3 / args.steps
    tflops = step_flops / (ms * 1e-3) / 1e12
    kflops = {"varlen_fwd_kernel": fwd_flops, "varlen_dkdv_kernel": 2.0 * fwd_flops,
              "varlen_dq_kernel": 0.5 * fwd_flops, "varlen_dq_stored_kernel": 0.5 * fwd_flops}
    per = totals
    dominant = max((kk for kk in per if kk in kflops), key=lambda kk: per[kk][1])
    n_launch, total_ms = per[dominant]
    achieved = kflops[dominant] / (total_ms / n_launch * 1e-3) / 1e12
    result = {
        "metric": "varlen causal attention fwd+bwd TFLOP/s, 32 seqs U[512,4096], H=16 D=128, "
                  "bf16, 1xMI355X",
        "value": tflops, "unit": "TFLOP/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": ms, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "bf16",
        "data": "synthetic (seeded lengths, q,k,v,dout ~N(0,1))",
        "config": {"workload": "c5-varlen-causal-fwd-bwd", "tokens": T, "sequences": 32,
                   "heads": H, "head_dim": D, "causal_pairs": pairs,
                   "flop_convention": "fwd 4*H*D*pairs, bwd 2.5x fwd (useful FLOPs: the "
                                      "dK/dV pass computes S, dP, dV and dK and stores dS, "
                                      "the dQ pass reads dS back)"},
        "mfma_utilization": tflops / BF16_PEAK_TFLOPS,
        "cold_ms_per_step": cold_ms,
        "roofline": {"kernel": dominant, "bound": "mfma", "achieved": achieved,
                     "peak": BF16_PEAK_TFLOPS, "unit": "TFLOP/s",
                     "frac": achieved / BF16_PEAK_TFLOPS,
                     "traffic": measured_traffic("c5", dominant)[0],
                     "traffic_source": measured_traffic("c5", dominant)[1],
                     "avg_ms": total_ms / n_launch, "algorithmic_flops": kflops[dominant]},
        "kernels": {kk: {"launches": n, "avg_ms": t / n,
                         "tflops": (kflops[kk] / (t / n * 1e-3) / 1e12) if kk in kflops else None}
                    for kk, (n, t) in sorted(per.items())},
    }
    result["profiled_ms_per_step"] = profiled * 1e3 / args.steps
    if not args.no_cpu:
        result["cpu_baseline"] = cpu_baseline_varlen(lengths, q, k, v, dout, D ** -0.5)
    return result


def run_dense(args):
    """The reference's dense attention benchmark shapes
    (benchmarks/neural_networks/dense_attention.py, sparse_attention.py;
    evidence cases b1_h16_n4096_d64_fp16[_causal]): Graph.dense /
    Graph.triangular with 4096 nodes, 16 heads, head_dim 64, fp16 inputs in
    the lane-major [H, N, D] storage viewed as [N, H, D], forward only; the
    pruned case uses block_prune_threshold = D / N as the reference's."""
    import torch

    import tiga as tg
    from tiga import _native

    dev = torch.device("cuda")
    N, H, D = (args.nodes or 4096), 16, 64
    causal = args.config == "dense-causal"
    prune = args.config == "dense-pruned"
    g = torch.Generator(device=dev).manual_seed(args.seed)
    q, k, v = (torch.randn(H, N, D, device=dev, dtype=torch.float16, generator=g).permute(1, 0, 2)
               for _ in range(3))
    graph = tg.Graph.triangular(N, device=dev) if causal else tg.Graph.dense(N, device=dev)
    tg.config.strict = True

    class Attention(tg.MessagePassing):
        def __init__(self, threshold):
            super().__init__()
            self.reducer = tg.online_softmax(block_prune_threshold=threshold)

        def edge(self, src, dst, edge, scale):
            score = (src.key * dst.query).sum(dim=-1) * scale
            return self.reducer(score, src.value)

    kernel = Attention(D / N if prune else None)

    def step():
        with torch.no_grad():
            return kernel(graph=graph, src={"key": k, "value": v}, dst={"query": q},
                          scale=D ** -0.5)

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    assert kernel.last_variant.backend == "hip"
    elapsed, profiled, totals = timed_steps(step, args.steps)
    pairs = N * (N + 1) // 2 if causal else N * N
    flops = 4.0 * H * D * pairs            # useful: q.k and p.v per pair (pruned: as if dense)
    ms = elapsed * 1e3 / args.steps
    # The forward kernel plus, where the key ranges are split, the merge of
    # its chunks: both run every step, so both count in the roofline's time.
    n_launch, total_ms = totals["varlen_fwd_kernel"]
    roof_kernels = ["varlen_fwd_kernel"]
    if "varlen_fwd_merge_kernel" in totals:
        roof_kernels.append("varlen_fwd_merge_kernel")
        total_ms += totals["varlen_fwd_merge_kernel"][1]
    kernel_ms = total_ms / n_launch
    achieved = flops / (kernel_ms * 1e-3) / 1e12
    what = {"dense": "all pairs", "dense-causal": "lower-triangular",
            "dense-pruned": f"all pairs, block_prune_threshold={D / N:g}"}[args.config]
    return {
        "metric": f"dense attention forward TFLOP/s ({what}), N={N}, H={H}, D={D}, fp16, "
                  "1xMI355X",
        "value": flops / (ms * 1e-3) / 1e12, "unit": "TFLOP/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": ms,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "fp16",
        "data": "synthetic (q,k,v ~N(0,1), lane-major storage)",
        "config": {"workload": args.config, "nodes": N, "heads": H, "head_dim": D,
                   "pairs": pairs, "flop_convention": "4*H*D per pair (the reference counts "
                   "(4D+5) per pair and head)"},
        "roofline": {"kernel": "+".join(roof_kernels), "bound": "mfma", "achieved": achieved,
                     "peak": BF16_PEAK_TFLOPS, "unit": "TFLOP/s",
                     "frac": achieved / BF16_PEAK_TFLOPS,
                     "traffic": measured_traffic(args.config, "+".join(roof_kernels))[0],
                     "traffic_source": measured_traffic(args.config,
                                                        "+".join(roof_kernels))[1],
                     "avg_ms": kernel_ms},
        "kernels": {kk: {"launches": n, "avg_ms": t / n} for kk, (n, t) in totals.items()},
        "profiled_ms_per_step": profiled * 1e3 / args.steps,
        # The reference's own FLOP convention and published time for this
        # case (benchmarks/evidence_snapshot/output/roofline/dense_attention/
        # b1_h16_n4096_d64_fp16[_causal]; its own GPU, not an MI355X).
        "reference_convention_tflops": (4 * D + 5) * H * pairs / (ms * 1e-3) / 1e12,
        "reference_ms_own_gpu": {"dense": 0.772, "dense-causal": 0.4459,
                                 "dense-pruned": 0.907}[args.config],
    }


def run_nn(args):
    """The reference's nn-scored GAT training step (benchmarks/neural_networks/
    gat_attention.py, evidence case cuda_n131072_degree32): 131072 nodes,
    about 4.0M edges, score network Linear(3 + 2*8, 16) -> LeakyReLU(0.2) ->
    Linear(16, 1) over [displacement | x_src | x_dst], value x_src (width 8),
    fp32, forward + backward (gradients of x, the displacement and the
    network).  The reference builds a radius graph (Graph.radius, out of scope
    here); this uses the same node and mean edge count with Poisson(30.6)
    in-degrees and uniformly random sources, and the displacement as an edge
    field."""
    import torch
    from torch import nn

    import tiga as tg
    from tiga import _native

    dev = torch.device("cuda")
    N = args.nodes or 131072
    row_ptr, col = poisson_self_loop_csr(N, 29.6, args.seed, dev)
    E = col.numel()
    g = torch.Generator(device=dev).manual_seed(args.seed + 1)
    pos = torch.rand(N, 3, device=dev, generator=g)
    x = torch.randn(N, 8, device=dev, generator=g).requires_grad_(True)
    graph = tg.Graph.from_csr(row_ptr, col, num_src=N)
    disp = (pos[col] - pos[graph.destination_index()]).requires_grad_(True)
    torch.manual_seed(args.seed)
    attn = nn.Sequential(nn.Linear(19, 16), nn.LeakyReLU(0.2), nn.Linear(16, 1)).to(dev)
    dout = torch.randn(N, 8, device=dev, generator=g)
    tg.config.strict = True

    class GAT(tg.MessagePassing):
        reducer = tg.online_softmax()

        def __init__(self):
            super().__init__()
            self.attn = tg.nn.trace(attn)

        def edge(self, src, dst, edge):
            return self.reducer(self.attn(edge.displacement, src.x, dst.x), src.x)

    kernel = GAT()

    def step():
        x.grad = disp.grad = None
        attn.zero_grad(set_to_none=True)
        kernel(graph=graph, src={"x": x}, dst={"x": x},
               edge={"displacement": disp}).backward(dout)

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    assert kernel.last_variant.backend == "hip"
    elapsed, profiled, totals = timed_steps(step, args.steps)
    ms = elapsed * 1e3 / args.steps
    # Algorithmic bytes per pass (no-reuse model, 4 B indices).  Per edge the
    # score pass reads col, dst, the 19 input floats (displacement 3, x_src 8,
    # x_dst 8) and writes the score; the backward reads the same plus dscore
    # and writes the 19 input-gradient floats (the weight gradients are summed
    # on chip).  The kernels that apply x_dst's columns once per row read and
    # write it per row instead (score pass: its 16 products' row written and
    # read; backward: the row sums of dz, the gradient rows come after it).
    inputs = 4 * (3 + 8 + 8)
    bytes_per = {
        "edge_mlp_fwd_kernel": E * (4 + 4 + inputs + 4),
        "edge_mlp_bwd_kernel": E * (4 + 4 + inputs + 4 + inputs),
        "projected_scores_kernel": E * (4 + 4 + 12 + 32 + 4) + N * 64,
        "projected_bwd_kernel": E * (4 + 4 + 2 * (12 + 32)) + N * (64 + 64 + 4 + 4 + 64),
        "csr_sum_fwd": E * (4 + 4 + 32) + N * (4 + 32),
    }
    per = totals
    dominant = max((k for k in per if k in bytes_per), key=lambda k: per[k][1])
    n_launch, total_ms = per[dominant]
    achieved = bytes_per[dominant] / (total_ms / n_launch * 1e-3) / 1e9
    result = {
        "metric": "nn-scored GAT training step edges/s (score net 19-16-1, value 8, fp32), "
                  "131072 nodes, 1xMI355X",
        "value": E * args.steps / elapsed, "unit": "edges/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": ms,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "fp32",
        "data": "synthetic (Poisson(30.6) in-degree, uniform sources, x ~N(0,1), "
                "displacement from uniform positions)",
        "config": {"workload": "nn-gat-fwd-bwd", "nodes": N, "edges": E, "attn": "19-16-1",
                   "value_width": 8, "reference_ms_own_gpu": 10.97},
        "roofline": {"kernel": dominant, "bound": "hbm", "achieved": achieved,
                     "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS,
                     "traffic": measured_traffic("nn", dominant)[0],
                     "traffic_source": measured_traffic("nn", dominant)[1],
                     "algorithmic_bytes": bytes_per[dominant],
                     "note": "the edge MLP kernels are issue- and latency-bound fp32 work "
                             "(weights in scalar registers) on 32-byte gathered rows, far "
                             "from the HBM roof"},
        "kernels": {k: {"launches": n, "avg_ms": t / n} for k, (n, t) in sorted(per.items())},
    }
    result["profiled_ms_per_step"] = profiled * 1e3 / args.steps
    if not args.no_cpu:
        result["cpu_baseline"] = cpu_baseline_nn(row_ptr, col, x, disp, attn, min(N, 32768))
    return result


def reference_case_graph(nodes, degree, topology, locality, seed, device):
    """The reference's sparse benchmark graphs (benchmarks/sparse_compute/
    cases.py:42-117): "regular" rows of `degree` edges, or "powerlaw" rows of
    degree/2, 4 degree and 16 degree edges with probabilities 0.90, 0.09 and
    0.01; sources "local" (dst + 1 + (edge ordinal mod degree), mod nodes)
    or "random" (uniform).  int64 row_ptr/col.  Torch's generator here is
    not the reference's, so the random draws differ; the shapes do not."""
    import torch

    g = torch.Generator(device=device).manual_seed(seed)
    if topology == "regular":
        deg = torch.full((nodes,), degree, device=device, dtype=torch.int64)
    else:
        u = torch.rand(nodes, device=device, generator=g)
        deg = torch.where(u < 0.90, max(1, degree // 2),
                          torch.where(u < 0.99, 4 * degree, 16 * degree)).to(torch.int64)
    row_ptr = torch.zeros(nodes + 1, dtype=torch.int64, device=device)
    row_ptr[1:] = torch.cumsum(deg, 0)
    E = int(row_ptr[-1].item())
    dst = torch.repeat_interleave(torch.arange(nodes, device=device), deg)
    if locality == "local":
        col = (dst + 1 + torch.arange(E, device=device) % max(1, degree)) % nodes
    else:
        col = torch.randint(nodes, (E,), device=device, generator=g)
    return row_ptr, col, dst


def _event_median_ms(fn, reps=50, warmup=5):
    """Median of `reps` HIP-event samples of fn() on Torch's stream, hot
    cache (the reference's samples_ms protocol, benchmarks/common/
    hardware_roofline.py)."""
    import statistics

    import torch

    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    out = []
    for _ in range(reps):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        fn()
        b.record()
        b.synchronize()
        out.append(a.elapsed_time(b))
    return statistics.median(out)


def run_refcases(args):
    """The reference's own archived GPU benchmark cases for this path, run on
    this build at the same shapes (hot cache, medians of HIP-event samples),
    each beside the reference's published figure.  The reference's numbers
    come from an RTX 5070 Ti (benchmarks/evidence_snapshot/output/roofline/),
    so the ratio compares two machines, not two implementations on one.
    Every case is checked against a Torch computation before it is timed."""
    import torch

    import tiga as tg

    dev = torch.device("cuda")
    tg.config.strict = True
    N = 131072

    class WeightedAggregation(tg.MessagePassing):
        # benchmarks/sparse_compute/weighted_aggregation.py:62-67
        reducer = tg.sum()

        def edge(self, src, dst, edge):
            return edge.weight * src.x

    class SegmentedSoftmax(tg.MessagePassing):
        # benchmarks/neural_networks/online_softmax.py:54-58 (its user-defined
        # stable weighted mean is the online softmax reducer's algebra)
        reducer = tg.online_softmax()

        def edge(self, src, dst, edge):
            return self.reducer(src.score, src.value)

    cases = {}

    def record(name, E, ms, ms_prepared, ref_gedges, ref_ms, source, note):
        # Both ratios are reported: the ordinary call (through autograd for
        # the backward cases) and the prepared launch, where there is one.
        cases[name] = {
            "edges": E, "ms": ms, "ms_prepared": ms_prepared,
            "gedges_per_s": E / (ms * 1e-3) / 1e9,
            "gedges_per_s_prepared": (E / (ms_prepared * 1e-3) / 1e9
                                      if ms_prepared is not None else None),
            "reference_gedges_per_s": ref_gedges, "reference_ms": ref_ms,
            "reference_hardware": "RTX 5070 Ti", "reference_source": source,
            "ratio_call": ref_ms / ms,
            "ratio_prepared": ref_ms / ms_prepared if ms_prepared is not None else None,
            "what": note}

    g = torch.Generator(device=dev).manual_seed(args.seed)
    # Weighted sum forward (weighted_aggregation.py:252-314): x [N, F] (or
    # [N] for F = 1), weight [E, 1] (or [E]), tg.sum() of weight * x.
    for name, F_, topology, locality, ref, ref_ms, src_file in (
            ("sum_fwd_regular_local_i64_f64", 64, "regular", "local", 22.06, 0.0951,
             "weighted_aggregation/regular_local_cuda_i64_n131072_degree16_f1_16_64"),
            ("sum_fwd_regular_local_i64_f1", 1, "regular", "local", 102.5, 0.0205,
             "weighted_aggregation/regular_local_cuda_i64_n131072_degree16_f1_16_64"),
            ("sum_fwd_powerlaw_random_i64_f1", 1, "powerlaw", "random", 38.2, 0.0536,
             "weighted_aggregation/powerlaw_random_cuda_i64_n131072_degree16_f1")):
        row_ptr, col, dst = reference_case_graph(N, 16, topology, locality, 20260807, dev)
        E = col.numel()
        x = torch.rand((N,) if F_ == 1 else (N, F_), device=dev, generator=g)
        w = torch.rand((E,) if F_ == 1 else (E, 1), device=dev, generator=g)
        graph = tg.Graph.from_csr(row_ptr, col, num_src=N)
        kernel = WeightedAggregation()
        call = lambda: kernel(graph=graph, src={"x": x}, dst={"x": x}, edge={"weight": w})
        got = call()
        assert kernel.last_variant.backend == "hip", name
        want = torch.zeros_like(x).index_add_(0, dst, w * x[col])
        torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-4)
        prepared = kernel.prepare(graph=graph, src={"x": x}, dst={"x": x}, edge={"weight": w})
        record(name, E, _event_median_ms(call), _event_median_ms(prepared), ref, ref_ms,
               src_file, f"tg.sum() of edge.weight * src.x, {topology} {locality} rows, F={F_}")
        del graph, kernel, prepared, x, w, row_ptr, col, dst
    # Segmented online softmax forward (online_softmax.py:92-127): 32 random
    # sources per row, scalar score (N(0,1) + 1000) and value per source.
    E = N * 32
    row_ptr = torch.arange(0, E + 1, 32, dtype=torch.int64, device=dev)
    col = torch.randint(N, (E,), dtype=torch.int64, device=dev, generator=g)
    score = torch.randn(N, device=dev, generator=g) + 1000
    value = torch.randn(N, device=dev, generator=g)
    graph = tg.Graph.from_csr(row_ptr, col, num_src=N)
    kernel = SegmentedSoftmax()
    call = lambda: kernel(graph=graph, src={"score": score, "value": value}, dst={})
    got = call()
    assert kernel.last_variant.backend == "hip"
    want = (torch.softmax(score[col].reshape(N, 32), dim=1) * value[col].reshape(N, 32)).sum(1)
    torch.testing.assert_close(got, want, rtol=3e-4, atol=3e-4)
    prepared = kernel.prepare(graph=graph, src={"score": score, "value": value}, dst={})
    record("online_softmax_fwd_random_i64_deg32_f1", E, _event_median_ms(call),
           _event_median_ms(prepared), 25.0, 0.1678,
           "online_softmax/cuda_n131072_degree32_f1",
           "softmax over each row's 32 source scores, weighted sum of the source values")
    del graph, kernel, prepared, score, value, row_ptr, col
    # Sum backward (autograd/message_passing_backward.py:99-160): regular
    # random rows, x and weight N(0,1), a random cotangent; dx alone for
    # F = 1, the per-edge weight gradient alone for F = 64.  The reference
    # times dx as its generated source VJP (compile_source_vjp: the weighted
    # sum of the cotangent over the transposed relation with the weights in
    # transposed edge order), so `ms_prepared` is that sum here, prepared;
    # `ms` is torch.autograd.grad through this build's backward.
    for name, F_, wrt, ref, ref_ms, src_file in (
            ("sum_bwd_dx_regular_random_i64_f1", 1, "x", 35.85, 0.0585,
             "message_passing_backward/regular_random_cuda_i64_n131072_degree16_dx"),
            ("sum_bwd_dweight_regular_random_i64_f64", 64, "weight", 0.91, 2.30,
             "message_passing_backward/regular_random_cuda_i64_n131072_degree16_dweight_f64")):
        row_ptr, col, dst = reference_case_graph(N, 16, "regular", "random", 20260807, dev)
        E = col.numel()
        x = torch.randn((N,) if F_ == 1 else (N, F_), device=dev, generator=g,
                        requires_grad=True)
        w = torch.randn((E,) if F_ == 1 else (E, 1), device=dev, generator=g,
                        requires_grad=True)
        cot = torch.randn((N,) if F_ == 1 else (N, F_), device=dev, generator=g)
        graph = tg.Graph.from_csr(row_ptr, col, num_src=N)
        kernel = WeightedAggregation()
        out = kernel(graph=graph, src={"x": x}, dst={}, edge={"weight": w})
        assert kernel.last_variant.backend == "hip", name
        target = x if wrt == "x" else w
        grad = lambda: torch.autograd.grad(out, target, cot, retain_graph=True)[0]
        got = grad()
        with torch.no_grad():
            if wrt == "x":
                want = torch.zeros_like(x).index_add_(0, col, (w * cot[dst]))
            else:
                want = (cot[dst] * x[col]).sum(1, keepdim=True)
        torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-4)
        ms_vjp = None
        if wrt == "x":
            graph_t = graph.transpose()
            w_t = w.detach()[torch.argsort(col, stable=True)]
            vjp = WeightedAggregation()
            torch.testing.assert_close(
                vjp(graph=graph_t, src={"x": cot}, dst={}, edge={"weight": w_t}), want,
                rtol=1e-4, atol=1e-4)
            ms_vjp = _event_median_ms(
                vjp.prepare(graph=graph_t, src={"x": cot}, dst={}, edge={"weight": w_t}))
            del graph_t, w_t, vjp
        record(name, E, _event_median_ms(grad), ms_vjp, ref, ref_ms, src_file,
               f"torch.autograd.grad of the weighted sum with respect to {wrt} alone, F={F_}"
               + ("; prepared: the sum of the cotangent over the transposed relation"
                  if wrt == "x" else ""))
        del graph, kernel, out, x, w, cot, row_ptr, col, dst
    return {
        "metric": "the reference's archived GPU cases for this path, edges/s on 1xMI355X",
        "unit": "edges/s", "n_gpus": 1, "data": "synthetic (the reference's generators)",
        "config": {"workload": "reference-benchmark-cases", "nodes": N},
        "cases": cases,
    }


def _release_gpu_memory():
    import gc

    import torch

    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()


def run_all(args):
    """Every BASELINE configuration in one process: C2 (the headline) as the
    top-level line, C1, C3, C4 and C5 under "configs", each with its own
    step time, roofline of its dominant kernel and CPU baseline; then the
    reference's own benchmark shapes this path also covers (the nn-scored
    GAT step, with its CPU baseline, the dense / triangular / pruned
    attention forwards, and the reference's archived sum and softmax cases).  Progress goes to stderr; stdout gets the one JSON
    line."""
    t_all = time.perf_counter()

    def progress(name, t0):
        print(f"bench: {name} done in {time.perf_counter() - t0:.1f} s", file=sys.stderr,
              flush=True)

    t0 = time.perf_counter()
    result = run_c2(args)
    progress("c2", t0)
    configs = {}
    for name, fn in (("c1", run_c1), ("c3+c4", lambda a: run_dot(a, ("c3", "c4"))),
                     ("c5", run_c5)):
        _release_gpu_memory()
        t0 = time.perf_counter()
        got = fn(args)
        configs.update(got if name == "c3+c4" else {name: got})
        progress(name, t0)
    for name in ("nn", "dense", "dense-causal", "dense-pruned", "refcases"):
        _release_gpu_memory()
        t0 = time.perf_counter()
        sub_args = argparse.Namespace(**vars(args))
        sub_args.config = name
        runner = {"nn": run_nn, "refcases": run_refcases}.get(name, run_dense)
        configs[name] = runner(sub_args)
        progress(name, t0)
    for sub in configs.values():
        if isinstance(sub.get("cpu_baseline"), dict):
            sub["cpu_baseline"]["cpu_model"] = cpu_model()
    result["configs"] = configs
    result["bench_wall_s"] = time.perf_counter() - t_all
    return result


ARGS = None


def cpu_model():
    """The host CPU's model name (the CPU baselines' hardware)."""
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return None


def measured_roofs(samples=10):
    """In-run roof calibration, as the reference's benchmarks measure theirs
    (benchmarks/common/hardware_roofline.py:102-120): the bytes read plus
    written by a 1 GiB fp32 device copy per second, and a dense bf16 GEMM
    (torch.mm, 8192^3) in FLOP/s; medians of HIP-event samples on Torch's
    stream after warm-up.  Reported beside the published peaks, which stay
    the roofline's denominator."""
    import statistics

    import torch

    def median_ms(fn):
        for _ in range(3):
            fn()
        torch.cuda.synchronize()
        out = []
        for _ in range(samples):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            fn()
            b.record()
            b.synchronize()
            out.append(a.elapsed_time(b))
        return statistics.median(out)

    n = 1 << 28
    src = torch.ones(n, device="cuda")
    dst = torch.empty_like(src)
    copy_gbs = 2 * 4 * n / (median_ms(lambda: dst.copy_(src)) * 1e-3) / 1e9
    del src, dst
    m = 8192
    g = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randn(m, m, device="cuda", generator=g).to(torch.bfloat16)
    y = torch.randn(m, m, device="cuda", generator=g).to(torch.bfloat16)
    z = torch.empty(m, m, device="cuda", dtype=torch.bfloat16)
    gemm_tflops = 2.0 * m ** 3 / (median_ms(lambda: torch.mm(x, y, out=z)) * 1e-3) / 1e12
    del x, y, z
    torch.cuda.empty_cache()
    return {"copy_GBps": copy_gbs, "bf16_gemm_TFLOPs": gemm_tflops,
            "how": "1 GiB fp32 device copy (read + write bytes) and torch.mm bf16 8192^3, "
                   f"median of {samples} HIP-event samples"}


def _sig(x, digits=4):
    """Floats rounded to `digits` significant digits (the compact line)."""
    if isinstance(x, float):
        return float(f"{x:.{digits}g}")
    if isinstance(x, dict):
        return {k: _sig(v, digits) for k, v in x.items()}
    if isinstance(x, list):
        return [_sig(v, digits) for v in x]
    return x


_ROOF_KEYS = ("kernel", "bound", "achieved", "peak", "unit", "frac", "traffic", "avg_ms",
              "algorithmic_bytes", "algorithmic_flops", "achieved_over_measured")


def _compact_roofline(rl):
    return {k: rl[k] for k in _ROOF_KEYS if k in rl}


def _compact_cpu(cb):
    if not isinstance(cb, dict):
        return cb
    out = {k: cb[k] for k in ("value", "unit", "cores", "kind") if k in cb}
    out["sample"] = cb.get("sample", "")[:110]
    return out


def _kernel_ms(sub):
    return {k: v["avg_ms"] for k, v in sub.get("kernels", {}).items()}


def compact_line(result):
    """The one stdout line of the default run, kept to a few KB so that a
    driver storing only the tail of stdout keeps all of it: the headline
    (C2) fields; for C1, C3, C4 and C5 the step time, throughput, dominant
    kernel's roofline, per-kernel averages and CPU baseline; for the
    reference's other shapes (nn, dense, refcases) one summary each.  The
    full record goes to --detail PATH."""
    top = {k: v for k, v in result.items()
           if k not in ("configs", "kernels", "roofline", "cpu_baseline", "measured_roofs",
                        "profiled_ms_per_step")}
    top["roofline"] = _compact_roofline(result["roofline"])
    top["kernels_ms"] = _kernel_ms(result)
    if "cpu_baseline" in result:
        top["cpu_baseline"] = _compact_cpu(result["cpu_baseline"])
    if "measured_roofs" in result:
        mr = result["measured_roofs"]
        top["measured_roofs"] = {"copy_GBps": mr["copy_GBps"],
                                 "bf16_gemm_TFLOPs": mr["bf16_gemm_TFLOPs"]}
    configs = {}
    for name, sub in result.get("configs", {}).items():
        if name in ("c1", "c3", "c4", "c5"):
            c = {k: sub[k] for k in ("value", "unit", "ms_per_step", "dtype", "hbm_frac_step",
                                     "mfma_utilization", "cold_ms_per_step") if k in sub}
            c["config"] = {k: v for k, v in sub["config"].items() if k != "flop_convention"}
            c["roofline"] = _compact_roofline(sub["roofline"])
            c["kernels_ms"] = _kernel_ms(sub)
            if "cpu_baseline" in sub:
                c["cpu_baseline"] = _compact_cpu(sub["cpu_baseline"])
        elif name == "refcases":
            c = {case: [v["ms"], v["ms_prepared"], v["reference_ms"]]
                 for case, v in sub["cases"].items()}
            c["columns"] = "ms, ms_prepared, reference_ms (reference: RTX 5070 Ti)"
        else:
            c = {k: sub[k] for k in ("value", "unit", "ms_per_step", "dtype") if k in sub}
            c["workload"] = sub["config"]["workload"]
            rl = sub["roofline"]
            c["roofline"] = {k: rl[k] for k in ("kernel", "bound", "achieved", "unit", "frac",
                                                "avg_ms") if k in rl}
            if isinstance(sub.get("cpu_baseline"), dict):
                c["cpu_baseline"] = {k: sub["cpu_baseline"][k] for k in ("value", "unit")}
        configs[name] = c
    if configs:
        top["configs"] = configs
    out = _sig(top)
    for k in ("value", "ms_per_step"):      # the headline figures at full precision
        out[k] = result[k]
    return out


def main():
    global ARGS
    args = ARGS = parse()
    if args.calibrate_copy:
        calibrate_copy()
        return
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU only: this build has no multi-GPU path "
              "(collectives and sharding are out of scope); run with --gpus 1.",
              file=sys.stderr)
        sys.exit(2)
    runners = {"c1": run_c1, "c2": run_c2, "c3": lambda a: run_dot(a, ("c3",))["c3"],
               "c4": lambda a: run_dot(a, ("c4",))["c4"], "c5": run_c5,
               "dense": run_dense, "dense-causal": run_dense, "dense-pruned": run_dense,
               "nn": run_nn, "refcases": run_refcases}
    if args.config == "all":
        result = run_all(args)
    else:
        result = runners[args.config](args)
    if isinstance(result.get("cpu_baseline"), dict):
        result["cpu_baseline"]["cpu_model"] = cpu_model()
    roofs = measured_roofs()
    result["measured_roofs"] = roofs
    rl = result.get("roofline")
    if rl:
        # The dominant kernel against the same unit's in-run calibration: a
        # plain copy (which gathers can beat) or a library GEMM.
        measured = roofs["copy_GBps"] if rl.get("unit") == "GB/s" else roofs["bf16_gemm_TFLOPs"]
        rl["achieved_over_measured"] = rl["achieved"] / measured
    if args.detail:
        Path(args.detail).parent.mkdir(parents=True, exist_ok=True)
        Path(args.detail).write_text(json.dumps(result, indent=1) + "\n")
    line = compact_line(result) if args.config == "all" else result
    print(json.dumps(line, separators=(",", ":")), flush=True)


if __name__ == "__main__":
    main()
