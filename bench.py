#!/usr/bin/env python3
"""Benchmark of the KV-cache compression path on one MI355X.

``python bench.py --gpus 1 --steps K --warmup W`` prints ONE JSON line.  A step is one pass of the
hot path over one batch of synthetic input that is already resident in HBM.  Without ``--workload``
the line's headline (``value``, ``roofline``, ``cpu_baseline``) is configuration 2 (SnapKV press over a
Qwen3-8B-shaped paged pool: score -> window fill -> top-k -> in-place compaction, all 36 layers, batch 8,
4096 tokens per sequence), ``decode_tokens_per_s`` is configuration 4 (128 decode steps in one HIP graph),
and ``configs`` holds the same measurement of every configuration: ms per step, throughput, roofline of the
dominant kernel, CPU baseline, and the result of the check below.  ``--workload`` measures one
configuration alone (knorm, snapkv, ccm, decode, hybrid, hybrid-decode = the 64 decode steps of
configuration 5; decode-eager / hybrid-decode-eager = the decode launches without a graph, the variants
to run under a profiler; snapkv-lse = cfg2 with the window queries' log-sum-exp given; copy = the
calibration copy of the traffic counters).

Objects on the line:
  roofline      the dominant kernel of the workload: algorithmic bytes per launch divided by its
                average launch time, measured with HIP events on the launch stream inside the timed
                region, against the published 8 TB/s HBM peak; ``traffic`` is the HBM byte count of one
                launch from an earlier rocprofv3 counter run of the same workload (``traffic_recorded``
                says of which commit and when), not a measurement of this run;
  cpu_baseline  the CPU restatement of the reference path (oracle/) timed on this host on a bounded
                sample of the same workload and scaled to the full pass;
  checked       one sampled (layer, sequence) column of the step that precedes the timed ones, compared with
                the oracle (scores / outputs within the parity tolerance, indices and moved bytes exact).

The graph workloads are refused under rocprofv3 (the profiler has crashed while tracing the long graphs);
use the ``*-eager`` variants there.
"""
from __future__ import annotations

import argparse
import ctypes as C
import json
import os
import sys
import time

import torch

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0          # MI355X HBM3E, published
MFMA_PEAK_TFLOPS = 2500.0      # dense bf16/fp16, published
D = 128


def _sync_time():
    torch.cuda.synchronize()
    return time.perf_counter()


CPU_THREAD_CAP = 16            # the share of host cores one GPU of the box comes with


def _cpu_threads():
    n = min(os.cpu_count() or 1, CPU_THREAD_CAP)
    torch.set_num_threads(n)
    return n


def _cpu_info(threads):
    """cores = threads the baseline actually used; the host's own count is stated beside it."""
    return {"cores": threads, "threads": torch.get_num_threads(), "host_cpu_count": os.cpu_count()}


def _under_profiler():
    """rocprofv3 announces itself through ROCPROF* / ROCP_* variables before the program starts."""
    return any(k.startswith(("ROCPROF", "ROCP_")) for k in os.environ)


class Bracket:
    """HIP events around the dominant kernel's launches (on the stream they are launched on)."""

    def __init__(self):
        self.pairs = []
        self.on = False

    def __enter__(self):
        if self.on:
            self._e0 = torch.cuda.Event(enable_timing=True)
            self._e0.record()
        return self

    def __exit__(self, *a):
        if self.on:
            e1 = torch.cuda.Event(enable_timing=True)
            e1.record()
            self.pairs.append((self._e0, e1))

    def mean_ms(self):
        return sum(a.elapsed_time(b) for a, b in self.pairs) / max(1, len(self.pairs))


class Workload:
    metric = "KV tokens compressed/sec"
    unit = "KV tokens/s"
    launches_per_bracket = 1
    kernel_flops = 0

    def __init__(self):
        self.br = Bracket()
        self.keep = False        # set for the checked step: the step keeps what check_after() needs
        self.kept = None

    # One sampled (layer, sequence) column of one step (the one before the timed steps) against the oracle:
    # check_before() snapshots the column's inputs, the step keeps references to its outputs, check_after()
    # compares and returns a summary or raises.  The line reports "checked".
    def check_before(self):
        pass

    def check_after(self):
        return None

    def check_collect(self):
        """What measure() calls right after the checked step: returns a callable that gives check_after()'s result.
        Here the check is evaluated at once; a workload whose check takes seconds of host work copies what the check
        needs and evaluates it when called, i.e. after the timed steps, so that the GPU does not idle before them."""
        result = self.check_after()
        return lambda: result


def _column_dense(kv_cache, plane, layer, table, n, cpu=True):
    """Tokens [0, n) of one sequence of one layer as a tensor [1, Hkv, n, D] (HuggingFace layout), on the CPU or, for
    a snapshot that must not make the GPU wait for the host, as a copy on the device."""
    bs = kv_cache.shape[3]
    blocks = torch.as_tensor(list(table)[:(n + bs - 1) // bs], device=kv_cache.device, dtype=torch.long)
    rows = kv_cache[plane, layer, blocks].reshape(-1, kv_cache.shape[4], kv_cache.shape[5])[:n]
    rows = rows.permute(1, 0, 2).unsqueeze(0)
    return rows.cpu() if cpu else rows.contiguous()


def _check_press_column(name, before_k, before_v, after_k, after_v, scores, ref_scores, idx, n_scored):
    """scores within 1e-3 of the oracle, indices = the oracle's stable selection on these scores, moved rows exact."""
    from oracle import presses as opress
    sc, ref = scores[..., :n_scored].cpu(), ref_scores[..., :n_scored]
    tol = 1e-3 * ref.abs() + 1e-3 * float(ref.abs().mean())
    if not bool(((sc - ref).abs() <= tol).all()):
        raise AssertionError(f"{name}: scores of the sampled column differ from the oracle by "
                             f"{float(((sc - ref).abs() / tol).max()):.2f} x the tolerance")
    want = opress.topk_lowest_index(scores.cpu(), idx.shape[-1])
    if not torch.equal(want, idx.cpu().long()):
        raise AssertionError(f"{name}: kept indices differ from the stable top-k of the scores")
    n = idx.shape[-1]
    for tag, b4, aft in (("K", before_k, after_k), ("V", before_v, after_v)):
        if not torch.equal(opress.gather_tokens(b4, idx.cpu().long().unsqueeze(0)), aft[:, :, :n]):
            raise AssertionError(f"{name}: compacted {tag} rows differ from the gathered source rows")
    return {"column": name, "scores_max_err_over_tol": round(float(((sc - ref).abs() / tol).max()), 4),
            "indices": "exact", "bytes": "exact"}


# ---------------------------------------------------------------------------------------------------
# configuration 2: SnapKV press
# ---------------------------------------------------------------------------------------------------
class SnapKVWorkload(Workload):
    name = "cfg2-snapkv-qwen3-8b"
    dtype_name = "bf16"
    kernel_name = "snapkv_kernel"
    one_launch = True              # scoring, selection and compaction of a column by one workgroup (fc_snapkv_press);
                                   # False: fc_snapkv_score, then fc_select_compact (shapes the press does not take)
    separate_selection = False     # with one_launch False: fc_topk_select and fc_compact as launches of their own

    def __init__(self, seed, device, given_lse=False, window_on_top=False):
        super().__init__()
        from fastcache_amd import synth
        self.L, self.B, self.Hq, self.Hkv, self.S, self.W, self.ksz = 36, 8, 32, 8, 4096, 64, 7
        self.given_lse = given_lse
        if given_lse:
            self.name = self.name + "+given-lse"
        # "keep 25 % plus the window" read as 1024 + 64 kept instead of 1024 with the window inside (the headline)
        self.window_on_top = window_on_top
        if window_on_top:
            self.name = self.name + "+window-on-top"
        self.ratio = 0.75
        self.device = device
        self.case = synth.snapkv_case(seed=seed, num_layers=self.L, batch=self.B, num_q_heads=self.Hq,
                                      num_kv_heads=self.Hkv, seq_len=self.S, window=self.W,
                                      dtype=torch.bfloat16, device=device, device_draw=True)
        self.tables = self.case.table_tensor(device)
        self.lens = self.case.lens_tensor(device)
        self.queries = self.case.queries
        self.tokens_per_step = self.B * self.S
        self.n_kept = int(self.S * (1 - self.ratio)) + (self.W if window_on_top else 0)
        e = 2
        q_bytes = self.L * self.B * self.Hq * self.W * D * e
        k_bytes = self.L * self.B * self.Hkv * self.S * D * e
        gather_bytes = 4 * self.L * self.B * self.Hkv * self.n_kept * D * e
        score_bytes = self.L * self.B * self.Hkv * self.S * 4
        # SnapKV scoring: Q window and K read once, fp32 scores written once; the one-launch press also moves the
        # kept K and V rows (read + written) in the same launch
        self.score_bytes_total = q_bytes + k_bytes + score_bytes
        self.kernel_bytes = self.score_bytes_total + gather_bytes
        self.kernel_flops = 2 * self.B * self.L * self.Hq * self.W * self.S * D
        self.pass_bytes = q_bytes + k_bytes + gather_bytes
        self.lse = None
        if given_lse:
            # what the prefill's attention kernel would hand over: ln sum exp(scale * q.k) per window query
            self.lse = torch.empty((self.L, self.B, self.Hq, self.W), dtype=torch.float32, device=device)
            G = self.Hq // self.Hkv
            mask = torch.triu(torch.full((self.W, self.S), float("-inf"), device=device), diagonal=self.S - self.W + 1)
            for layer in range(self.L):
                for b in range(self.B):
                    blocks = self.tables[b, :self.S // 256].long()
                    k = self.case.kv_cache[0, layer, blocks].reshape(self.S, self.Hkv, D).permute(1, 0, 2).float()
                    logits = torch.matmul(self.queries[layer, b].float(), k.repeat_interleave(G, 0).transpose(1, 2))
                    self.lse[layer, b] = torch.logsumexp(logits * D ** -0.5 + mask, dim=-1)

    def config(self):
        return {"workload": self.name, "layers": self.L, "batch": self.B, "q_heads": self.Hq,
                "kv_heads": self.Hkv, "head_dim": D, "seq_len": self.S, "window": self.W,
                "kernel_size": self.ksz, "keep": self.n_kept, "block_size": 256,
                "reductions": "sum", "causal_window": True, "window_in_budget": not self.window_on_top,
                "compaction": "in place"}

    def step(self):
        """score (bracketed) -> window fill -> top-k -> in-place compaction."""
        from fastcache_amd import _lib, ops
        from fastcache_amd._lib import check, current_stream, fn
        kv = self.case.kv_cache
        L, B, Hkv, S = self.L, self.B, self.Hkv, self.S
        kview = _lib.paged_view(kv[0], self.tables, self.lens, S)
        vview = _lib.paged_view(kv[1], self.tables, self.lens, S)
        scores = torch.empty((L, B, Hkv, S), dtype=torch.float32, device=self.device)
        row_max = torch.empty((L, B, Hkv), dtype=torch.float32, device=self.device)
        st = current_stream()
        if self.one_launch:                       # what paged_press.snapkv_compress_paged issues for this shape
            with self.br:
                scores, idx = ops.snapkv_press(kview, vview, self.queries, self.W, self.ksz, self.n_kept, True, "sum",
                                               seq_lens=self.lens, lse=self.lse)
            if self.keep:
                self.kept, self.keep = (scores, idx), False
            return
        with self.br:
            if self.lse is None:
                check(fn("fc_snapkv_score")(C.byref(kview), self.queries.data_ptr(), self.Hq, self.W, self.ksz, 1,
                                            D ** -0.5, 1.0, scores.data_ptr(), S, row_max.data_ptr(), st),
                      "fc_snapkv_score")
            else:
                check(fn("fc_snapkv_score_lse")(C.byref(kview), self.queries.data_ptr(), self.lse.data_ptr(), self.Hq,
                                                self.W, self.ksz, 1, D ** -0.5, 1.0, scores.data_ptr(), S,
                                                row_max.data_ptr(), st), "fc_snapkv_score_lse")
        # the window fill needs every row maximum of the layer, so it is its own (small) launch
        check(fn("fc_snapkv_fill_window")(scores.data_ptr(), S, L, B, Hkv, self.lens.data_ptr(), S, self.W,
                                          row_max.data_ptr(), st), "fc_snapkv_fill_window")
        if self.separate_selection:
            idx = ops.topk_select(scores, self.n_kept)
            ops.compact(kview, vview, kview, vview, idx)
        else:                                    # what paged_press.snapkv_compress_paged issues
            idx = ops.select_compact(kview, vview, scores, self.n_kept)
        if self.keep:
            self.kept, self.keep = (scores, idx), False

    def check_before(self):
        # snapshots stay on the device until the comparison: no host copy, hence no idle GPU, before the timed steps
        self.cl, self.cb = self.L // 2, self.B // 2
        tab = self.case.block_tables[self.cb]
        self.snap = [_column_dense(self.case.kv_cache, p, self.cl, tab, self.S, cpu=False) for p in range(2)]
        self.keep = True

    def check_collect(self):
        scores, idx = self.kept
        l, b = self.cl, self.cb
        tab = self.case.block_tables[b]
        after = [_column_dense(self.case.kv_cache, p, l, tab, self.n_kept, cpu=False) for p in range(2)]   # before any later step
        sc, ix, q = scores[l, b].clone(), idx[l, b].clone(), self.queries[l, b:b + 1]
        self.kept = None

        def evaluate():
            from oracle import presses as opress
            snap = [t.cpu() for t in self.snap]
            ref = opress.snapkv_score(q.cpu(), snap[0], self.W, self.ksz, True, "sum")[0]
            return _check_press_column(f"layer {l}, sequence {b}", snap[0], snap[1], after[0].cpu(), after[1].cpu(),
                                       sc.cpu(), ref, ix.cpu(), self.S - self.W)
        return evaluate

    def cpu_baseline(self, budget_s=12.0):
        """CPU restatement of the same pass, layer by layer until the time budget, scaled linearly."""
        from oracle import pipeline as opipe
        threads = _cpu_threads()
        tables, lens = self.case.block_tables, [self.S] * self.B
        t_total, layers_done = 0.0, 0
        for layer in range(self.L):
            pool = self.case.kv_cache[:, layer:layer + 1].cpu()
            q = self.queries[layer:layer + 1].cpu()
            comp = opipe.snapkv_press_compressor(q, self.ratio, self.W, self.ksz, True, "sum", not self.window_on_top)
            t0 = time.perf_counter()
            opipe.compress_batch(pool, tables, lens, comp)
            dt = time.perf_counter() - t0
            if layer == 0:          # warm-up layer is not counted
                continue
            t_total += dt
            layers_done += 1
            if t_total > budget_s:
                break
        full_pass_s = t_total / layers_done * self.L
        return {"value": round(self.tokens_per_step / full_pass_s, 1), "unit": self.unit, **_cpu_info(threads),
                "kind": "port",
                "sample": f"{layers_done} of {self.L} layers x all {self.B} sequences, "
                          f"{t_total:.2f} s measured, scaled linearly to the full pass"}


# ---------------------------------------------------------------------------------------------------
# configuration 1: Knorm press
# ---------------------------------------------------------------------------------------------------
class KnormWorkload(Workload):
    name = "cfg1-knorm-llama-7b"
    dtype_name = "f32"
    kernel_name = "knorm_press_kernel"

    def __init__(self, seed, device):
        super().__init__()
        from fastcache_amd import synth
        self.L, self.B, self.H, self.S, self.ratio = 32, 1, 32, 1024, 0.5
        self.device = device
        self.case = synth.knorm_case(seed=seed, device=device, device_draw=True)
        self.tables, self.lens = self.case.table_tensor(device), self.case.lens_tensor(device)
        self.tokens_per_step = self.B * self.S
        self.n_kept = int(self.S * (1 - self.ratio))
        e = 4
        moved = 4 * self.L * self.B * self.H * self.n_kept * D * e                 # kept K,V read + written
        self.pass_bytes = self.L * self.B * self.H * D * e * self.S + moved         # + K read once for the norms
        self.kernel_bytes = self.pass_bytes                                        # one launch does all of it

    def config(self):
        return {"workload": self.name, "layers": self.L, "batch": self.B, "kv_heads": self.H, "head_dim": D,
                "seq_len": self.S, "keep": self.n_kept, "block_size": 256, "compaction": "in place"}

    def step(self):
        from fastcache_amd import paged_press
        with self.br:
            res = paged_press.knorm_compress_paged(self.case.kv_cache, self.tables, self.lens, self.S, self.ratio)
        if self.keep:
            self.kept, self.keep = (res.scores, res.indices), False

    def check_before(self):
        self.cl = self.L // 2
        tab = self.case.block_tables[0]
        self.snap = [_column_dense(self.case.kv_cache, p, self.cl, tab, self.S, cpu=False) for p in range(2)]
        self.keep = True

    def check_collect(self):
        scores, idx = self.kept
        l = self.cl
        tab = self.case.block_tables[0]
        after = [_column_dense(self.case.kv_cache, p, l, tab, self.n_kept, cpu=False) for p in range(2)]   # before any later step
        sc, ix = scores[l, 0].clone(), idx[l, 0].clone()
        self.kept = None

        def evaluate():
            from oracle import presses as opress
            snap = [t.cpu() for t in self.snap]
            return _check_press_column(f"layer {l}, sequence 0", snap[0], snap[1], after[0].cpu(), after[1].cpu(),
                                       sc.cpu(), opress.knorm_score(snap[0])[0], ix.cpu(), self.S)
        return evaluate

    def cpu_baseline(self, budget_s=12.0):
        from oracle import pipeline as opipe
        threads = _cpu_threads()
        pool = self.case.kv_cache.cpu()
        comp = opipe.knorm_press_compressor(self.ratio)
        opipe.compress_batch(pool[:, :1].clone(), self.case.block_tables, [self.S], comp)     # warm-up
        t0 = time.perf_counter()
        opipe.compress_batch(pool, self.case.block_tables, [self.S], comp)
        dt = time.perf_counter() - t0
        return {"value": round(self.tokens_per_step / dt, 1), "unit": self.unit, **_cpu_info(threads), "kind": "port",
                "sample": f"the full pass (all {self.L} layers), {dt:.2f} s"}


class KnormThreeLaunchWorkload(KnormWorkload):
    """The same pass as three launches (norms, top-k, compaction), the form that columns too long for LDS take."""
    name = "cfg1-knorm-llama-7b-three-launches"
    kernel_name = "compact_kernel"

    def __init__(self, seed, device):
        super().__init__(seed, device)
        self.kernel_bytes = 4 * self.L * self.B * self.H * self.n_kept * D * 4

    def step(self):
        from fastcache_amd import _lib, ops
        kv = self.case.kv_cache
        kview = _lib.paged_view(kv[0], self.tables, self.lens, self.S)
        vview = _lib.paged_view(kv[1], self.tables, self.lens, self.S)
        scores = ops.knorm_score(kview, self.device)
        idx = ops.topk_select(scores, self.n_kept)
        with self.br:
            ops.compact(kview, vview, kview, vview, idx)
        if self.keep:
            self.kept, self.keep = (scores, idx), False


# ---------------------------------------------------------------------------------------------------
# configurations 3 and 5: CCM MLP compressors
# ---------------------------------------------------------------------------------------------------
class CCMWorkload(Workload):
    name = "cfg3-ccm-linear-decouple-llava-1.5-7b"
    dtype_name = "f16"
    kernel_name = "mlp_kernel"
    launches_per_bracket = 4

    def __init__(self, seed, device, hybrid=False):
        super().__init__()
        from types import SimpleNamespace
        from fastcache_amd import synth
        from fastcache_amd.utils_ccm import KVCacheHybridCompressor, KVCacheLinearDecoupleCompressor
        self.device, self.hybrid = device, hybrid
        if hybrid:
            self.name, self.dtype_name, self.launches_per_bracket = "cfg5-ccm-hybrid-minicpm-v-2.6", "bf16", 2
            self.L, self.B, self.H, self.S, self.cf, dtype = 28, 16, 4, 16384, 5, torch.bfloat16
            self.it_len = [0, self.S]
            self.case = synth.hybrid_case(seed=seed, device=device, device_draw=True)
            cfg = SimpleNamespace(architectures=["MiniCPMV"], num_hidden_layers=self.L, num_key_value_heads=self.H,
                                  num_attention_heads=28, hidden_size=28 * D)
            torch.manual_seed(seed)
            self.module = KVCacheHybridCompressor(cfg, compression_factor=self.cf, min_seq_len=1)
        else:
            self.L, self.B, self.H, self.S, self.cf, dtype = 32, 45, 32, 640, 2, torch.float16
            self.it_len = [576, 64]
            self.case = synth.ccm_case(seed=seed, device=device, device_draw=True)
            cfg = SimpleNamespace(text_config=SimpleNamespace(num_hidden_layers=self.L, num_key_value_heads=self.H,
                                                              hidden_size=self.H * D))
            torch.manual_seed(seed)
            self.module = KVCacheLinearDecoupleCompressor(cfg)      # constructor defaults: cf 2, min_seq_len 1
        self.module = self.module.to(device).to(dtype).eval()
        self.tables, self.lens = self.case.table_tensor(device), self.case.lens_tensor(device)
        self.tokens_per_step = self.B * self.S
        segs = [n for n in ([self.S] if hybrid else self.it_len) if n]
        rows = sum(n // self.cf for n in segs)
        self.C = sum(n // self.cf + n % self.cf for n in segs)
        cols = 2 * self.L * self.B * self.H
        e = 2
        w_bytes = (2 if hybrid else 4) * self.L * (self.cf * D * D + 2 * D * D + 3 * D) * e
        self.kernel_bytes = cols * (rows * self.cf * D * e + rows * D * e) + w_bytes
        self.kernel_flops = cols * rows * 2 * (self.cf * D * D + 2 * D * D)
        self.pass_bytes = self.kernel_bytes + cols * 2 * (self.C - rows) * D * e

    def config(self):
        return {"workload": self.name, "layers": self.L, "batch": self.B, "kv_heads": self.H, "head_dim": D,
                "seq_len": self.S, "it_len": self.it_len, "compression_factor": self.cf, "compressed_len": self.C,
                "block_size": 256, "write_back": "in place"}

    def step(self):
        with self.br:
            self.module.paged_forward(self.case.kv_cache, self.tables, self.lens, self.S, self.it_len)

    def check_before(self):
        self.cl, self.cb = self.L // 2, self.B // 2
        tab = self.case.block_tables[self.cb]
        self.snap = [_column_dense(self.case.kv_cache, p, self.cl, tab, self.S) for p in range(2)]

    def check_after(self):
        """Compressed rows of the sampled column: error norm within 1e-3 of the oracle's norm (both sides
        accumulate in fp32 and round to the storage dtype after every Linear)."""
        from oracle import ccm as occm
        l, b = self.cl, self.cb
        sd = {}
        for k, v in self.module.state_dict().items():          # keys are group.layer.index.name
            g, lay, rest = k.split(".", 2)
            if int(lay) == l:
                sd[f"{g}.0.{rest}"] = v.detach().cpu().float()
        fwd = occm.hybrid_forward if self.hybrid else occm.linear_decouple_forward
        (rk, rv), = fwd([(self.snap[0], self.snap[1])], self.it_len, sd, self.cf, 1)
        tab = self.case.block_tables[b]
        worst = 0.0
        for p, ref in enumerate((rk, rv)):
            got = _column_dense(self.case.kv_cache, p, l, tab, self.C).float()
            ref = ref.float()
            assert got.shape == ref.shape, (got.shape, ref.shape)
            rel = float((got - ref).norm() / ref.norm())
            worst = max(worst, rel)
            if rel > 1e-3:
                raise AssertionError(f"cfg MLP: layer {l}, sequence {b}, plane {p}: relative error norm {rel:.2e}")
        return {"column": f"layer {l}, sequence {b}", "rel_error_norm": float(f"{worst:.3e}")}

    def cpu_baseline(self, budget_s=12.0):
        from oracle import ccm as occm
        from oracle import pipeline as opipe
        threads = _cpu_threads()
        sd = {k: v.detach().cpu().float() for k, v in self.module.state_dict().items()}
        fwd = occm.hybrid_forward if self.hybrid else occm.linear_decouple_forward
        nb = self.B
        tables, lens = self.case.block_tables[:nb], [self.S] * nb
        t_total, done = 0.0, 0
        for layer in range(self.L):
            pool = self.case.kv_cache[:, layer:layer + 1].cpu()
            lsd = {}
            for k, v in sd.items():          # keys are group.layer.index.name
                g, lay, rest = k.split(".", 2)
                if int(lay) == layer:
                    lsd[f"{g}.0.{rest}"] = v
            comp = lambda hf, i, n: fwd(hf, self.it_len, lsd, self.cf, 1)
            t0 = time.perf_counter()
            opipe.compress_batch(pool, tables, lens, comp)
            dt = time.perf_counter() - t0
            if layer == 0:
                continue
            t_total += dt
            done += 1
            if t_total > budget_s:
                break
        full = t_total / done * self.L * (self.B / nb)
        return {"value": round(self.tokens_per_step / full, 1), "unit": self.unit, **_cpu_info(threads), "kind": "port",
                "sample": f"{done} of {self.L} layers x {nb} of {self.B} sequences, {t_total:.2f} s measured, "
                          "scaled linearly to the full pass"}


# ---------------------------------------------------------------------------------------------------
# configuration 4: decode paged attention, 128 steps in one HIP graph
# ---------------------------------------------------------------------------------------------------
class DecodeWorkload(Workload):
    name = "cfg4-decode-paged-attention-llava-1.5-7b"
    dtype_name = "f16"
    kernel_name = "decode_attn_kernel"
    metric = "decode tokens/sec"
    unit = "tokens/s"

    def __init__(self, seed, device, graph_steps=128, eager=False, hybrid=False):
        super().__init__()
        from fastcache_amd import synth
        from fastcache_amd.engine.decode_graph import DecodeGraph
        self.eager = eager
        self.device = device
        if hybrid:   # the decode half of configuration 5: 16 caches compressed to 3280 tokens, 7 query heads per kv head
            self.name, self.dtype_name = "cfg5-decode-after-hybrid-minicpm-v-2.6", "bf16"
            self.kernel_name = "decode_column_kernel"
            self.L, self.B, self.Hq, self.Hkv, self.T, dtype = 28, 16, 28, 4, graph_steps, torch.bfloat16
            self.lens_text = "3280 (16384 compressed to 20 %)"
            self.case = synth.decode_case(seed=seed, num_layers=self.L, batch=self.B, num_kv_heads=self.Hkv,
                                          min_len=3280, max_len=3280, steps=self.T, dtype=dtype, device=device,
                                          device_draw=True)
        else:
            self.L, self.B, self.Hq, self.Hkv, self.T, dtype = 32, 90, 32, 32, graph_steps, torch.float16
            self.lens_text = "uniform[128, 2048]"
            self.case = synth.decode_case(seed=seed, steps=self.T, device=device, device_draw=True)
        self.tables = self.case.table_tensor(device)
        self.lens0 = self.case.lens_tensor(device)
        self.lens = self.lens0.clone()
        g = torch.Generator(device=device).manual_seed(seed + 1)
        mk = lambda h: torch.randn((self.T, self.L, self.B, h, D), generator=g, device=device,
                                   dtype=torch.float32).to(dtype)
        self.dg = DecodeGraph(self.case.kv_cache, self.tables, self.lens, mk(self.Hq), mk(self.Hkv), mk(self.Hkv),
                              D ** -0.5)
        if not eager:
            self.dg.capture()
        self.tokens_per_step = self.B * self.T
        sum_len = sum(self.case.seq_lens)
        e = 2
        # mean over the graph's steps of one layer's launch: K and V of every cached token read once
        mean_len = sum_len + self.B * (self.T + 1) / 2
        per_launch = int(2 * self.Hkv * D * e * mean_len + 2 * self.B * self.Hq * D * e)
        self.launches_per_bracket = self.L * self.T
        self.kernel_bytes = per_launch * self.launches_per_bracket      # summed over the bracket
        self.pass_bytes = self.kernel_bytes

    def config(self):
        return {"workload": self.name, "layers": self.L, "batch": self.B, "q_heads": self.Hq, "kv_heads": self.Hkv,
                "head_dim": D, "context_lens": self.lens_text, "sum_context_lens": sum(self.case.seq_lens),
                "block_size": 256, "decode_steps_per_graph": self.T,
                "graph": "none (eager launches, for the profiler)" if self.eager else "one hipGraph of all steps and layers"}

    def step(self):
        self.lens.copy_(self.lens0)
        with self.br:
            if self.eager:
                self.dg.run_eager()
            else:
                self.dg.replay()

    def check_after(self):
        """Attention outputs of a few sequences at the first and last step of one layer (every replay appends the
        same rows, so the pool holds the final state): within 2e-2 absolute of the fp32 oracle."""
        from oracle import attention as oattn
        torch.cuda.synchronize()
        layer, seqs = self.L // 2, [0, self.B // 2, self.B - 1]
        kc, vc = self.case.kv_cache[0, layer].cpu(), self.case.kv_cache[1, layer].cpu()
        tab = self.tables[seqs].cpu()
        worst = 0.0
        for t in (0, self.T - 1):
            lens = (self.lens0[seqs] + (t + 1)).cpu()
            ref = oattn.decode_attention(self.dg.q_steps[t, layer, seqs].cpu(), kc, vc, lens, tab, D ** -0.5)
            err = float((self.dg.out[t, layer, seqs].cpu().float() - ref.float()).abs().max())
            worst = max(worst, err)
            if err > 2e-2:
                raise AssertionError(f"decode: layer {layer}, step {t}: attention output off by {err:.3e}")
        return {"column": f"layer {layer}, sequences {seqs}, steps 0 and {self.T - 1}", "max_abs_err": float(f"{worst:.3e}")}

    def cpu_baseline(self, budget_s=12.0):
        from oracle import attention as oattn
        threads = _cpu_threads()
        nb = 8
        q = self.dg.q_steps[0, 0, :nb].cpu()
        lens = self.lens0[:nb].cpu()
        tab = self.tables[:nb].cpu()
        kc, vc = self.case.kv_cache[0, 0].cpu(), self.case.kv_cache[1, 0].cpu()
        oattn.decode_attention(q, kc, vc, lens, tab, D ** -0.5)
        t0, reps = time.perf_counter(), 0
        while time.perf_counter() - t0 < budget_s and reps < 50:
            oattn.decode_attention(q, kc, vc, lens, tab, D ** -0.5)
            reps += 1
        dt = (time.perf_counter() - t0) / reps
        share = float(lens.sum()) / float(self.lens0.sum())
        step_s = dt / share * self.L
        return {"value": round(self.B / step_s, 1), "unit": self.unit, **_cpu_info(threads), "kind": "port",
                "sample": f"attention of {nb} of {self.B} sequences, 1 of {self.L} layers, {reps} repetitions, "
                          "scaled by cached tokens and layers to one decode step"}


# ---------------------------------------------------------------------------------------------------
# calibration: a plain copy of known size through fc_copy_tokens (for scaling FETCH_SIZE / WRITE_SIZE)
# ---------------------------------------------------------------------------------------------------
class CopyWorkload(Workload):
    """Plain streams of known size, for the counter calibration (`copy`) and as the practical ceilings the HBM-bound
    kernels are compared with: this library's copy kernel, the runtime's device-to-device copy (through torch and
    called directly), a torch elementwise kernel, read-only streams (this library's and torch's reduction) and
    write-only streams (torch's fill kernel, the runtime's memset).  Each moves 512 MiB per tensor."""
    name = "copy-calibration-1GiB"
    dtype_name = "bf16"
    kernel_name = "copy_rows_kernel"
    metric = "tokens copied/sec"
    unit = "tokens/s"
    KINDS = {  # kind -> (workload name, kernel name as a trace shows it, tensors read, tensors written)
        "compact": ("copy-calibration-1GiB", "copy_rows_kernel", 1, 1),
        # the same bytes between two sets of pages of ONE pool: the views may overlap, so the rows move in order
        "compact-ordered": ("copy-ordered-walk-1GiB", "compact_kernel", 1, 1),
        "torch-copy": ("copy-torch-copy_-1GiB", "hipMemcpyAsync device to device (torch Tensor.copy_)", 1, 1),
        "hip-memcpy": ("copy-hipMemcpyDtoDAsync-1GiB", "hipMemcpyDtoDAsync", 1, 1),
        "torch-kernel": ("copy-torch-elementwise-1GiB", "torch elementwise kernel (torch.neg, out=)", 1, 1),
        "read": ("read-key-channel-energy-512MiB", "key_channel_energy_kernel", 1, 0),
        "torch-read": ("read-torch-sum-512MiB", "torch reduce kernel (Tensor.sum over the bytes viewed as fp32)", 1, 0),
        "torch-fill": ("write-torch-fill-512MiB", "torch fill kernel (Tensor.fill_)", 0, 1),
        "hip-memset": ("write-hipMemsetAsync-512MiB", "hipMemsetAsync", 0, 1),
    }

    def __init__(self, seed, device, kind="compact"):
        super().__init__()
        self.device, self.kind = device, kind
        self.name, self.kernel_name, n_read, n_written = self.KINDS[kind]
        # 16 * 16 * 8 * 1024 rows of 256 B = 512 MiB per tensor, as 2048 (layer, sequence, head) columns: this library's
        # kernels take a workgroup per column, so a tensor of a few very long columns would measure the grid, not the memory
        L, B, H, S = 16, 16, 8, 1024
        if kind == "compact-ordered":
            pages = S // 256
            self.pool = torch.randn((L, 2 * B * pages, 256, H, D), device=device, dtype=torch.float32).to(torch.bfloat16)
            t = torch.arange(B * pages, dtype=torch.int32, device=device).view(B, pages)
            self.tables = (t, t + B * pages)
            self.src = self.pool[:, :B * pages]
        else:
            self.src = torch.randn((L, B, H, S, D), device=device, dtype=torch.float32).to(torch.bfloat16)
            self.dst = torch.empty_like(self.src)
        self.S = S
        self.tokens_per_step = B * S
        self.nbytes = self.src.numel() * 2
        self.kernel_bytes = (n_read + n_written) * self.nbytes
        self.pass_bytes = self.kernel_bytes
        self.n_read, self.n_written = n_read, n_written
        self.hip = None
        if kind in ("hip-memcpy", "hip-memset"):
            import ctypes
            self.hip = ctypes.CDLL("libamdhip64.so")
            self.hip.hipMemcpyDtoDAsync.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_void_p]
            self.hip.hipMemsetAsync.argtypes = [C.c_void_p, C.c_int, C.c_size_t, C.c_void_p]

    def config(self):
        return {"workload": self.name, "bytes_read": self.n_read * self.nbytes, "bytes_written": self.n_written * self.nbytes}

    def step(self):
        from fastcache_amd import _lib, ops
        st = torch.cuda.current_stream().cuda_stream
        with self.br:
            if self.kind == "compact":
                ops.copy_tokens(_lib.dense_view(self.src), _lib.dense_view(self.dst), 0, self.S, 0)
            elif self.kind == "compact-ordered":
                ops.copy_tokens(_lib.paged_view(self.pool, self.tables[0], None, self.S),
                                _lib.paged_view(self.pool, self.tables[1], None, self.S), 0, self.S, 0)
            elif self.kind == "torch-copy":
                self.dst.copy_(self.src)
            elif self.kind == "hip-memcpy":
                if self.hip.hipMemcpyDtoDAsync(self.dst.data_ptr(), self.src.data_ptr(), self.nbytes, st) != 0:
                    raise RuntimeError("hipMemcpyDtoDAsync failed")
            elif self.kind == "torch-kernel":
                torch.neg(self.src, out=self.dst)
            elif self.kind == "read":
                ops.key_channel_energy(_lib.dense_view(self.src), self.device)
            elif self.kind == "torch-read":
                self.src.view(torch.float32).sum()
            elif self.kind == "torch-fill":
                self.dst.fill_(1.5)
            elif self.kind == "hip-memset":
                if self.hip.hipMemsetAsync(self.dst.data_ptr(), 0, self.nbytes, st) != 0:
                    raise RuntimeError("hipMemsetAsync failed")

    def cpu_baseline(self, budget_s=0):
        threads = _cpu_threads()
        a = self.src[0, :1].cpu()
        t0 = time.perf_counter()
        b = a.clone()
        dt = time.perf_counter() - t0
        return {"value": round(a.shape[0] * a.shape[2] / dt, 1), "unit": self.unit, **_cpu_info(threads), "kind": "port",
                "sample": "torch clone of 1 of 4 sequences on the host"}


def _separate(w, three):
    """cfg2 as two launches (scoring; selection + compaction) or three (scoring; selection; compaction)."""
    w.one_launch = False
    w.separate_selection = three
    w.kernel_bytes = w.score_bytes_total
    w.name += "-three-launches" if three else "-two-launches"
    return w


CEILINGS = ("compact", "compact-ordered", "torch-copy", "hip-memcpy", "torch-kernel", "read", "torch-read", "torch-fill", "hip-memset")

WORKLOADS = {"copy": CopyWorkload,
             **{f"stream-{k}": (lambda seed, dev, k=k: CopyWorkload(seed, dev, kind=k)) for k in CEILINGS},
             "snapkv": SnapKVWorkload, "knorm": KnormWorkload, "knorm-3": KnormThreeLaunchWorkload, "ccm": CCMWorkload, "decode": DecodeWorkload,
             "hybrid": lambda seed, dev: CCMWorkload(seed, dev, hybrid=True),
             # cfg2 with the window queries' log-sum-exp handed in (not the BASELINE metric: the reference has no such input)
             "snapkv-lse": lambda seed, dev: SnapKVWorkload(seed, dev, given_lse=True),
             # cfg2 under the other reading of its budget: the 64 window positions kept on top of the quarter (1088)
             "snapkv-top": lambda seed, dev: SnapKVWorkload(seed, dev, window_on_top=True),
             # cfg2 with the selection and compaction as launches of their own
             "snapkv-two": lambda seed, dev: _separate(SnapKVWorkload(seed, dev), False),
             "snapkv-three": lambda seed, dev: _separate(SnapKVWorkload(seed, dev), True),
             "snapkv-lse-two": lambda seed, dev: _separate(SnapKVWorkload(seed, dev, given_lse=True), False),
             # the decode launches without a graph, 4 steps per bracket: rocprofv3 cannot walk the 128-step graph
             "decode-eager": lambda seed, dev: DecodeWorkload(seed, dev, graph_steps=4, eager=True),
             # the 64 decode steps that follow the compression in configuration 5, in one graph
             "hybrid-decode": lambda seed, dev: DecodeWorkload(seed, dev, graph_steps=64, hybrid=True),
             "hybrid-decode-eager": lambda seed, dev: DecodeWorkload(seed, dev, graph_steps=4, eager=True, hybrid=True)}


# HBM-side bytes per launch of a workload's dominant kernel, from two rocprofv3 counter runs
# (FETCH_SIZE, WRITE_SIZE in KiB per dispatch), each scaled by what the same counter reads for the
# copy workload below, whose traffic is known (512 MiB read, 512 MiB written):
#   copy:   FETCH_SIZE 2.623e5 KiB -> scale 1.999;  WRITE_SIZE 5.284e5 KiB -> scale 0.992
# The commands and raw readings are in profiles/*_hbm_traffic.txt.
_COUNTER_RUN = {"commit": "76bf753", "date": "2026-11-25"}   # the tree whose kernels the counter runs below measured
# (the press launches of cfg1 and cfg2, the calibration and cfg5's MLP launch were counted again at commit cbd5ec4;
#  cfg5's readings came out as at commit 3ee0b1a)
_COUNTER_RUN_OF = {"cfg5-ccm-hybrid-minicpm-v-2.6": {"commit": "cbd5ec4", "date": "2026-11-25"},
                   "cfg1-knorm-llama-7b": {"commit": "cbd5ec4", "date": "2026-11-25"},
                   "cfg2-snapkv-qwen3-8b": {"commit": "cbd5ec4", "date": "2026-11-25"},
                   "cfg5-decode-after-hybrid-minicpm-v-2.6": {"commit": "0a758fa", "date": "2026-12-02"}}
_FETCH_SCALE = 524288 / 2.623e5
_WRITE_SCALE = 524288 / 5.284e5
_COUNTER_KIB = {  # workload name -> (FETCH_SIZE, WRITE_SIZE) per dispatch of the dominant kernel
    "cfg1-knorm-llama-7b": (5.247e5, 5.304e5),
    "cfg1-knorm-llama-7b-three-launches": (2.641e5, 5.263e5),
    "cfg2-snapkv-qwen3-8b": (3.004e6, 1.225e6),                       # the one-launch press: kept rows moved as well
    "cfg2-snapkv-qwen3-8b-two-launches": (2.390e6, 3.636e4),
    "cfg2-snapkv-qwen3-8b+given-lse-two-launches": (1.273e6, 3.636e4),           # one sweep: K is read once
    "cfg3-ccm-linear-decouple-llava-1.5-7b": (1.861e6, 1.845e6),      # mean over the 4 launches of a step
    "cfg5-ccm-hybrid-minicpm-v-2.6": (3.921e6, 1.468e6),
    # The decode launches were counted without the graph, 4 steps per bracket (the profiler is not run on the long
    # graphs).  A launch reads every cached token once and the caches grow by a token per step, so the reading
    # is scaled from that run's algorithmic bytes per launch (third entry) to those of the measured graph.
    "cfg4-decode-paged-attention-llava-1.5-7b": (8.059e5, 7414.0, 1648099328),
    "cfg5-decode-after-hybrid-minicpm-v-2.6": (5.270e4, 924.0, 107790336),
}


def _measured_traffic(workload_name, algorithmic_bytes_per_launch):
    kib = _COUNTER_KIB.get(workload_name)
    if kib is None:
        return None
    scale = algorithmic_bytes_per_launch / kib[2] if len(kib) > 2 else 1.0
    return int(round((kib[0] * _FETCH_SCALE + kib[1] * _WRITE_SCALE) * 1024 * scale))


GRAPH_WORKLOADS = {"decode": "decode-eager", "hybrid-decode": "hybrid-decode-eager"}


def measure(workload, seed, dev, steps, warmup, cpu_baseline=True, cpu_budget_s=12.0, check=True, min_warm_s=0.0):
    """One workload: one checked step, warm-up, a timed run of exactly `steps` steps right behind it, roofline of
    the dominant kernel, then a longer run for the sustained rate.
    The checked step comes first and its comparison with the CPU oracle last: that comparison leaves the GPU idle for
    seconds, and after any idle gap, even 5 ms, the next ~25 passes of the SnapKV workload run at a lower shader
    clock (2.4 ms falling to 1.9 ms), so nothing may separate the warm-up from the timed steps and as little as
    possible the workload's set-up from the warm-up.
    `min_warm_s` keeps warming up until that much time has passed (used for the configurations whose warm-up count
    is this file's own choice, not the caller's)."""
    w = WORKLOADS[workload](seed, dev)
    checked = pending = None
    if check:                              # one step of its own, on the fresh pool
        w.check_before()
        w.step()
        pending = w.check_collect()        # evaluated below, after the timed steps, where it costs seconds of host work
    t_warm = _sync_time()
    done = 0
    while done < warmup or _sync_time() - t_warm < min_warm_s:
        w.step()
        done += 1
    warmup = done
    w.br.on = True
    t0 = _sync_time()
    for _ in range(steps):
        w.step()
    t1 = _sync_time()
    ms_per_step = (t1 - t0) * 1e3 / steps
    value = w.tokens_per_step / (ms_per_step * 1e-3)
    if pending is not None:
        checked = pending()                # raises when the sampled column is off: no number without a right result
    # the rate once the clocks have settled: the same step for another ~0.3 s, not part of `value`
    sustained = None
    w.br.on = False
    if ms_per_step < 30.0:
        n = max(steps, int(300.0 / ms_per_step))
        for _ in range(n // 2):
            w.step()
        t2 = _sync_time()
        for _ in range(n):
            w.step()
        t3 = _sync_time()
        s_ms = (t3 - t2) * 1e3 / n
        sustained = {"steps": n, "after_steps": steps + n // 2, "ms_per_step": round(s_ms, 4),
                     "value": round(w.tokens_per_step / (s_ms * 1e-3), 1)}

    # the bracket may hold several launches of the dominant kernel: bytes and time are summed over
    # them, which equals (mean bytes per launch) / (mean launch duration)
    k_ms = w.br.mean_ms() / w.launches_per_bracket
    per_launch = w.kernel_bytes // w.launches_per_bracket
    achieved = w.kernel_bytes / w.launches_per_bracket / (k_ms * 1e-3) / 1e9
    roofline = {"bound": "hbm", "kernel": w.kernel_name, "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS,
                "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 4),
                "traffic": _measured_traffic(w.name, per_launch),
                "traffic_recorded": _COUNTER_RUN_OF.get(w.name, _COUNTER_RUN) if w.name in _COUNTER_KIB else None,
                "kernel_ms": round(k_ms, 4), "launches_per_step": w.launches_per_bracket,
                "algorithmic_bytes_per_launch": per_launch,
                "pass_gbs": round(w.pass_bytes / (ms_per_step * 1e-3) / 1e9, 1),
                "pass_frac": round(w.pass_bytes / (ms_per_step * 1e-3) / 1e9 / HBM_PEAK_GBS, 4)}
    if w.kernel_flops:
        tf = w.kernel_flops / w.launches_per_bracket / (k_ms * 1e-3) / 1e12
        roofline["mfma_tflops"] = round(tf, 1)
        roofline["mfma_frac"] = round(tf / MFMA_PEAK_TFLOPS, 4)
    out = {"metric": w.metric, "value": round(value, 1), "unit": w.unit, "ms_per_step": round(ms_per_step, 4),
           "steps": steps, "warmup": warmup, "dtype": w.dtype_name, "config": w.config(), "roofline": roofline,
           "sustained": sustained, "checked": checked is not None, "check": checked}
    if cpu_baseline:
        out["cpu_baseline"] = w.cpu_baseline(cpu_budget_s)
    del w
    torch.cuda.empty_cache()
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--seed", type=int, default=0)
    ap.add_argument("--workload", choices=sorted(WORKLOADS), default=None,
                    help="one configuration alone; default: cfg2 as the headline plus every configuration")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-check", action="store_true")
    ap.add_argument("--hbm-ceilings", action="store_true",
                    help="plain copy / read / write streams of known size (this library's, torch's, the runtime's): "
                         "what the memory system delivers to the simplest kernels; prints one JSON line and exits")
    args = ap.parse_args()

    if args.gpus != 1:
        print("bench.py: this build runs on ONE GPU (no collectives, no sharding); "
              f"--gpus {args.gpus} is not supported", file=sys.stderr)
        sys.exit(2)
    profiled = _under_profiler()
    if profiled and args.workload in GRAPH_WORKLOADS:
        # before any GPU call: rocprofv3 has ended in a segmentation fault while tracing the long decode graphs
        print(f"bench.py: --workload {args.workload} replays a HIP graph of thousands of nodes and is not run under "
              f"rocprofv3; profile --workload {GRAPH_WORKLOADS[args.workload]} (the same launches without a graph)",
              file=sys.stderr)
        sys.exit(3)
    if not torch.cuda.is_available():
        print("bench.py: no GPU visible", file=sys.stderr)
        sys.exit(1)
    from fastcache_amd import _lib
    _lib.load()          # fail loudly when the HIP library is missing
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    cpu, check = not args.no_cpu_baseline, not args.no_check
    if args.hbm_ceilings:
        rows = {}
        for kind in CEILINGS:
            r = measure(f"stream-{kind}", args.seed, dev, args.steps, args.warmup, False, 0.0, False, min_warm_s=0.2)
            rows[kind] = {"workload": r["config"]["workload"], "kernel": r["roofline"]["kernel"],
                          "bytes_read": r["config"]["bytes_read"], "bytes_written": r["config"]["bytes_written"],
                          "ms": r["roofline"]["kernel_ms"], "GB/s": r["roofline"]["achieved"],
                          "frac_of_8TB/s": r["roofline"]["frac"],
                          "sustained_ms": r["sustained"]["ms_per_step"] if r["sustained"] else None}
        print(json.dumps({"hbm_ceilings": rows, "steps": args.steps, "warmup": args.warmup}), flush=True)
        return

    head_name = args.workload or "snapkv"
    head = measure(head_name, args.seed, dev, args.steps, args.warmup, cpu, 12.0, check)
    out = {"metric": head["metric"], "value": head["value"], "unit": head["unit"], "n_gpus": 1,
           "steps": args.steps, "warmup": args.warmup, "ms_per_step": head["ms_per_step"],
           "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": head["dtype"],
           "data": "synthetic", "config": head["config"], "roofline": head["roofline"], "sustained": head["sustained"],
           "checked": head["checked"], "check": head["check"]}
    if cpu:
        out["cpu_baseline"] = head["cpu_baseline"]
    if args.workload is None:
        # every configuration on the same line; the decode graphs give way to their eager forms under a profiler
        configs = {"cfg2": head}
        plan = [("cfg2-window-on-top", "snapkv-top", args.steps, args.warmup),
                ("cfg1", "knorm", 50, 3), ("cfg3", "ccm", 10, 3), ("cfg4", "decode", 3, 1),
                ("cfg5-compress", "hybrid", 10, 3), ("cfg5-decode", "hybrid-decode", 5, 2)]
        for key, name, steps, warmup in plan:
            if profiled and name in GRAPH_WORKLOADS:
                name = GRAPH_WORKLOADS[name]
            configs[key] = measure(name, args.seed, dev, steps, warmup, cpu, 6.0, check, min_warm_s=0.2)
        out["configs"] = configs
        out["decode_tokens_per_s"] = configs["cfg4"]["value"]
        out["decode_tokens_per_s_after_compression"] = configs["cfg5-decode"]["value"]
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
