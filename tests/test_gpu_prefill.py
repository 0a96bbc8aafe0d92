"""GPU parity of the whole-ubatch prefill (sulimo_hip_execute_prefill_ubatch[_ex]) against
the oracle's fp32 reference prefill (prefill.rs:362-560 op order, rounding points of
crates/sulimo-ocl/tests/test_prefill.rs:582-885) and the CPU path forward_token
(crates/sulimo-engine/src/forward_pass.rs:190-417).

Asserts mirror test_prefill.rs:829-885 (KV within one Q8_0 step, logits cosine,
argmax) with the tighter bounds of this build: logits max rel err <= 1e-2 of the
logit scale, top-1 agreement >= 99.5 % over all positions.
"""
import dataclasses
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

import oracle
from sulimo_amd import hip
from sulimo_amd import synthetic as S
from tests.helpers import cosine, kv_within_one_step, ulp_perturb

pytestmark = pytest.mark.gpu

TINY_NEOX = S.ModelConfig(2, 256, 512, 4, 2, 64, 64, 512, 10000.0, 1e-6, 1)
TINY_NORM = S.ModelConfig(2, 256, 512, 6, 2, 128, 128, 512, 500000.0, 1e-5, 0)


def run_both(cfg, seed, chunks, cap, all_logits=False, **model_kw):
    """Prefill the same token stream in `chunks` micro-batches on the GPU and in the oracle."""
    ctx = hip.HipContext.get_or_init(0)
    hm = S.make_model(cfg, seed, **model_kw)
    n_total = sum(chunks)
    toks = S.random_tokens(seed + 1, n_total, cfg.vocab)
    dm = hip.DeviceModel(ctx, hm, cap, max(chunks))
    om, okv = oracle.OracleModel(hm), oracle.OracleKv(cfg, cap)
    pos = 0
    res = []
    for m in chunks:
        t = toks[pos:pos + m]
        dm.embed(t)
        if all_logits:
            lb = hip.HipBuffer.device_only(ctx, m * cfg.vocab * 4)
            ab = hip.HipBuffer.device_only(ctx, m * 4)
            dm.execute_prefill_ubatch(pos, m, logits_all=lb, argmax_all=ab)
            g_all = lb.download(np.float32, (m, cfg.vocab))
            g_arg = ab.download(np.int32, (m,))
        else:
            dm.execute_prefill_ubatch(pos, m)
            g_all = g_arg = None
        g_last = dm.logits()
        r = oracle.prefill_reference(om, okv, S.embed_host(hm, t), pos, all_logits=all_logits)
        res.append((g_last, g_all, g_arg, r))
        pos += m
    dm.kv_sync_to_host(0, cap)
    return dm, okv, res


@pytest.mark.parametrize("cfg", [TINY_NEOX, TINY_NORM], ids=["neox", "norm"])
def test_tiny_prefill_matches_oracle(cfg):
    dm, okv, res = run_both(cfg, 21, [16], 64)
    g, _, _, r = res[0]
    scale = float(np.abs(r).max())
    assert np.max(np.abs(g - r)) <= 1e-2 * scale
    assert cosine(g, r) >= 0.999
    assert int(np.argmax(g)) == int(np.argmax(r))
    dk, dv = dm.kv_host()
    for l in range(cfg.n_layers):
        assert kv_within_one_step(dk[l], okv.k[l], np.arange(16), dm.bpp)
        assert kv_within_one_step(dv[l], okv.v[l], np.arange(16), dm.bpp)
    dm.release()


@pytest.mark.parametrize("cfg,qk_norm", [(TINY_NEOX, True), (TINY_NORM, True),
                                         (S.ModelConfig(2, 256, 512, 4, 2, 64, 40, 512, 10000.0, 1e-6, 1), True),
                                         (TINY_NEOX, False), (TINY_NORM, False)],
                         ids=["neox", "norm", "neox_rope40", "neox_bias_only", "norm_bias_only"])
def test_bias_and_qk_norm(cfg, qk_norm):
    """Optional q/k/v biases and QK-norm (forward_pass.rs:250-272): added to the GEMM
    output before its f16 rounding, per-head RMSNorm before RoPE; matches the oracle
    in two chunks and differs from the same model without them. Biases without QK-norm
    (Qwen2.5) run in the q/k/v GEMM's RoPE epilogue, the others in the separate kernel."""
    dm, okv, res = run_both(cfg, 27, [16, 12], 64, biases=True, qk_norm=qk_norm)
    for g, _, _, r in res:
        scale = float(np.abs(r).max())
        assert np.max(np.abs(g - r)) <= 1e-2 * scale
        assert cosine(g, r) >= 0.999
        assert int(np.argmax(g)) == int(np.argmax(r))
    dk, dv = dm.kv_host()
    for l in range(cfg.n_layers):
        assert kv_within_one_step(dk[l], okv.k[l], np.arange(28), dm.bpp)
        assert kv_within_one_step(dv[l], okv.v[l], np.arange(28), dm.bpp)
    dm.release()
    _, _, plain = run_both(cfg, 27, [16, 12], 64)
    assert np.max(np.abs(plain[-1][0] - res[-1][0])) > 0.05 * float(np.abs(res[-1][3]).max())


def test_resume_and_ring_wrap():
    """Three micro-batches on a capacity-48 ring: 24 tokens, 16 more (resume at 24), then 20
    that wrap past the capacity (each query sees exactly the last 48 positions)."""
    cfg = TINY_NEOX
    dm, okv, res = run_both(cfg, 33, [24, 16, 20], 48)
    for g, _, _, r in res:
        assert np.max(np.abs(g - r)) <= 1e-2 * float(np.abs(r).max())
        assert int(np.argmax(g)) == int(np.argmax(r))
    dk, dv = dm.kv_host()
    for l in range(cfg.n_layers):
        assert kv_within_one_step(dk[l], okv.k[l], np.arange(48), dm.bpp)
        assert kv_within_one_step(dv[l], okv.v[l], np.arange(48), dm.bpp)
    dm.release()


@pytest.mark.parametrize("cfg", [TINY_NEOX, TINY_NORM], ids=["neox", "norm"])
def test_fused_rope_store_odd_ubatches(cfg):
    """Ubatches of more than 4 tokens run RoPE, the Q8_0 K/V store and the attention-window
    entries in the q/k/v GEMM's epilogue. Odd chunk sizes put the window start of the
    second and fourth ubatch at positions 13 and 23 (element-wise V^T stores) and tiles
    past the last token; the 3-token ubatch takes the GEMV and the separate kernel; the
    last ubatch wraps the capacity-40 ring (staged K/V)."""
    dm, okv, res = run_both(cfg, 41, [13, 7, 3, 21], 40)
    for g, _, _, r in res:
        assert np.max(np.abs(g - r)) <= 1e-2 * float(np.abs(r).max())
        assert cosine(g, r) >= 0.999
        assert int(np.argmax(g)) == int(np.argmax(r))
    dk, dv = dm.kv_host()
    for l in range(cfg.n_layers):
        assert kv_within_one_step(dk[l], okv.k[l], np.arange(40), dm.bpp)
        assert kv_within_one_step(dv[l], okv.v[l], np.arange(40), dm.bpp)
    dm.release()


@pytest.mark.parametrize("cfg", [TINY_NEOX, TINY_NORM], ids=["neox", "norm"])
def test_micro_batches_of_one_to_five_tokens(cfg):
    """Decode-sized micro-batches: 1, 2, 4 and 3 tokens take the GEMV for every linear but
    SwiGLU (one, two and four token rows, f16 and residual epilogues) and the separate
    RoPE + Q8_0 store; the 5-token one the MFMA GEMMs with the fused store. Each matches
    the oracle, and the ring wraps in the last micro-batch."""
    dm, okv, res = run_both(cfg, 47, [1, 2, 4, 5, 1, 3], 14)
    for g, _, _, r in res:
        assert np.max(np.abs(g - r)) <= 1e-2 * float(np.abs(r).max())
        assert cosine(g, r) >= 0.999
        assert int(np.argmax(g)) == int(np.argmax(r))
    dk, dv = dm.kv_host()
    for l in range(cfg.n_layers):
        assert kv_within_one_step(dk[l], okv.k[l], np.arange(14), dm.bpp)
        assert kv_within_one_step(dv[l], okv.v[l], np.arange(14), dm.bpp)
    dm.release()


def test_llama_3b_layer_shapes():
    """One layer of the Llama-3.2-3B shape (hidden 3072, FFN 8192, 24/8 heads, head_dim
    128, Norm RoPE base 5e5; small vocab for the oracle's sake), prefilled in two chunks."""
    cfg = S.ModelConfig(1, 3072, 8192, 24, 8, 128, 128, 2048, 500000.0, 1e-5, 0)
    dm, okv, res = run_both(cfg, 55, [48, 40], 128)
    for g, _, _, r in res:
        assert np.max(np.abs(g - r)) <= 1e-2 * float(np.abs(r).max())
        assert cosine(g, r) >= 0.999
        assert int(np.argmax(g)) == int(np.argmax(r))
    dk, dv = dm.kv_host()
    assert kv_within_one_step(dk[0], okv.k[0], np.arange(88), dm.bpp)
    assert kv_within_one_step(dv[0], okv.v[0], np.arange(88), dm.bpp)
    dm.release()


def test_qwen_layer_one_ubatch_of_2048():
    """One layer of the Qwen2.5-1.5B shape (hidden 1536, FFN 8960, 12/2 heads, head_dim
    128, NeoX RoPE, biases; small vocab for the oracle's sake) on one 2048-token ubatch,
    the benchmark's ubatch: the gate/up GEMM runs persistent (more tiles than resident
    workgroups) with the SwiGLU epilogue, QKV with the fused RoPE epilogue, and the down
    projection splits K across workgroups."""
    cfg = S.ModelConfig(1, 1536, 8960, 12, 2, 128, 128, 2048, 1e6, 1e-6, 1)
    dm, okv, res = run_both(cfg, 91, [2048], 2048, biases=True)
    for g, _, _, r in res:
        assert np.max(np.abs(g - r)) <= 1e-2 * float(np.abs(r).max())
        assert cosine(g, r) >= 0.999
        assert int(np.argmax(g)) == int(np.argmax(r))
    dk, dv = dm.kv_host()
    assert kv_within_one_step(dk[0], okv.k[0], np.arange(2048), dm.bpp)
    assert kv_within_one_step(dv[0], okv.v[0], np.arange(2048), dm.bpp)
    dm.release()


def test_split_down_projection_runs_the_next_norm():
    """Two layers shaped so that the down projection (K = 4096) splits K across
    workgroups: its reduction also writes the next layer's attention RMSNorm (layer 0)
    and the output RMSNorm with the f16 residual (layer 1) in place of the separate norm
    launches; matches the oracle in two chunks."""
    cfg = S.ModelConfig(2, 1024, 4096, 8, 2, 128, 128, 512, 1e6, 1e-6, 1)
    dm, okv, res = run_both(cfg, 77, [64, 40], 128)
    for g, _, _, r in res:
        assert np.max(np.abs(g - r)) <= 1e-2 * float(np.abs(r).max())
        assert cosine(g, r) >= 0.999
        assert int(np.argmax(g)) == int(np.argmax(r))
    dk, dv = dm.kv_host()
    for l in range(cfg.n_layers):
        assert kv_within_one_step(dk[l], okv.k[l], np.arange(104), dm.bpp)
        assert kv_within_one_step(dv[l], okv.v[l], np.arange(104), dm.bpp)
    dm.release()


def _graph_sequence(ctx, hm, toks, cap, calls, reps):
    """Runs the prefill calls (start_pos, n) in order `reps` times on one device model
    and returns the logits and both rings after every call."""
    dm = hip.DeviceModel(ctx, hm, cap, max(n for _, n in calls))
    out = []
    for rep in range(reps):
        for pos, n in calls:
            dm.embed(toks[pos:pos + n])
            dm.execute_prefill_ubatch(pos, n)
            dm.kv_sync_to_host(0, cap)
            k, v = dm.kv_host()
            out.append((dm.logits(), [a.copy() for a in k], [a.copy() for a in v]))
            # eager work of the program's own between replays: a GEMM and a wait
            hip.enqueue_gemm_q4_0_f16(ctx, dm.layers[0]["q"].scales, dm.layers[0]["q"].quants,
                                      dm.scratch_bufs["h"], dm.scratch_bufs["q"], hm.cfg.q_dim, hm.cfg.embd, n)
            ctx.wait()
    dm.release()
    return out


@pytest.mark.parametrize("layers,calls,cap", [
    (2, [(0, 512)], 1024),                # prompt from position 0, kept window
    (2, [(0, 512), (512, 256)], 1024),    # resume over the kept window
    (2, [(0, 512), (512, 256)], 600),     # the second ubatch wraps the ring
    (1, [(0, 40), (40, 1)], 256),         # the first layer is the last
    (5, [(0, 96), (96, 23), (119, 23), (142, 5)], 1024),  # short turns, each at its own start
], ids=["fresh", "resume", "wrap", "one_layer", "turns"])
def test_graph_replay_bit_identical(layers, calls, cap):
    """Graph replay (the default) against eager launches: the same sequence of prefill
    calls, repeated three times with the program's own GEMM and wait between calls, gives
    logits and K/V ring bytes identical to the same sequence run eagerly, after every
    call (the first repetition captures each call's graphs, the others replay them; the
    context's counts show that both happened, whatever the depth of the model)."""
    cfg = dataclasses.replace(S.QWEN25_1_5B, n_layers=layers, vocab=4096)
    hm = S.make_model(cfg, 70, zero_mean=True)
    toks = S.random_tokens(71, 768, cfg.vocab)
    ctx = hip.HipContext.get_or_init(0)
    try:
        ctx.set_graph_replay(False)
        before = ctx.graph_replay_counts()
        eager = _graph_sequence(ctx, hm, toks, cap, calls, 3)
        assert ctx.graph_replay_counts() == before
        ctx.set_graph_replay(True)
        replay = _graph_sequence(ctx, hm, toks, cap, calls, 3)
        captured, replayed = (b - a for a, b in zip(before, ctx.graph_replay_counts()))
    finally:
        ctx.set_graph_replay(True)
    # every call captured or replayed; once the workspace has its size (one repetition), all replay
    assert captured + replayed == 3 * len(calls)
    assert captured >= len(calls) and replayed >= len(calls)
    for i, (lg, k, v) in enumerate(replay):
        le, ke, ve = eager[i]
        assert np.array_equal(lg.view(np.uint32), le.view(np.uint32)), f"logits of call {i}"
        for l in range(cfg.n_layers):
            assert np.array_equal(k[l], ke[l]) and np.array_equal(v[l], ve[l]), f"K/V of call {i}, layer {l}"


# hipGraphInstantiate in front of the runtime's, found first because it is loaded first:
# reports out of memory while `fail` is set.
_INSTANTIATE_SHIM = """
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
int fail = 1, calls = 0;
int hipGraphInstantiate(void **exec, void *graph, void **node, char *log, size_t size) {
  calls++;
  if (fail) return 2;
  void *rt = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
  if (!rt) rt = dlopen("libamdhip64.so", RTLD_LAZY);
  int (*real)(void **, void *, void **, char *, size_t) = rt ? dlsym(rt, "hipGraphInstantiate") : NULL;
  return real ? real(exec, graph, node, log, size) : 1;
}
"""
_FAILED_CAPTURE = """
import ctypes, sys
import numpy as np
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
from sulimo_amd import hip
from sulimo_amd import synthetic as S
fail, calls = (ctypes.c_int.in_dll(shim, n) for n in ("fail", "calls"))
cfg = S.ModelConfig(5, 256, 512, 4, 2, 64, 64, 512, 1e6, 1e-6, 1)
toks = S.random_tokens(5, 40, cfg.vocab)
ctx = hip.HipContext.get_or_init(0)
dm = hip.DeviceModel(ctx, S.make_model(cfg, 4), 64, 40)
dm.embed(toks)
x = dm.scratch_bufs["x"].download(np.uint16, (40, cfg.embd))
try:
    dm.execute_prefill_ubatch(0, 40)
    raise SystemExit("the call did not report the failed capture")
except hip.HipError as e:
    print("refused:", e, flush=True)
assert calls.value > 0
ctx.wait()
dm.kv_sync_to_host(0, 64)
assert not any(a.any() for ring in dm.kv_host() for a in ring), "K/V written by a call that failed"
assert np.array_equal(dm.scratch_bufs["x"].download(np.uint16, (40, cfg.embd)), x)
fail.value = 0
dm.execute_prefill_ubatch(0, 40)
got = dm.logits()
ctx.set_graph_replay(False)
dm.embed(toks)
dm.execute_prefill_ubatch(0, 40)
assert np.array_equal(got, dm.logits())
print("capture ok", flush=True)
"""


def test_failed_capture_launches_nothing(tmp_path):
    """A call whose graphs cannot be instantiated returns the error with nothing of the
    ubatch launched: the rings and the embeddings are what they were, and the next call,
    whose capture works, gives the eager result."""
    if shutil.which("gcc") is None:
        pytest.skip("gcc is not installed")
    (tmp_path / "shim.c").write_text(_INSTANTIATE_SHIM)
    (tmp_path / "run.py").write_text(_FAILED_CAPTURE)
    subprocess.run(["gcc", "-shared", "-fPIC", str(tmp_path / "shim.c"), "-o", str(tmp_path / "shim.so"), "-ldl"], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(hip.__file__)))
    path = os.pathsep.join([root] + [p for p in [os.environ.get("PYTHONPATH")] if p])
    r = subprocess.run([sys.executable, str(tmp_path / "run.py"), str(tmp_path / "shim.so")], capture_output=True, text=True,
                       timeout=100, cwd=root, env=dict(os.environ, PYTHONPATH=path))
    assert r.returncode == 0 and "capture ok" in r.stdout, r.stdout + r.stderr


def test_profiled_prefill_is_unchanged_and_counts_launches():
    """Per-launch timing (set_profiling) changes no result: with the GEMM kernels stamping
    their own start and end events, logits and K/V equal an unprofiled run bit for bit,
    and the statistics hold one launch of each GEMM role per layer (the down projection
    splitting K, so its interval runs from the partial-sum kernel to the reduction) plus
    the LM head, each with a positive time."""
    cfg = S.ModelConfig(2, 1024, 4096, 8, 2, 128, 128, 512, 1e6, 1e-6, 1)
    ctx = hip.HipContext.get_or_init(0)
    hm = S.make_model(cfg, 83, biases=True)
    toks = S.random_tokens(84, 64, cfg.vocab)
    dm = hip.DeviceModel(ctx, hm, 128, 64)
    runs = []
    try:
        for prof in (False, True):
            ctx.set_profiling(prof)
            dm.embed(toks)
            dm.execute_prefill_ubatch(0, 64)
            dm.kv_sync_to_host(0, 64)
            k, v = dm.kv_host()
            runs.append((dm.logits(), [a.copy() for a in k], [a.copy() for a in v]))
        st = ctx.prefill_stats()
    finally:
        ctx.set_profiling(False)
    (l0, k0, v0), (l1, k1, v1) = runs
    assert np.array_equal(l0, l1)
    for l in range(cfg.n_layers):
        assert np.array_equal(k0[l], k1[l]) and np.array_equal(v0[l], v1[l])
    roles = [st.gemm_qkv, st.gemm_o, st.gemm_gate_up, st.gemm_down]
    for r in roles:
        assert r.launches == cfg.n_layers and r.total_ms > 0 and r.flop > 0
    assert st.gemm_lm_head.launches == 1 and st.gemm_lm_head.total_ms > 0
    assert st.gemm.launches == 4 * cfg.n_layers + 1
    total = sum(r.total_ms for r in roles) + st.gemm_lm_head.total_ms
    assert abs(st.gemm.total_ms - total) <= 1e-6 * total
    assert st.attention.launches == cfg.n_layers and st.attention.total_ms > 0
    dm.release()


def test_resume_at_1536_with_wrap_at_2048():
    """Edge-shape resume: 1536 positions written in ubatches of 512, then 1024 new tokens
    appended to the capacity-2048 ring, wrapping at 2048 (the last ubatch's queries see
    exactly the last 2048 positions)."""
    cfg = TINY_NEOX
    dm, okv, res = run_both(cfg, 66, [512, 512, 512, 1024], 2048)
    for g, _, _, r in res:
        assert np.max(np.abs(g - r)) <= 1e-2 * float(np.abs(r).max())
        assert int(np.argmax(g)) == int(np.argmax(r))
    dk, dv = dm.kv_host()
    for l in range(cfg.n_layers):
        assert kv_within_one_step(dk[l], okv.k[l], np.arange(2048), dm.bpp)
        assert kv_within_one_step(dv[l], okv.v[l], np.arange(2048), dm.bpp)
    dm.release()


@pytest.mark.parametrize("weights", ["prescribed", "zero_mean"])
def test_all_positions_top1_agreement(weights):
    """All-positions LM-head validation mode: device argmax per position against the
    oracle's top-1, logits within 1e-2 of their scale. On the prescribed weights
    (positive scales) every position has nearly the same top-1, and agreement must be
    >= 99.5 %. The zero-mean variant (random-sign scales) gives distinct top-1 tokens at
    >= 90 % of positions, so that agreement measures something; there the oracle itself,
    fed the same embeddings with 10 % of them moved by one f16 ulp, keeps only about
    98 % of its top-1 tokens, and the device must reach 99.5 % or that floor less its
    sampling error."""
    zero_mean = weights == "zero_mean"
    cfg = S.ModelConfig(2, 512, 1024, 8, 2, 64, 64, 8192, 1e6, 1e-6, 1)
    dm, okv, res = run_both(cfg, 44, [96, 64], 256, all_logits=True, zero_mean=zero_mean)
    agree, total, r_args = 0, 0, []
    for _, g_all, g_arg, r_all in res:
        assert np.max(np.abs(g_all - r_all)) <= 1e-2 * float(np.abs(r_all).max())
        assert np.array_equal(g_arg, np.argmax(g_all, axis=1))
        r_args.append(np.argmax(r_all, axis=1))
        agree += int(np.sum(g_arg == r_args[-1]))
        total += g_arg.size
    distinct = len(set(np.concatenate(r_args).tolist())) / total
    bar = 0.995
    if zero_mean:
        # the oracle's floor: the same two chunks on one-ulp-perturbed embeddings
        hm = S.make_model(cfg, 44, zero_mean=True)
        toks = S.random_tokens(45, 160, cfg.vocab)
        om, pkv = oracle.OracleModel(hm), oracle.OracleKv(cfg, 256)
        kept = 0
        for pos, m in ((0, 96), (96, 64)):
            p_all = oracle.prefill_reference(om, pkv, ulp_perturb(S.embed_host(hm, toks[pos:pos + m])), pos,
                                             all_logits=True)
            kept += int(np.sum(np.argmax(p_all, axis=1) == r_args[0 if pos == 0 else 1]))
        floor = kept / total
        bar = min(0.995, floor - 2.0 * np.sqrt(floor * (1.0 - floor) / total) - 1.0 / total)
        print(f"all-positions top-1: oracle floor {floor:.4%}")
    print(f"all-positions top-1: agreement {agree / total:.4%} (bar {bar:.4%}), oracle top-1 distinct at "
          f"{distinct:.2%}")
    if zero_mean:
        assert distinct >= 0.9
    assert agree / total >= bar
    dm.release()


def test_prefill_rejects_oversized_ubatch():
    cfg = TINY_NEOX
    ctx = hip.HipContext.get_or_init(0)
    dm = hip.DeviceModel(ctx, S.make_model(cfg, 1), 64, 8)
    with pytest.raises(hip.HipError) as e:
        dm.execute_prefill_ubatch(0, 9)
    assert e.value.code == hip.ERR_INVALID_ARGUMENT
    dm.release()


def test_cpu_decode_after_gpu_prefill():
    """Prefill-to-CPU-decode hand-over: the KV bytes the GPU wrote, synced to the host
    ring, let forward_token continue the sequence like a CPU-only run would."""
    cfg = TINY_NEOX
    ctx = hip.HipContext.get_or_init(0)
    hm = S.make_model(cfg, 55)
    toks = S.random_tokens(56, 33, cfg.vocab)
    dm = hip.DeviceModel(ctx, hm, 64, 32)
    dm.prefill_tokens(toks[:32])
    dm.kv_sync_to_host(0, 32)
    dk, dv = dm.kv_host()
    om = oracle.OracleModel(hm)
    kv_gpu = oracle.OracleKv(cfg, 64, k=[a.copy() for a in dk], v=[a.copy() for a in dv])
    dec_gpu = oracle.forward_token(om, kv_gpu, int(toks[32]), 32)
    kv_cpu = oracle.OracleKv(cfg, 64)
    for p in range(32):
        oracle.forward_token(om, kv_cpu, int(toks[p]), p)
    dec_cpu = oracle.forward_token(om, kv_cpu, int(toks[32]), 32)
    assert cosine(dec_gpu, dec_cpu) >= 0.99
    # the CPU-decoded position goes back to the device ring (H2D of the dirty range)
    dm_k_before = dm.kv_k[0].download(np.uint8, (64 * dm.bpp,))
    for l in range(cfg.n_layers):
        dk[l][:] = kv_gpu.k[l]
        dv[l][:] = kv_gpu.v[l]
    dm.kv_sync_from_host(32, 1)
    after = dm.kv_k[0].download(np.uint8, (64 * dm.bpp,))
    assert np.array_equal(after[32 * dm.bpp:33 * dm.bpp], kv_gpu.k[0][32 * dm.bpp:33 * dm.bpp])
    assert np.array_equal(after[:32 * dm.bpp], dm_k_before[:32 * dm.bpp])
    dm.release()


@pytest.mark.parametrize("cfg", [TINY_NEOX, TINY_NORM], ids=["neox", "norm"])
def test_kept_window_follows_ring_writes(cfg):
    """The attention's f16 copy of the ring is kept between prefills of a prompt that fits
    the ring, and must follow every other write to it: after a first ubatch, the host
    rewrites positions 0..23 of every layer's ring (as CPU decode of another sequence
    would) and pushes them with kv_sync_from_host; the next ubatch must attend to the
    new bytes. A third ubatch after an untouched second one reuses the kept window."""
    ctx = hip.HipContext.get_or_init(0)
    hm = S.make_model(cfg, 61)
    toks = S.random_tokens(62, 64, cfg.vocab)
    cap = 96
    dm = hip.DeviceModel(ctx, hm, cap, 24)
    om = oracle.OracleModel(hm)
    dm.embed(toks[:24])
    dm.execute_prefill_ubatch(0, 24)
    dm.kv_sync_to_host(0, 24)
    dk, dv = dm.kv_host()
    rng = np.random.default_rng(63)
    for l in range(cfg.n_layers):  # other Q8_0 rows: f16 scale + int8 codes
        for ring in (dk[l], dv[l]):
            ring[:24 * dm.bpp] = oracle.quantize_f32_to_q8_0(
                rng.standard_normal(24 * cfg.kv_dim).astype(np.float32) * 2)
    dm.kv_sync_from_host(0, 24)
    okv = oracle.OracleKv(cfg, cap, k=[a.copy() for a in dk], v=[a.copy() for a in dv])
    for pos, m in ((24, 24), (48, 16)):
        dm.embed(toks[pos:pos + m])
        dm.execute_prefill_ubatch(pos, m)
        g = dm.logits()
        r = oracle.prefill_reference(om, okv, S.embed_host(hm, toks[pos:pos + m]), pos)
        assert np.max(np.abs(g - r)) <= 1e-2 * float(np.abs(r).max())
        assert cosine(g, r) >= 0.999
    dm.release()


def test_llama_3b_four_prompts_of_4096():
    """The Llama-3.2-3B-shaped model at its full size (28 layers, hidden 3072, 24/8
    heads, FFN 8192, vocab 128256, Norm RoPE base 5e5) on 4 independent prompts of 4096
    tokens, checked through size-independent properties (the oracle is too slow here):
    every prompt gives finite last-token logits; a prompt re-run after the others gives
    the same logits bit for bit (no state leaks between prompts); and one 4096-token
    ubatch agrees with 8 ubatches of 512 (all 4096 KV positions of every layer within one
    Q8_0 step, logits within 1e-2 of their scale)."""
    cfg = S.LLAMA32_3B
    T = 4096
    ctx = hip.HipContext.get_or_init(0)
    hm = S.make_model(cfg, 0x5EED0003)
    prompts = [S.random_tokens(0x70 + i, T, cfg.vocab) for i in range(4)]
    dm = hip.DeviceModel(ctx, hm, T, T)
    first = []
    for p in prompts:
        lg = dm.prefill_tokens(p, 0, T)
        assert np.all(np.isfinite(lg))
        first.append(lg)
    # prompt 0 again, after the other three
    again = dm.prefill_tokens(prompts[0], 0, T)
    assert np.array_equal(again.view(np.uint32), first[0].view(np.uint32))
    dm.kv_sync_to_host(0, T)
    dk, dv = dm.kv_host()
    k_one = [a.copy() for a in dk]
    v_one = [a.copy() for a in dv]
    # the same prompt in the reference's default micro-batches of 512
    dm_u = hip.DeviceModel(ctx, hm, T, 512)
    lg_u = dm_u.prefill_tokens(prompts[0], 0, 512)
    scale = float(np.abs(first[0]).max())
    assert np.max(np.abs(lg_u - first[0])) <= 1e-2 * scale
    assert cosine(lg_u, first[0]) >= 0.999
    dm_u.kv_sync_to_host(0, T)
    dk_u, dv_u = dm_u.kv_host()
    for l in range(cfg.n_layers):
        assert kv_within_one_step(dk_u[l], k_one[l], np.arange(T), dm.bpp)
        assert kv_within_one_step(dv_u[l], v_one[l], np.arange(T), dm.bpp)
    dm_u.release()
    dm.release()
