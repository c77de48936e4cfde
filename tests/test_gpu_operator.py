"""The whole operator on the GPU: REFRESH and SPARSE calls against the oracle operator at
small shapes, and size-independent properties at the full HunyuanVideo-720p shape."""

import dataclasses
import math

import pytest
import torch

import oracle as O
from gpu_util import (SMALL, assert_parity, assert_sparse_parity, inject, metrics,
                      parity_tolerance)
from recap_amd import HostBankOperator, Operator, OperatorConfig, REFRESH, SPARSE
from recap_amd.layout import Layout, SparseGeometry, hilbert_permutation
from recap_amd.synthetic import WORKLOADS, Workload, make_qkv, perturb

pytestmark = pytest.mark.gpu


def build(wl, *, chunks=1, host_banks=False, prefetch=True, layers=2):
    perm = hilbert_permutation(wl.grid)
    layout = Layout.from_permutation(perm, text_tokens=wl.text_tokens, text_first=wl.text_first)
    geo = SparseGeometry.build(layout, 128)
    cfg = OperatorConfig(head_density=wl.density, bank_chunks=chunks, host_banks=host_banks)
    cls = HostBankOperator if host_banks else Operator
    op = cls.build(cfg, geo, n_layers=layers)
    if host_banks:
        op.set_prefetch(prefetch)
    return op, perm


@pytest.mark.parametrize("name", list(SMALL))
def test_refresh_sparse_sequence_vs_oracle(cuda, name):
    """REFRESH / SPARSE / REFRESH (revalidation) / SPARSE against the oracle operator.

    Each sparse call is compared on the same refinement state (the GPU's state is handed to
    the oracle after every refresh): every output element within max-abs 2e-2 of the
    oracle's bf16 output (one bf16 ulp where that is larger) and cosine >= 0.999."""
    wl = SMALL[name]
    print(f"case {name}", flush=True)
    q, k, v = make_qkv(wl, seed=0)
    op, perm = build(wl)
    ref = O.OracleOperator(wl.grid, wl.text_tokens, wl.text_first, wl.density, permutation=perm)
    g = lambda x: x.to(cuda)  # noqa: E731
    op.begin_step(0, REFRESH)
    out = op.attend(0, g(q), g(k), g(v))
    ref.refresh(0, q, k, v)
    assert_parity(out.cpu().float(), ref.last["out_f32"], f"refresh-0 {name}")
    bank = op.banks[0][0]
    assert torch.equal(bank.partition.cpu().reshape(ref.layers[0].partition.shape),
                       ref.layers[0].partition)
    inject(ref, op, 0, wl)
    q1, k1, v1 = (perturb(x, 0.02, seed=1, step=1) for x in (q, k, v))
    op.begin_step(1, SPARSE)
    out = op.attend(0, g(q1), g(k1), g(v1))
    ref.sparse(0, q1, k1, v1)
    assert_sparse_parity(out, ref, op, q1, k1, v1, wl, cuda, f"sparse-1 {name}")
    q2, k2, v2 = (perturb(x, 0.03, seed=1, step=2) for x in (q, k, v))
    op.begin_step(2, REFRESH)
    out = op.attend(0, g(q2), g(k2), g(v2))
    ref.refresh(0, q2, k2, v2)
    assert_parity(out.cpu().float(), ref.last["out_f32"], f"refresh-2 {name}")
    age, error = op.drain_validation()
    num, den = (float(x) for x in ref.layers[0].pending_stats)
    print(f"  validation error gpu={error:.5f} oracle={math.sqrt(num / den):.5f} "
          f"rerank={ref.last['rerank']}", flush=True)
    assert age == 2 and abs(error - math.sqrt(num / den)) < 2e-3
    inject(ref, op, 0, wl)
    q3, k3, v3 = (perturb(x, 0.02, seed=1, step=3) for x in (q, k, v))
    op.begin_step(3, SPARSE)
    out = op.attend(0, g(q3), g(k3), g(v3))
    ref.sparse(0, q3, k3, v3)
    assert_sparse_parity(out, ref, op, q3, k3, v3, wl, cuda, f"sparse-3 {name}")


@pytest.mark.parametrize("name,dtype,batch", [
    ("text-first-ragged", torch.float16, 1),   # fp16 inputs (the boundary accepts both)
    ("text-last-d128", torch.float16, 1),
    ("text-first-ragged", torch.bfloat16, 2),  # CFG-batched calls, banks = B * H
])
def test_fp16_and_batched_calls_vs_oracle(cuda, name, dtype, batch):
    wl = SMALL[name]
    print(f"case {name} {dtype} batch={batch}", flush=True)
    q, k, v = make_qkv(wl, seed=3, batch=batch, dtype=dtype)
    op, perm = build(wl)
    ref = O.OracleOperator(wl.grid, wl.text_tokens, wl.text_first, wl.density, permutation=perm)
    g = lambda x: x.to(cuda)  # noqa: E731
    op.begin_step(0, REFRESH)
    out = op.attend(0, g(q), g(k), g(v))
    assert out.dtype == dtype and out.shape == q.shape
    ref.refresh(0, q, k, v, dtype=dtype)
    assert_parity(out.cpu().float(), ref.last["out_f32"], f"refresh {name} {dtype} b{batch}",
                  dtype=dtype)
    inject(ref, op, 0, wl)
    q1, k1, v1 = (perturb(x, 0.02, seed=4, step=1) for x in (q, k, v))
    op.begin_step(1, SPARSE)
    out = op.attend(0, g(q1), g(k1), g(v1))
    assert out.dtype == dtype
    ref.sparse(0, q1, k1, v1, dtype=dtype)
    assert_sparse_parity(out, ref, op, q1, k1, v1, wl, cuda, f"sparse {name} {dtype} b{batch}",
                         dtype=dtype)


@pytest.mark.parametrize("name", list(SMALL))
def test_sparse_vs_oracle_with_independent_state(cuda, name):
    """End to end with separately computed refinement states.  The coarse tail's gate
    [s^2 qsq.w <= theta^2] is discontinuous, the closure basis of each side comes from its
    own eigensolver (rotations within nearly equal eigenvalues move qsq), and
    D = (of - ratio oh)/(1 - ratio) - go amplifies last-bit differences of the bf16
    dense/head outputs, so a few elements may move by more than a bf16 ulp.  The same call
    on the oracle given the GPU's state (basis, partition, D, DL, gl_ref) must meet the
    strict bar, and every element of the GPU's output must lie within the bar plus the
    oracle's own change between its state and the GPU's: the differences beyond the bar
    come from the state alone (whose capture the refresh tests check on identical inputs),
    and they are no larger than the oracle's sensitivity to it.  Cosine >= 0.999 overall."""
    wl = SMALL[name]
    q, k, v = make_qkv(wl, seed=0)
    op, perm = build(wl)
    new_ref = lambda: O.OracleOperator(wl.grid, wl.text_tokens, wl.text_first,  # noqa: E731
                                       wl.density, permutation=perm)
    ref = new_ref()
    op.begin_step(0, REFRESH)
    op.attend(0, q.to(cuda), k.to(cuda), v.to(cuda))
    ref.refresh(0, q, k, v)
    q1, k1, v1 = (perturb(x, 0.02, seed=1, step=1) for x in (q, k, v))
    op.begin_step(1, SPARSE)
    out_dev = op.attend(0, q1.to(cuda), k1.to(cuda), v1.to(cuda))
    out = out_dev.cpu().float()
    ref.sparse(0, q1, k1, v1)
    want = ref.last["out_f32"]
    m, c = metrics(out, want)
    beyond = lambda x, r: (x - r.to(torch.bfloat16).float()).abs() > parity_tolerance(r)  # noqa: E731
    far = beyond(out, want)
    frac = float(far.float().mean())
    print(f"[independent {name}] max_abs={m:.3e} cos={c:.6f} frac-beyond-tolerance={frac:.2e}",
          flush=True)
    assert c >= 0.999
    # The oracle given the GPU's state: strict parity.
    ref_g = new_ref()
    inject(ref_g, op, 0, wl)
    ref_g.sparse(0, q1, k1, v1)
    assert_sparse_parity(out_dev, ref_g, op, q1, k1, v1, wl, cuda, f"given the GPU state {name}")
    # The state's own effect on the oracle: its output with its own state against its output
    # with the GPU's (basis alone, then the whole state).
    state = op.layers[0][0]
    ref_b = new_ref()
    ref_b.refresh(0, q, k, v)
    ref_b.layers[0].basis = state.basis.cpu().float()
    ref_b.sparse(0, q1, k1, v1)
    by_state = beyond(ref_g.last["out_f32"].float(), want)
    by_basis = beyond(ref_b.last["out_f32"].float(), want)
    print(f"  oracle with the GPU's state vs its own: {int(by_state.sum())} elements beyond the "
          f"bar (GPU vs oracle: {int(far.sum())}; both: {int((far & by_state).sum())}); "
          f"with the GPU's basis only: {int(by_basis.sum())}", flush=True)
    # |out - own| <= |out - given| + |given - own|, each side rounded as the outputs are
    given = ref_g.last["out_f32"].float()
    r16 = lambda x: x.to(torch.bfloat16).double()  # noqa: E731
    gap = (r16(given) - r16(want)).abs()
    excess = (out.double() - r16(want)).abs() - (parity_tolerance(given) + gap)
    print(f"  worst against the bar plus the state's effect: {float(excess.max()):+.3e}",
          flush=True)
    assert float(excess.max()) <= 0


def test_alpha_override_knob_vs_oracle(cuda):
    wl = SMALL["tiny"]
    q, k, v = make_qkv(wl, seed=2)
    op, perm = build(wl)
    ref = O.OracleOperator(wl.grid, wl.text_tokens, wl.text_first, wl.density, permutation=perm)
    op.begin_step(0, REFRESH)
    op.attend(0, q.to(cuda), k.to(cuda), v.to(cuda))
    inject(ref, op, 0, wl)
    q1, k1, v1 = (perturb(x, 0.05, seed=2, step=1) for x in (q, k, v))
    op.alpha_override = 0.8
    op.begin_step(1, SPARSE)
    out = op.attend(0, q1.to(cuda), k1.to(cuda), v1.to(cuda))
    ref.sparse(0, q1, k1, v1, alpha_override=0.8)
    assert_sparse_parity(out, ref, op, q1, k1, v1, wl, cuda, "alpha=0.8", alpha_override=0.8)


def test_sparse_before_refresh_raises(cuda):
    wl = SMALL["tiny"]
    op, _ = build(wl)
    q, k, v = (x.to(cuda) for x in make_qkv(wl, seed=0))
    op.begin_step(0, SPARSE)
    with pytest.raises(RuntimeError, match="before an exact refresh"):
        op.attend(0, q, k, v)
    hop, _ = build(wl, host_banks=True)
    hop.begin_step(0, SPARSE)
    with pytest.raises(RuntimeError, match="before an exact refresh"):
        hop.attend(0, q, k, v)


def test_non_contiguous_inputs_and_exact_kind(cuda):
    wl = SMALL["text-last-d128"]
    q, k, v = (x.to(cuda) for x in make_qkv(wl, seed=4))
    op, _ = build(wl)
    # diffusers hands [B, N, H, D] projections transposed to [B, H, N, D]
    qt, kt, vt = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v))
    op.begin_step(0, REFRESH)
    a = op.attend(0, q, k, v)
    op2, _ = build(wl)
    op2.begin_step(0, REFRESH)
    b = op2.attend(0, qt, kt, vt)
    assert torch.equal(a, b)
    op.begin_step(1, SPARSE)
    op2.begin_step(1, SPARSE)
    assert torch.equal(op.attend(0, q, k, v), op2.attend(0, qt, kt, vt))
    op.begin_step(2, "exact")
    exact = op.attend(0, q, k, v)
    assert_parity(exact.float(), a.float(), "exact vs refresh dense")


# -- full HunyuanVideo-720p shape: size-independent properties ----------------------------


@pytest.mark.parametrize("layers", [3, 4])
def test_host_banks_multi_step_schedule_identical(cuda, layers):
    """REFRESH, SPARSE, SPARSE, REFRESH (re-scoring valid banks), SPARSE, SPARSE over odd and
    even layer counts: pinned host banks with and without prefetch give the same outputs
    and validation statistics as banks resident on the GPU, call by call."""
    wl = SMALL["text-last-d128"]
    base = make_qkv(wl, seed=2, device=cuda)
    schedule = [REFRESH, SPARSE, SPARSE, REFRESH, SPARSE, SPARSE]
    inputs = [tuple(perturb(x, 0.03, seed=i, step=step) for i, x in enumerate(base))
              for step in range(len(schedule))]
    runs = {}
    counts = {}
    for label, kw in [("gpu", {}), ("host", {"host_banks": True}),
                      ("host-noprefetch", {"host_banks": True, "prefetch": False})]:
        op, _ = build(wl, layers=layers, **kw)
        outs, stats = [], []
        for step, kind in enumerate(schedule):
            op.begin_step(step, kind)
            for layer in range(layers):
                outs.append(op.attend(layer, *inputs[step]).clone())
            if kind == REFRESH:
                stats.append(op.drain_validation())
        if hasattr(op, "finish"):
            op.finish()
            counts[label] = op.pager_counts()
        torch.cuda.synchronize()
        runs[label] = (outs, stats)
    for label in ("host", "host-noprefetch"):
        for i, (a, b) in enumerate(zip(runs["gpu"][0], runs[label][0])):
            assert torch.equal(a, b), (label, i)
        assert runs["gpu"][1] == runs[label][1], label
    assert runs["gpu"][1][1] is not None  # the second refresh scored the first refinement
    print(f"  pager counts {counts}", flush=True)
    # Every bank a layer reads after the first refresh is staged in.  With prefetch all come
    # from the prefetch stream (the first refresh, which loads nothing, prefetches the next
    # step's layer 0 once its last layer's bank is on its way out; the two slots alternate
    # call by call, so with an odd number of layers too each step's layer 0 goes to the slot
    # the last layer does not hold); without prefetch all are copied on the compute stream.
    # Each refresh writes every layer's bank back.
    steps_with_loads = len(schedule) - 1
    loads = layers * steps_with_loads
    assert counts["host"]["written_back"] == counts["host-noprefetch"]["written_back"] \
        == layers * schedule.count(REFRESH)
    assert counts["host-noprefetch"]["from_prefetch"] == 0
    assert counts["host-noprefetch"]["copied"] == loads
    assert counts["host"]["from_prefetch"] + counts["host"]["copied"] == loads
    assert counts["host"]["copied"] == 0


@pytest.mark.parametrize("name,heads", [("wan2.1-480p", 2), ("cogvideox1.5", 2),
                                        ("hunyuan-720p", 1)])
def test_full_length_refresh_and_sparse_vs_oracle(cuda, name, heads):
    """REFRESH then a corrected SPARSE call at a reference workload's full sequence length
    (N = 32,760 Wan; 45,106 CogVideoX with its 226 text tokens first and a ragged last video
    block; 119,056 HunyuanVideo-720p with its 16-token last video block and 256 text tokens
    last), on one or two of its heads (heads are independent banks), against the oracle
    operator on the GPU's refinement state."""
    wl = dataclasses.replace(WORKLOADS[name], heads=heads)
    print(f"case {name} N={wl.tokens} d={wl.dim} heads={heads}", flush=True)
    q, k, v = make_qkv(wl, seed=0)
    op, perm = build(wl, layers=1)
    ref = O.OracleOperator(wl.grid, wl.text_tokens, wl.text_first, wl.density, permutation=perm)
    g = lambda x: x.to(cuda)  # noqa: E731
    op.begin_step(0, REFRESH)
    out = op.attend(0, g(q), g(k), g(v))
    ref.refresh(0, q, k, v)
    assert_parity(out.cpu().float(), ref.last["out_f32"], f"refresh {name}")
    print(f"  refresh {name}: oracle done, outputs agree", flush=True)
    bank = op.banks[0][0]
    assert torch.equal(bank.partition.cpu().reshape(ref.layers[0].partition.shape),
                       ref.layers[0].partition)
    inject(ref, op, 0, wl)
    q1, k1, v1 = (perturb(x, 0.02, seed=1, step=1) for x in (q, k, v))
    op.begin_step(1, SPARSE)
    got = op.attend(0, g(q1), g(k1), g(v1)).cpu().double()
    ref.sparse(0, q1, k1, v1)
    want = ref.last["out_f32"].double()
    assert_sparse_parity(got, ref, op, q1, k1, v1, wl, cuda, f"sparse {name}")


@pytest.fixture(scope="module")
def hunyuan_inputs(cuda):
    wl = WORKLOADS["hunyuan-720p"]
    q, k, v = make_qkv(wl, seed=0, device=cuda)
    return wl, q, k, v


def test_hunyuan_refresh_then_sparse_reproduces_dense(hunyuan_inputs):
    wl, q, k, v = hunyuan_inputs
    op, _ = build(wl)
    op.begin_step(0, REFRESH)
    dense = op.attend(0, q, k, v)
    ref = torch.nn.functional.scaled_dot_product_attention(q[:, :2], k[:, :2], v[:, :2])
    assert_parity(dense[:, :2].float(), ref.float(), "hunyuan dense vs sdpa (2 heads)")
    op.begin_step(1, SPARSE)
    sparse = op.attend(0, q, k, v)
    assert_parity(sparse.float(), dense.float(), "hunyuan refresh->sparse == dense")


def test_hunyuan_bank_chunks_and_host_banks_are_identical(hunyuan_inputs):
    wl, q, k, v = hunyuan_inputs
    q1, k1, v1 = (perturb(x, 0.03, seed=5, step=1) for x in (q, k, v))
    outs = {}
    for label, kw in [("plain", {}), ("chunks4", {"chunks": 4}),
                      ("host", {"host_banks": True}),
                      ("host-noprefetch", {"host_banks": True, "prefetch": False})]:
        op, _ = build(wl, layers=2, **kw)
        res = []
        op.begin_step(0, REFRESH)
        for layer in range(2):
            res.append(op.attend(layer, q, k, v))
        op.begin_step(1, SPARSE)
        for layer in range(2):
            res.append(op.attend(layer, q1, k1, v1))
        if hasattr(op, "finish"):
            op.finish()
        torch.cuda.synchronize()
        outs[label] = res
        print(f"  {label}: done", flush=True)
    for label in ("chunks4", "host", "host-noprefetch"):
        for a, b in zip(outs["plain"], outs[label]):
            assert torch.equal(a, b), label


@pytest.mark.parametrize("name", ["text-first-ragged", "text-last-d128"])
def test_sparse_call_on_a_bank_handed_in(cuda, name):
    """A SPARSE call of an operator that was given another one's bank and has no basis yet
    takes it from its own keys, stage by stage: with the keys of the other's refresh that is
    the same basis, and the output is the other's SPARSE output but for the order in which
    C_vk is summed.  Both routes record every stage event once a call."""
    wl = SMALL[name]
    print(f"case {name}", flush=True)
    q, k, v = (x.to(cuda) for x in make_qkv(wl, seed=0))
    outs, ops = [], []
    for _ in range(2):
        op, _ = build(wl, layers=1)
        op.stage_events = {}
        if ops:
            op.banks[0][0] = ops[0].banks[0][0]
        else:
            op.begin_step(0, REFRESH)
            op.attend(0, q, k, v)
        op.begin_step(1, SPARSE)
        assert op.layers[0][0].frozen != bool(ops)
        outs.append(op.attend(0, q, k, v))
        ops.append(op)
    torch.cuda.synchronize()
    assert torch.equal(ops[0].layers[0][0].basis, ops[1].layers[0][0].basis)
    assert_parity(outs[1].float(), outs[0].float(), f"handed-in bank {name}")
    for op in ops:
        events = op.stage_events
        assert list(events) == ["start", "pack", "closure", "coarse", "attention"]
        assert all(len(e) == 1 for e in events.values())
        times = [events["start"][0].elapsed_time(e[0]) for e in events.values()]
        assert times == sorted(times) and times[-1] > 0.0, times


@pytest.mark.parametrize("name", ["wan2.1-480p", "hunyuan-720p"])
def test_work_queue_schedule_gives_identical_outputs(cuda, monkeypatch, name):
    """The attention launches with per-XCD claim queues (XCDs that finish early take the
    others' last query blocks) and with the static assignment give bit-identical refresh
    and sparse outputs: only which workgroup computes a query block changes.  The SPARSE call
    always claims its items, so it is compared with its stages on the operator's own bank and
    geometry, the merge launch of which runs either way."""
    from recap_amd import kernels as K
    wl = WORKLOADS[name]
    print(f"case {name}", flush=True)
    q, k, v = make_qkv(wl, seed=0, device=cuda)
    q1, k1, v1 = (perturb(x, 0.02, seed=i, step=1) for i, x in enumerate((q, k, v)))
    dense, ran = {}, []
    dense_head = K.dense_head_attn
    for balance in (True, False):
        def patched(*a, balance=balance, **kw):
            ran.append(balance)
            return dense_head(*a, **kw, balance=balance)

        monkeypatch.setattr(K, "dense_head_attn", patched)
        op, _ = build(wl, layers=1)
        op.begin_step(0, REFRESH)
        dense[balance] = op.attend(0, q, k, v).clone()
        print(f"  refresh balance={balance}: done", flush=True)
    assert ran == [True, False]
    assert torch.equal(dense[True], dense[False])
    op.begin_step(1, SPARSE)
    sparse = op.attend(0, q1, k1, v1)
    layer, bank = op.layers[0][0], op.banks[0][0]
    geo, rowmap, scale = op._geometry(q1), op.layout.rowmap(q1.device), K.scale_for(wl.dim)
    kv = K.kv_pack(k1, v1, rowmap, geo)
    go, gl, drift = layer.coarse_tail_apply(
        q1, rowmap, layer.coarse_tail_context(kv, geo),
        bank.partition.reshape(-1, geo.nb, geo.nb), geo, scale, glref=bank.coarse_lse)
    for balance in (True, False):
        merged = K.sparse_merge_attn(q1, kv, rowmap, bank.head_kernel_mask, geo, scale, go, gl,
                                     bank.value, bank.log_mass, bank.coarse_lse,
                                     K.drift_center(drift, geo), balance=balance)
        print(f"  merge balance={balance}, {geo.attn_split} segments a long row: done", flush=True)
        assert torch.equal(merged, sparse), balance


def test_wan_refresh_then_four_drifting_sparse_calls_vs_oracle(cuda):
    """The Wan2.1-480p configuration as specified: N = 32,760 video tokens (21 x 30 x 52),
    128-dim heads, 20% density, bf16, one dense REFRESH followed by four corrected SPARSE
    calls whose inputs drift 2% further each step (fresh N(0,1) noise per step), on 2 of the
    12 heads (heads are independent banks).  The GPU's refinement state is handed to the
    oracle once, after the refresh; each sparse call is then compared with the oracle's on
    the same inputs (the state is read, never written, by a sparse call)."""
    wl = dataclasses.replace(WORKLOADS["wan2.1-480p"], heads=2)
    print(f"case wan2.1-480p N={wl.tokens} heads=2: REFRESH + 4 x SPARSE, 2% drift per step",
          flush=True)
    x = make_qkv(wl, seed=0)
    op, perm = build(wl, layers=1)
    ref = O.OracleOperator(wl.grid, wl.text_tokens, wl.text_first, wl.density, permutation=perm)
    g = lambda t: t.to(cuda)  # noqa: E731
    op.begin_step(0, REFRESH)
    out = op.attend(0, *(g(t) for t in x))
    ref.refresh(0, *x)
    assert_parity(out.cpu().float(), ref.last["out_f32"], "wan refresh")
    inject(ref, op, 0, wl)
    for step in range(1, 5):
        x = tuple(perturb(t, 0.02, seed=i, step=step) for i, t in enumerate(x))
        op.begin_step(step, SPARSE)
        got = op.attend(0, *(g(t) for t in x)).cpu()
        ref.sparse(0, *x)
        assert_sparse_parity(got, ref, op, *x, wl, cuda, f"wan sparse step {step}")


def test_two_host_threads_on_two_streams_match_serial(cuda):
    """The library keeps no mutable global state on the call path: two host threads, each
    with its own stream and operator, run a REFRESH and three SPARSE calls at the same time
    (three rounds); every output equals the same sequence run alone, bit for bit."""
    import threading

    wl = SMALL["text-last-d128"]
    schedule = [REFRESH, SPARSE, SPARSE, SPARSE]

    def run(seed, stream):
        with torch.cuda.stream(stream):
            op, _ = build(wl, layers=1)
            q, k, v = make_qkv(wl, seed=seed, device=cuda)
            outs = []
            for step, kind in enumerate(schedule):
                x = tuple(perturb(t, 0.02, seed=j, step=step) for j, t in enumerate((q, k, v)))
                op.begin_step(step, kind)
                outs.append(op.attend(0, *x).clone())
            stream.synchronize()
        return [o.cpu() for o in outs]

    streams = [torch.cuda.Stream() for _ in range(2)]
    serial = [run(10 + i, streams[i]) for i in range(2)]
    for rnd in range(3):
        results, errors = [None, None], []

        def worker(i):
            try:
                results[i] = run(10 + i, streams[i])
            except Exception as exc:  # re-raised below, in the test's thread
                errors.append(exc)

        threads = [threading.Thread(target=worker, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        if errors:
            raise errors[0]
        for i in range(2):
            for step, (a, b) in enumerate(zip(serial[i], results[i])):
                assert torch.equal(a, b), (rnd, i, step)
        print(f"  round {rnd}: both threads equal their serial runs", flush=True)


@pytest.mark.parametrize("grid,text,text_first", [
    ((1, 5, 20), 60, False),    # 100 video tokens: no full block, no refined rows
    ((1, 4, 25), 30, True),     # the same, text first
    ((1, 1, 128), 10, False),   # one full video block: it keeps every block, no tail
    ((1, 2, 100), 0, False),    # two blocks, the ragged last one forced: no tail either
])
def test_short_videos_vs_oracle(cuda, grid, text, text_first):
    """Videos of at most two blocks, against the oracle (the GPU's state handed over after
    the refresh).  Under one full block there are no refined rows: the refresh is the dense
    call and the sparse call the head.  When a query block keeps every video block its
    coarse tail is empty (log-mass -inf, also in the refresh's gl_ref) and the reference's
    merge makes its rows NaN: the drift weight exp(-|gl - gl_ref - c|) takes -inf - (-inf)
    (recap/kernels/detail_cache.py:267-284).  The same elements are NaN here; every other
    element meets the bar."""
    wl = Workload("short", 2, 64, grid, text, text_first, 0.25, torch.bfloat16)
    print(f"case grid={grid} text={text} text_first={text_first}", flush=True)
    q, k, v = make_qkv(wl, seed=0)
    op, perm = build(wl, layers=1)
    ref = O.OracleOperator(wl.grid, wl.text_tokens, wl.text_first, wl.density, permutation=perm)
    op.begin_step(0, REFRESH)
    out = op.attend(0, q.to(cuda), k.to(cuda), v.to(cuda)).cpu().float()
    ref.refresh(0, q, k, v)
    assert_parity(out, ref.last["out_f32"], f"refresh {grid}")
    inject(ref, op, 0, wl)
    q1, k1, v1 = (perturb(x, 0.02, seed=1, step=1) for x in (q, k, v))
    op.begin_step(1, SPARSE)
    got = op.attend(0, q1.to(cuda), k1.to(cuda), v1.to(cuda)).cpu().float()
    ref.sparse(0, q1, k1, v1)
    want = ref.last["out_f32"]
    nan = want.isnan()
    print(f"  NaN elements: oracle {int(nan.sum())}, here {int(got.isnan().sum())}", flush=True)
    assert torch.equal(got.isnan(), nan)
    if not bool(nan.all()):
        assert_parity(got.nan_to_num(), want.nan_to_num(), f"sparse {grid}")
    if wl.video_tokens < 128:
        assert not bool(nan.any())
    # A revalidating refresh: with no refined rows both sums are zero (error inf, as the
    # reference's drain gives for a zero denominator); with the empty tails both are NaN.
    q2, k2, v2 = (perturb(x, 0.03, seed=1, step=2) for x in (q, k, v))
    op.begin_step(2, REFRESH)
    out = op.attend(0, q2.to(cuda), k2.to(cuda), v2.to(cuda)).cpu().float()
    ref.refresh(0, q2, k2, v2)
    assert_parity(out, ref.last["out_f32"], f"refresh-2 {grid}")
    age, error = op.drain_validation()
    num, den = (float(x) for x in ref.layers[0].pending_stats)
    want_err = math.sqrt(num / den) if den > 0 else float("inf")
    print(f"  validation error here {error} oracle {want_err}", flush=True)
    assert age == 2
    if math.isnan(want_err) or math.isinf(want_err):
        assert (math.isnan(error) and math.isnan(want_err)) or error == want_err
    else:
        assert abs(error - want_err) < 2e-3


@pytest.mark.parametrize("grid,text,text_first,dim", [
    ((2, 16, 16), 100, False, 128),   # 512 video tokens: four whole blocks, text after
    ((2, 16, 16), 226, True, 64),     # the same video, text first (CogVideoX-like)
    ((3, 16, 24), 256, False, 128),   # 1,152 tokens: nine whole blocks, two text blocks
])
def test_video_in_whole_blocks_with_text_vs_oracle(cuda, grid, text, text_first, dim):
    """A video of whole 128-token blocks next to text: no ragged block is shared between
    video and text, so the text rows and columns stand alone.  REFRESH then SPARSE against
    the oracle, on the GPU's state, under the strict bar."""
    wl = Workload("whole", 2, dim, grid, text, text_first, 0.25, torch.bfloat16)
    print(f"case grid={grid} text={text} text_first={text_first} d={dim}", flush=True)
    q, k, v = make_qkv(wl, seed=2)
    op, perm = build(wl, layers=1)
    ref = O.OracleOperator(wl.grid, wl.text_tokens, wl.text_first, wl.density, permutation=perm)
    op.begin_step(0, REFRESH)
    out = op.attend(0, q.to(cuda), k.to(cuda), v.to(cuda))
    ref.refresh(0, q, k, v)
    assert_parity(out.cpu().float(), ref.last["out_f32"], f"refresh {grid}")
    assert torch.equal(op.banks[0][0].partition.cpu().reshape(ref.layers[0].partition.shape),
                       ref.layers[0].partition)
    inject(ref, op, 0, wl)
    q1, k1, v1 = (perturb(x, 0.02, seed=1, step=1) for x in (q, k, v))
    op.begin_step(1, SPARSE)
    out = op.attend(0, q1.to(cuda), k1.to(cuda), v1.to(cuda))
    ref.sparse(0, q1, k1, v1)
    assert_sparse_parity(out, ref, op, q1, k1, v1, wl, cuda, f"sparse {grid}")


@pytest.mark.parametrize("density,q_scale", [(0.03, 1.0), (0.9, 1.0), (0.25, 4.0)])
def test_density_extremes_and_peaky_queries_vs_oracle(cuda, density, q_scale):
    """The tiny shape (32 blocks) at the selection's extremes -- one kept block per query
    block (31 in the coarse tail), and 29 kept (3 in the tail) -- and with queries scaled
    by 4, so the softmax over keys and over block means is peaked (log-masses spread over
    tens of units).  REFRESH then SPARSE against the oracle on the GPU's state, strict bar."""
    wl = dataclasses.replace(SMALL["tiny"], density=density)
    print(f"case density={density} q_scale={q_scale}", flush=True)
    q, k, v = make_qkv(wl, seed=5)
    if q_scale != 1.0:
        q = (q.float() * q_scale).to(q.dtype)
    op, perm = build(wl, layers=1)
    ref = O.OracleOperator(wl.grid, wl.text_tokens, wl.text_first, wl.density, permutation=perm)
    op.begin_step(0, REFRESH)
    out = op.attend(0, q.to(cuda), k.to(cuda), v.to(cuda))
    ref.refresh(0, q, k, v)
    assert_parity(out.cpu().float(), ref.last["out_f32"], f"refresh d={density} s={q_scale}")
    part = ref.layers[0].partition
    assert torch.equal(op.banks[0][0].partition.cpu().reshape(part.shape), part)
    print(f"  kept per query block {int(part[0, 0].sum())} of {part.shape[-1]}", flush=True)
    inject(ref, op, 0, wl)
    q1, k1, v1 = (perturb(x, 0.02, seed=1, step=1) for x in (q, k, v))
    op.begin_step(1, SPARSE)
    out = op.attend(0, q1.to(cuda), k1.to(cuda), v1.to(cuda))
    ref.sparse(0, q1, k1, v1)
    assert_sparse_parity(out, ref, op, q1, k1, v1, wl, cuda, f"sparse d={density} s={q_scale}")


@pytest.mark.parametrize("name,theta,rank", [
    ("text-last-d128", 0.5, 0),      # tight gate, no leading closure directions
    ("text-last-d128", 8.0, 13),     # loose gate, the largest folded rank
    ("video-ragged-d128", 2.0, 20),  # rank past the folded form: the full w table
    ("text-first-ragged", 2.0, 64),  # rank = dim at d = 64
])
def test_gate_theta_and_closure_rank_vs_oracle(cuda, name, theta, rank):
    """The operator's coarse-tail knobs (closure_gate_theta, closure_rank of
    recap/config.py:56-80) away from their defaults: REFRESH then SPARSE against the oracle
    built with the same knobs, on the GPU's state, under the strict bar."""
    wl = SMALL[name]
    print(f"case {name} theta={theta} rank={rank}", flush=True)
    q, k, v = make_qkv(wl, seed=6)
    perm = hilbert_permutation(wl.grid)
    layout = Layout.from_permutation(perm, text_tokens=wl.text_tokens, text_first=wl.text_first)
    cfg = OperatorConfig(head_density=wl.density, closure_gate_theta=theta, closure_rank=rank)
    op = Operator.build(cfg, SparseGeometry.build(layout, 128), n_layers=1)
    ref = O.OracleOperator(wl.grid, wl.text_tokens, wl.text_first, wl.density, theta=theta,
                           rank=rank, permutation=perm)
    op.begin_step(0, REFRESH)
    out = op.attend(0, q.to(cuda), k.to(cuda), v.to(cuda))
    ref.refresh(0, q, k, v)
    assert_parity(out.cpu().float(), ref.last["out_f32"], f"refresh {name} {theta} {rank}")
    inject(ref, op, 0, wl)
    q1, k1, v1 = (perturb(x, 0.02, seed=1, step=1) for x in (q, k, v))
    op.begin_step(1, SPARSE)
    out = op.attend(0, q1.to(cuda), k1.to(cuda), v1.to(cuda))
    ref.sparse(0, q1, k1, v1)
    assert_sparse_parity(out, ref, op, q1, k1, v1, wl, cuda, f"sparse {name} {theta} {rank}")
