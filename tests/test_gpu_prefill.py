"""Grouped-GEMM prefill (mqh_moe_prefill) against the oracle.

The oracle is the reference's run_moe_sequence arithmetic (moe_layer.py:110-195):
every (token, slot) pair through moe_quant_expert, ``result[t] += w * y`` in
top-k order (FP32), then ``+ sigmoid(x . g_inp) * shared(x)``.  Tolerance: max
relative error <= 1e-3 per token; the kernels' integer MFMA operands are exact,
so the measured error is FP32 summation noise and is also held to 1e-4.
"""
from __future__ import annotations

import numpy as np
import pytest

from test_capi import workspace_16
from test_gpu_decode import host_expert, make_layer, oracle_layer

pytestmark = pytest.mark.gpu

TOL = 1e-3
TIGHT = 1e-4


def bf16(x: np.ndarray) -> np.ndarray:
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000
    return u.astype(np.uint32).view(np.float32)


def routing(rng, T, E, k):
    ids = np.stack([rng.choice(E, size=k, replace=False) for _ in range(T)]).astype(np.int32)
    w = rng.random((T, k)).astype(np.float32) + 0.05
    return ids, (w / w.sum(axis=1, keepdims=True)).astype(np.float32)


def run_prefill(layer, X, ids, ws, x_bf16=False, use_shared=True, runner=None):
    import torch

    from flash_moe_hip.moe_gpu import MoeRunner

    runner = runner or MoeRunner()
    x = torch.from_numpy(np.ascontiguousarray(X, np.float32)).cuda()
    if x_bf16:
        x = x.to(torch.bfloat16)
    tid = torch.from_numpy(np.ascontiguousarray(ids, np.int32)).cuda()
    tw = torch.from_numpy(np.ascontiguousarray(ws, np.float32)).cuda()
    y = runner.prefill(layer, x, tid, tw, use_shared=use_shared)
    return y.cpu().numpy(), runner.status()


def check(oracle_mod, layer, host, shared, X, ids, ws, got, label):
    worst = 0.0
    for t in range(X.shape[0]):
        want = oracle_layer(oracle_mod, layer, host, shared, X[t], list(ids[t]), list(ws[t]))
        worst = max(worst, oracle_mod.max_relative_error(got[t], want))
    print(f"  {label}: max rel err {worst:.3e}", flush=True)
    assert worst <= TOL
    assert worst <= TIGHT
    return worst


@pytest.fixture(scope="module")
def bench_shape_layer(hip):
    # 16 experts of the benchmark shape: gate/up Q4_K [512x2048], down Q6_K, shared the same
    types = {"gate": 12, "up": 12, "down": 14}
    return make_layer(11, 16, 2048, 512, types, shared_types=types)


@pytest.mark.parametrize("x_bf16", [True, False], ids=["bf16", "fp32"])
def test_prefill_bench_shape(bench_shape_layer, oracle_mod, x_bf16):
    layer, host, shared = bench_shape_layer
    rng = np.random.default_rng(3)
    T = 40
    X = rng.standard_normal((T, 2048)).astype(np.float32)
    if x_bf16:
        X = bf16(X)
    ids, ws = routing(rng, T, 16, 8)
    print(f"prefill T={T} E=16 top8 bf16={x_bf16}", flush=True)
    got, st = run_prefill(layer, X, ids, ws, x_bf16=x_bf16)
    assert st == 0
    check(oracle_mod, layer, host, shared, X, ids, ws, got, "bench shape")


@pytest.mark.parametrize("types", [(11, 11), (13, 12), (14, 14), (12, 13), (11, 14), (12, 11)])
# (intermediate 256 .. 2048: 4 .. 32 row chunks, so one to fifteen two-chunk
# workgroups a tile ahead of the one-chunk ones in the gate/up launch)
@pytest.mark.parametrize("shape", [(256, 256), (512, 1024), (1024, 256), (256, 2048), (2048, 1024)])
def test_prefill_type_pairs(oracle_mod, hip, types, shape):
    gt, dt = types
    H, I = shape
    kinds = {"gate": gt, "up": gt, "down": dt}
    layer, host, shared = make_layer(100 + gt + dt + H // 256 + I, 8, H, I, kinds, shared_types=kinds)
    rng = np.random.default_rng(gt * dt + H + I)
    T = 21
    X = rng.standard_normal((T, H)).astype(np.float32)
    ids, ws = routing(rng, T, 8, 3)
    print(f"prefill types={types} H={H} I={I} T={T}", flush=True)
    got, st = run_prefill(layer, X, ids, ws)
    assert st == 0
    check(oracle_mod, layer, host, shared, X, ids, ws, got, f"types {types} shape {shape}")


def test_prefill_multi_tile_experts_and_repeats(oracle_mod, hip):
    """More than 16 tokens per expert (several tiles per expert), the same
    workspace reused for a larger then a smaller prompt."""
    from flash_moe_hip.moe_gpu import MoeRunner

    kinds = {"gate": 12, "up": 12, "down": 14}
    layer, host, shared = make_layer(21, 4, 512, 256, kinds, shared_types=kinds)
    runner = MoeRunner()
    rng = np.random.default_rng(8)
    for T in (70, 9):
        X = rng.standard_normal((T, 512)).astype(np.float32)
        ids, ws = routing(rng, T, 4, 2)
        print(f"prefill multi-tile T={T}", flush=True)
        got, st = run_prefill(layer, X, ids, ws, runner=runner)
        assert st == 0
        check(oracle_mod, layer, host, shared, X, ids, ws, got, f"T={T}")


def test_prefill_single_token_matches_decode(bench_shape_layer, oracle_mod):
    import torch

    from flash_moe_hip.moe_gpu import MoeRunner

    layer, host, shared = bench_shape_layer
    rng = np.random.default_rng(4)
    X = rng.standard_normal((1, 2048)).astype(np.float32)
    ids, ws = routing(rng, 1, 16, 8)
    got, st = run_prefill(layer, X, ids, ws)
    assert st == 0
    check(oracle_mod, layer, host, shared, X, ids, ws, got, "T=1")
    runner = MoeRunner()
    y = runner.decode(layer, torch.from_numpy(X).cuda(), torch.from_numpy(ids).cuda(),
                      torch.from_numpy(ws).cuda()).cpu().numpy()
    assert oracle_mod.max_relative_error(got[0], y[0]) <= TIGHT


def test_prefill_without_shared_and_without_gate(oracle_mod, hip):
    kinds = {"gate": 14, "up": 14, "down": 12}
    layer, host, shared = make_layer(31, 8, 256, 512, kinds, shared_types=kinds)
    rng = np.random.default_rng(9)
    T = 17
    X = rng.standard_normal((T, 256)).astype(np.float32)
    ids, ws = routing(rng, T, 8, 4)
    got, st = run_prefill(layer, X, ids, ws, use_shared=False)
    assert st == 0
    check(oracle_mod, layer, host, None, X, ids, ws, got, "no shared")
    # shared expert without the sigmoid gate vector: scale 1
    layer.shared.gate_inp = None
    shared_nogate = dict(shared)
    got, st = run_prefill(layer, X, ids, ws)
    assert st == 0
    worst = 0.0
    for t in range(T):
        outs = [oracle_mod.expert_forward(host_expert(host, layer, e), layer.types, X[t], 256, 512) for e in ids[t]]
        sh = oracle_mod.expert_forward({r: shared_nogate[r] for r in ("gate", "up", "down")}, kinds, X[t], 256, 512)
        want = oracle_mod.combine(outs, list(ws[t]), sh)
        worst = max(worst, oracle_mod.max_relative_error(got[t], want))
    print(f"  shared without gate: max rel err {worst:.3e}", flush=True)
    assert worst <= TIGHT


def test_prefill_shared_of_other_type_goes_through_decode(oracle_mod, hip):
    kinds = {"gate": 12, "up": 12, "down": 14}
    sh_kinds = {"gate": 14, "up": 14, "down": 14}
    layer, host, shared = make_layer(41, 8, 512, 256, kinds, shared_types=sh_kinds, sh_I=512)
    rng = np.random.default_rng(10)
    T = 12
    X = rng.standard_normal((T, 512)).astype(np.float32)
    ids, ws = routing(rng, T, 8, 2)
    got, st = run_prefill(layer, X, ids, ws)
    assert st == 0
    check(oracle_mod, layer, host, shared, X, ids, ws, got, "shared via decode")


def test_prefill_bad_expert_id_flags(oracle_mod, hip):
    kinds = {"gate": 12, "up": 12, "down": 14}
    layer, host, shared = make_layer(51, 8, 256, 256, kinds, shared_types=kinds)
    rng = np.random.default_rng(12)
    T = 5
    X = rng.standard_normal((T, 256)).astype(np.float32)
    ids, ws = routing(rng, T, 8, 2)
    ids[2, 1] = 8          # out of range
    got, st = run_prefill(layer, X, ids, ws)
    assert st == -9
    # the valid tokens are still right
    for t in (0, 1, 3, 4):
        want = oracle_layer(oracle_mod, layer, host, shared, X[t], list(ids[t]), list(ws[t]))
        assert oracle_mod.max_relative_error(got[t], want) <= TIGHT


def test_backend_moe_tokens_uses_prefill(oracle_mod, hip):
    """run_moe_sequence through HipExpertBackend.moe_tokens on a multi-token prompt."""
    from flash_moe_hip.backend import HipExpertBackend
    from flash_moe_hip.moe_layer import run_moe_sequence
    from flash_moe_hip.shared_expert import SharedExpert

    kinds = {"gate": 12, "up": 12, "down": 14}
    layer, host, shared = make_layer(61, 16, 512, 256, kinds, shared_types=kinds)
    rng = np.random.default_rng(13)
    W = (rng.standard_normal((512, 16)) * 0.05).astype(np.float32)

    class Router:
        def route(self, x):
            return oracle_mod.route(x, W, 4)

    backend = HipExpertBackend({0: layer})
    sh = SharedExpert.from_backend(backend)
    X = rng.standard_normal((24, 512)).astype(np.float32)
    got = run_moe_sequence(0, X, Router(), backend, 512, 256, shared_expert=sh)
    worst = 0.0
    for t in range(24):
        ids, ws = oracle_mod.route(X[t], W, 4)
        want = oracle_layer(oracle_mod, layer, host, shared, X[t], ids, ws)
        worst = max(worst, oracle_mod.max_relative_error(got[t], want))
    print(f"  run_moe_sequence via prefill: max rel err {worst:.3e}", flush=True)
    assert worst <= TIGHT


def _sweep_case(seed):
    rng = np.random.default_rng(5000 + seed)
    gt, dt = (int(v) for v in rng.choice([11, 12, 13, 14], 2))
    T = int(rng.choice([5, 17, 33]))
    H = int(rng.choice([256, 512, 1024]))
    I = int(rng.choice([256, 512]))
    E = int(rng.choice([8, 32, 96]))
    k = int(rng.choice([1, 3, 8]))
    sh = str(rng.choice(["none", "same", "q6k"]))
    return gt, dt, T, H, I, E, k, sh, bool(rng.integers(2))


@pytest.mark.parametrize("seed", range(12))
def test_prefill_sweep(oracle_mod, hip, seed):
    """Seeded prefill cases with ragged token counts (the route pass stages four
    tokens a workgroup and cuts 16-token tiles, so 5, 17 and 33 tokens leave
    partial staging groups and tiles), BF16 or FP32 tokens, every prefill type
    as gate/up and as down, with no shared expert, one of the routed types or a
    Q6_K one: every token against the oracle."""
    gt, dt, T, H, I, E, k, sh, xb = _sweep_case(seed)
    kinds = {"gate": gt, "up": gt, "down": dt}
    st = None if sh == "none" else (kinds if sh == "same" else {"gate": 14, "up": 14, "down": 14})
    layer, host, shared = make_layer(7000 + seed, E, H, I, kinds, shared_types=st)
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((T, H)).astype(np.float32)
    if xb:
        X = bf16(X)
    ids, ws = routing(rng, T, E, k)
    print(f"prefill sweep {seed}: types {gt}/{dt} T={T} H={H} I={I} E={E} k={k} shared={sh} bf16={xb}", flush=True)
    got, st_ = run_prefill(layer, X, ids, ws, x_bf16=xb)
    assert st_ == 0
    check(oracle_mod, layer, host, shared, X, ids, ws, got, f"sweep {seed}")


@pytest.mark.parametrize("routed", [(11, 11), (12, 8), (13, 14), (12, 11), (11, 8)])
@pytest.mark.parametrize("shape", [(256, 256), (512, 1024), (1024, 2048), (2048, 512)])
def test_prefill_q6k_shared_beside_other_routed_types(oracle_mod, hip, routed, shape):
    """A Q6_K shared expert in the grouped launches beside routed experts of
    other types (its tiles run their own instance of the GEMM body), and Q8_0
    down projections (per-block scales applied per MFMA step): every token
    against the oracle, BF16 tokens for even intermediate sizes (the high
    plane only) and FP32 tokens for the others (both planes)."""
    from flash_moe_hip.moe_gpu import MoeRunner

    gt, dt = routed
    H, I = shape
    kinds = {"gate": gt, "up": gt, "down": dt}
    q6 = {"gate": 14, "up": 14, "down": 14}
    layer, host, shared = make_layer(700 + gt + dt + H // 256 + I, 12, H, I, kinds, shared_types=q6)
    assert MoeRunner._shared_in_prefill(layer)
    rng = np.random.default_rng(gt * 31 + dt + H + I)
    T = 37
    x_bf16 = (I // 256) % 2 == 0
    X = rng.standard_normal((T, H)).astype(np.float32)
    if x_bf16:
        X = bf16(X)
    ids, ws = routing(rng, T, 12, 4)
    print(f"prefill routed={routed} + Q6_K shared H={H} I={I} T={T} bf16={x_bf16}", flush=True)
    got, st = run_prefill(layer, X, ids, ws, x_bf16=x_bf16)
    assert st == 0
    check(oracle_mod, layer, host, shared, X, ids, ws, got, f"routed {routed} shape {shape}")


@pytest.mark.parametrize("shape", [(512, 256), (2048, 1024)])
def test_prefill_q8_0_down_without_shared(oracle_mod, hip, shape):
    """Q8_0 down projections with no shared expert, and the shared expert
    switched off on a layer that has one (use_shared=False)."""
    H, I = shape
    kinds = {"gate": 12, "up": 12, "down": 8}
    layer, host, shared = make_layer(750 + H + I, 6, H, I, kinds, shared_types={"gate": 14, "up": 14, "down": 14})
    rng = np.random.default_rng(H + I)
    T = 23
    X = rng.standard_normal((T, H)).astype(np.float32)
    ids, ws = routing(rng, T, 6, 3)
    print(f"prefill Q8_0 down, no shared, H={H} I={I}", flush=True)
    got, st = run_prefill(layer, X, ids, ws, use_shared=False)
    assert st == 0
    check(oracle_mod, layer, host, None, X, ids, ws, got, f"Q8_0 down {shape}")


@pytest.mark.parametrize("types,sh,shape,x_bf16", [
    ((12, 14), "same", (2048, 512), True),
    ((12, 8), "none", (512, 256), False),    # (Q8_0 down projections stay on 16-token tiles)
    ((11, 11), "q6k", (1024, 512), False),
    ((13, 12), "same", (256, 1024), False),
    ((14, 13), "same", (512, 512), True),
    ((11, 14), "q6k", (512, 2048), True),
    ((13, 14), "none", (256, 256), True),
    ((12, 12), "q6k", (1024, 256), True),    # gate, up and down of another type than the shared expert's
    ((13, 13), "q6k", (512, 512), False),
    ((11, 12), "same", (2048, 256), False),  # FP32 tokens of the largest hidden size
])
def test_prefill_wide_tiles(oracle_mod, hip, types, sh, shape, x_bf16):
    """Many tokens per expert (64-token tiles): experts of 0, 1, 16, 17, 32, 33,
    62 and 161 tokens per 161, so every number of column blocks, full and with
    one column, and one super-block of hidden or intermediate up to eight.  The
    161 tokens are checked against the oracle; the prompt repeats them until its
    size is the wide tiles' (every repetition's rows are the same bits: a pair's
    result does not depend on its column).  Alone they run on 16-token tiles, with
    the same bits."""
    (gt, dt), (H, I) = types, shape
    kinds = {"gate": gt, "up": gt, "down": dt}
    st = {"none": None, "same": kinds, "q6k": {"gate": 14, "up": 14, "down": 14}}[sh]
    layer, host, shared = make_layer(7100 + gt + dt + H, 8, H, I, kinds, shared_types=st)
    rng = np.random.default_rng(gt * dt + H)
    first = np.repeat([1, 2, 3, 4, 5, 6], [1, 16, 17, 32, 33, 62])
    T = len(first)
    first = rng.permutation(first)
    # the repetitions' second pairs go to expert 0 and theirs, too, to 7: the
    # other experts keep the counts above
    reps = 100 if H == 256 else 20 if I == 256 else 13
    X1 = rng.standard_normal((T, H)).astype(np.float32) * rng.uniform(0.01, 30, (T, 1)).astype(np.float32)
    X = np.concatenate([X1] * reps)
    ids = np.zeros((T * reps, 2), np.int64)
    ids[:T, 1] = first
    ids[T:, 1] = 7
    ws = rng.dirichlet(np.ones(2), size=T * reps).astype(np.float32)
    ws[2 * T:] = np.tile(ws[T:2 * T], (reps - 2, 1))
    if x_bf16:
        X = bf16(X)
    print(f"prefill wide tiles types={types} shared={sh} H={H} I={I} T={len(X)} bf16={x_bf16}", flush=True)
    got, status = run_prefill(layer, X, ids, ws, x_bf16=x_bf16)
    assert status == 0
    assert hip.mqh_last_prefill_tile() == (16 if dt == 8 else 64)
    check(oracle_mod, layer, host, shared, X[:T], ids[:T], ws[:T], got[:T], f"wide {types} {shape}")
    check(oracle_mod, layer, host, shared, X[T:T + 9], ids[T:T + 9], ws[T:T + 9], got[T:T + 9], "expert 7")
    for r in range(2, reps):
        np.testing.assert_array_equal(got[r * T:(r + 1) * T], got[T:2 * T])
    alone, status = run_prefill(layer, X[:T], ids[:T], ws[:T], x_bf16=x_bf16)
    assert status == 0 and hip.mqh_last_prefill_tile() == 16
    np.testing.assert_array_equal(got[:T], alone)


def test_prefill_wide_tiles_out_of_range_ids(hip):
    """Ids out of range on 64-token tiles are flagged and contribute nothing: the
    same bits as on 16-token tiles, with tokens of no, one and two such ids."""
    t = {"gate": 12, "up": 12, "down": 14}
    E, H, I, T, n = 8, 512, 512, 2700, 160
    layer, _, _ = make_layer(7300, E, H, I, t, shared_types=t)
    rng = np.random.default_rng(7300)
    X = rng.standard_normal((T, H)).astype(np.float32)
    ids = rng.integers(-2, E + 2, size=(T, 2)).astype(np.int32)
    ws = rng.dirichlet(np.ones(2), size=T).astype(np.float32)
    bad = ((ids < 0) | (ids >= E)).sum(axis=1)
    assert all((bad[:n] == i).any() for i in range(3))
    print("prefill wide tiles: ids out of range", flush=True)
    got, status = run_prefill(layer, X, ids, ws)
    assert status == -9 and hip.mqh_last_prefill_tile() == 64
    alone, status = run_prefill(layer, X[:n], ids[:n], ws[:n])
    assert status == -9 and hip.mqh_last_prefill_tile() == 16
    np.testing.assert_array_equal(got[:n], alone)


def test_prefill_in_a_16_token_workspace(hip):
    """A prompt whose size is the 64-token tiles' runs in a workspace that only
    has room for 16-token tiles, on those, with the same bits; one byte less is
    refused."""
    import torch

    from flash_moe_hip.layer_store import ExpertLayer
    from flash_moe_hip.moe_gpu import MoeRunner

    t = {"gate": 12, "up": 12, "down": 14}
    T, k, E, H, I = 1100, 4, 8, 2048, 512
    layer = ExpertLayer.synthetic(t, E, H, I, seed=9, shared_types=t)
    g = torch.Generator(device="cuda").manual_seed(9)
    x = torch.randn(T, H, generator=g, device="cuda")
    top = torch.topk(torch.randn(T, E, generator=g, device="cuda"), k, dim=1)
    ids, w = top.indices.int().contiguous(), torch.softmax(top.values, dim=1).contiguous()
    print("prefill in a 16-token workspace", flush=True)
    want = MoeRunner().prefill(layer, x, ids, w)
    assert hip.mqh_last_prefill_tile() == 64
    need = workspace_16(T, k, E, H, I, 1)
    assert need < hip.mqh_moe_prefill_workspace_bytes(T, k, E, H, I, 1)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    assert hip.mqh_workspace_init(ws.data_ptr(), need, stream) == 0
    y = torch.empty(T, H, device="cuda")
    sh, d = layer.shared, layer.tensors

    def call(nbytes):
        return hip.mqh_moe_prefill(
            12, d["gate"].data_ptr(), 12, d["up"].data_ptr(), 14, d["down"].data_ptr(), E, H, I,
            12, sh.gate.data_ptr(), 12, sh.up.data_ptr(), 14, sh.down.data_ptr(), I, sh.gate_inp.data_ptr(),
            x.data_ptr(), 0, T, ids.data_ptr(), w.data_ptr(), k, y.data_ptr(), ws.data_ptr(), nbytes, stream)

    assert call(need - 1) == -6
    assert call(need) == 0
    assert hip.mqh_last_prefill_tile() == 16
    assert hip.mqh_status(ws.data_ptr(), stream) == 0
    assert torch.equal(y, want)


@pytest.mark.parametrize("types,sh,shape,E,k,T,tile", [
    # (hidden 2048 and 256, either side of the pairs an expert and of the amount of work)
    ((12, 14), True, (2048, 512), 256, 8, 4096, 64),
    ((12, 14), True, (2048, 512), 256, 8, 909, 16),
    ((12, 14), True, (256, 512), 256, 8, 914, 16),
    ((13, 13), False, (256, 2048), 8, 2, 4096, 16),
    ((12, 14), True, (256, 256), 1, 0, 4096, 16),
    ((11, 11), True, (256, 512), 16, 8, 4096, 64),
    # amounts of work of each type
    ((12, 14), True, (512, 256), 60, 4, 1640, 16),
    ((12, 14), True, (1024, 512), 8, 2, 2048, 64),
    ((13, 13), False, (512, 512), 60, 8, 768, 16),
    ((13, 13), False, (512, 512), 60, 8, 1536, 64),
    ((11, 11), False, (512, 256), 60, 8, 520, 16),
    ((11, 11), False, (512, 512), 60, 8, 768, 64),
    ((14, 14), False, (512, 256), 60, 8, 520, 64),
    ((14, 14), True, (512, 256), 60, 8, 480, 16),     # (a shared expert asks for a quarter more)
    ((14, 14), True, (512, 256), 60, 8, 600, 64),
    ((14, 14), False, (2048, 256), 16, 8, 512, 64),
    ((12, 8), False, (2048, 512), 8, 2, 4096, 16),
])
def test_prefill_tile_width(hip, types, sh, shape, E, k, T, tile):
    """The tile width of a prompt follows the matrix size and type as well as its
    length: where the 64-token tiles measured slower the 16-token ones run."""
    import torch

    from flash_moe_hip.layer_store import ExpertLayer
    from flash_moe_hip.moe_gpu import MoeRunner

    (gt, dt), (H, I) = types, shape
    t = {"gate": gt, "up": gt, "down": dt}
    layer = ExpertLayer.synthetic(t, E, H, I, seed=T, shared_types=t if sh else None)
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(T, H, generator=g, device="cuda").to(torch.bfloat16)
    top = torch.topk(torch.randn(T, E, generator=g, device="cuda"), k, dim=1)
    ids, w = top.indices.int().contiguous(), torch.softmax(top.values, dim=1).contiguous()
    print(f"prefill tile width {types} H={H} I={I} E={E} k={k} T={T}", flush=True)
    runner = MoeRunner()
    y = runner.prefill(layer, x, ids, w)
    # (a new runner's workspace is what the query call says, to the byte)
    assert runner._ws.numel() == hip.mqh_moe_prefill_workspace_bytes(T, k, E, H, I, int(sh))
    assert runner.status() == 0 and bool(torch.isfinite(y).all())
    assert hip.mqh_last_prefill_tile() == tile
