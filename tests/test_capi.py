"""The C ABI library loads and exports what include/moe_quant_hip.h declares (CPU only).

Only host-side logic is called here: type queries and the argument validation
that returns before any HIP call (status codes of moe_quant_dot.cpp:181-188
and dequant_k.cpp:352-355).  No kernel runs.
"""
from __future__ import annotations

import ctypes as C
import re

import numpy as np
import pytest

from conftest import ROOT

HEADER = ROOT / "include" / "moe_quant_hip.h"


def declared_functions() -> list[str]:
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    return re.findall(r"^\s*(?:int|int64_t|void)\s+\**(\w+)\s*\(", text, flags=re.M)


@pytest.fixture(scope="module")
def lib():
    from flash_moe_hip import _lib

    return _lib.load()


def test_header_declares_the_binding_list():
    from flash_moe_hip import _lib

    assert sorted(declared_functions()) == sorted(_lib.EXPORTS)


def test_every_declared_symbol_is_exported(lib):
    for name in declared_functions():
        assert hasattr(lib, name), name


def test_type_queries(lib):
    expect = {8: 32, 11: 256, 12: 256, 13: 256, 14: 256}
    for t in range(0, 40):
        assert lib.dequant_k_supported(t) == (1 if t in expect else 0)
        assert lib.dequant_k_block_size(t) == expect.get(t, 0)


def test_dequant_k_rejects_bad_arguments(lib):
    buf = np.zeros(144, np.uint8)
    out = np.zeros(256, np.float32)
    assert lib.dequant_k(99, buf.ctypes.data, out.ctypes.data, 256, 0) == -1
    assert lib.dequant_k(12, None, out.ctypes.data, 256, 0) == -1
    assert lib.dequant_k(12, buf.ctypes.data, None, 256, 0) == -1
    assert lib.dequant_k(12, buf.ctypes.data, out.ctypes.data, 0, 0) == -1
    assert lib.dequant_k(12, buf.ctypes.data, out.ctypes.data, 257, 0) == -1


def test_moe_quant_expert_validation_codes(lib):
    H = I = 256
    g = np.zeros(I * 144, np.uint8)
    d = np.zeros(H * 210, np.uint8)
    x = np.zeros(H, np.float32)
    y = np.zeros(H, np.float32)

    def call(gt=12, gb=g.nbytes, ut=12, ub=g.nbytes, dt=14, db=d.nbytes, h=H, i=I, f16=0, gp=g, xp=x):
        return lib.moe_quant_expert(gt, None if gp is None else gp.ctypes.data, gb, ut, g.ctypes.data, ub,
                                    dt, d.ctypes.data, db, None if xp is None else xp.ctypes.data, h, i,
                                    y.ctypes.data, f16)

    assert call(gp=None) == -1
    assert call(xp=None) == -1
    assert call(h=0) == -1
    assert call(i=-1) == -1
    assert call(h=65537) == -1
    assert call(f16=2) == -1
    assert call(gt=999) == -2
    assert call(dt=7) == -2
    assert call(h=288) == -2            # 288 % 256
    assert call(gb=g.nbytes - 1) == -3
    assert call(db=d.nbytes + 210) == -3


def test_device_entry_validation(lib):
    assert lib.mqh_moe_workspace_bytes(0, 8, 512, 512) == -1
    assert lib.mqh_moe_workspace_bytes(1, 0, 512, 0) == -1
    ws = lib.mqh_moe_workspace_bytes(16, 8, 512, 512)
    assert ws >= 16 * 9 * 512 * 4 and ws % 256 == 0
    assert lib.mqh_moe_workspace_bytes(1, 0, 0, 512) > 0          # shared expert only
    assert lib.mqh_dequant(99, C.c_void_p(16), C.c_void_p(16), 256, 1, None) == -1
    assert lib.mqh_dequant(12, C.c_void_p(16), C.c_void_p(24), 256, 1, None) == -1   # dst not 16-B aligned
    args = [12, C.c_void_p(256), 12, C.c_void_p(256), 14, C.c_void_p(256), 256, 2048, 512,
            0, None, 0, None, 0, None, 0, None,
            C.c_void_p(256), 1, C.c_void_p(256), C.c_void_p(256), 8,
            C.c_void_p(256), 0, C.c_void_p(256), 1 << 20, None]
    bad_type = list(args)
    bad_type[0] = 99
    assert lib.mqh_moe_decode(*bad_type) == -2
    bad_k = list(args)
    bad_k[21] = 0                       # top_k 0 without a shared expert
    assert lib.mqh_moe_decode(*bad_k) == -1
    small_ws = list(args)
    small_ws[25] = 64
    assert lib.mqh_moe_decode(*small_ws) == -6


def test_route_validation(lib):
    p = C.c_void_p(256)
    ok = dict(x=p, t=1, h=2048, w=p, e=128, k=8, s=p, ids=p, wts=p)

    def call(**kw):
        a = {**ok, **kw}
        return lib.mqh_route(a["x"], a["t"], a["h"], a["w"], a["e"], a["k"], a["s"], a["ids"], a["wts"], None)

    assert call(x=None) == -1
    assert call(w=None) == -1
    assert call(s=None) == -1
    assert call(ids=None) == -1
    assert call(wts=None) == -1
    assert call(t=0) == -1
    assert call(h=0) == -1
    assert call(h=2046) == -1                 # rows are read 16 bytes at a time
    assert call(x=C.c_void_p(264)) == -1      # x not 16-byte aligned
    assert call(w=C.c_void_p(260)) == -1
    assert call(e=1025) == -1                 # at most 16 scores per lane
    assert call(k=0) == -1
    assert call(k=65) == -1                   # one selected score per lane
    assert call(e=4, k=5) == -1               # more slots than experts


def test_delta_heads_validation(lib):
    p = C.c_void_p(256)
    ok = dict(st=p, q=p, k=p, v=p, b=p, g=p, o=p, h=32, dk=128, dv=128)

    def call(fn, **kw):
        a = {**ok, **kw}
        args = [a["st"], a["q"], a["k"], a["v"], a["b"], a["g"], a["o"], a["h"], a["dk"], a["dv"]]
        return fn(*args) if fn is lib.moe_delta_heads else fn(*args, None, None)

    for fn in (lib.moe_delta_heads, lib.mqh_delta_heads):
        for key in ("st", "q", "k", "v", "b", "g", "o"):
            assert call(fn, **{key: None}) == -1
        for kw in (dict(h=0), dict(h=257), dict(dk=0), dict(dk=1025), dict(dv=0), dict(dv=1025)):
            assert call(fn, **kw) == -1          # moe_delta.cpp:21-24


def test_iq4_nl_stays_outside_the_reference_contracts(lib):
    # dequant_k and moe_quant_expert keep the reference's five types
    # (dequant_k.cpp:342-348); IQ4_NL has its own exports and the device paths
    assert lib.dequant_k_supported(20) == 0
    assert lib.dequant_k_block_size(20) == 0
    buf = np.zeros(18, np.uint8)
    out = np.zeros(32, np.float32)
    assert lib.dequant_k(20, buf.ctypes.data, out.ctypes.data, 32, 0) == -1


def test_word_calls_take_the_same_arguments(lib):
    """The calls with their arguments as 64-bit words validate as the plain ones
    do: each word reaches its argument (host-side statuses, no kernel runs)."""
    import struct

    bufs = [np.zeros(1 << 16, np.uint8) for _ in range(12)]
    p = [b.ctypes.data + (-b.ctypes.data) % 256 for b in bufs]

    def decode(**kw):
        a = dict(gt=12, g=p[0], ut=12, u=p[1], dt=14, d=p[2], E=4, H=256, I=256, sgt=12, sg=p[3], sut=12, su=p[4],
                 sdt=14, sd=p[5], sI=256, sgi=p[6], x=p[7], T=1, ids=p[8], w=p[9], k=2, y=p[10], f=0, ws=p[11], wb=0,
                 st=0)
        a.update(kw)
        v = list(a.values())
        plain = lib.mqh_moe_decode(*[None if i in (1, 3, 5, 10, 12, 14, 16, 17, 19, 20, 22, 24) and q == 0 else q
                                     for i, q in enumerate(v)])
        assert lib.mqh_moe_decode_words(struct.pack("27q", *v)) == plain, kw
        r = v[:18] + [v[18], p[9], v[21], p[6], v[19], v[20], v[22], v[23], v[24], v[25], v[26]]
        plain_r = lib.mqh_moe_decode_routed(*[None if i in (1, 3, 5, 10, 12, 14, 16, 17, 22, 23, 24, 26) and q == 0
                                              else q for i, q in enumerate(r)])
        assert lib.mqh_moe_decode_routed_words(struct.pack("29q", *r)) == plain_r, kw
        return plain

    assert decode() == -6   # every argument is right but the workspace's size
    assert decode(gt=99) == -2 and decode(ut=99) == -2 and decode(dt=99) == -2 and decode(sdt=99) == -2
    for name in ("g", "u", "d", "su", "sd", "x", "ids", "w", "y", "ws"):
        assert decode(**{name: 0}) == -1, name
    assert decode(H=100) == -2 and decode(I=100) == -2 and decode(sI=100) == -2 and decode(E=0) == -1
    assert decode(T=0) == -1 and decode(k=65) == -1 and decode(f=2) == -1 and decode(g=p[0] + 1) == -1
    assert lib.mqh_moe_decode_words(None) == -1 and lib.mqh_moe_decode_routed_words(None) == -1


def test_prefill_workspace_does_for_every_shorter_prompt(lib):
    """The workspace of a prompt is at least that of any shorter one, across the
    sizes at which the tile width changes (4096 pairs, 32 tokens an expert, and
    2^32 plane values, past which the 16-token tiles are back)."""
    for k, E, H, I, sh in ((8, 256, 2048, 512, 1), (2, 8, 256, 2048, 0), (8, 60, 512, 256, 1), (0, 1, 2048, 1024, 1)):
        sizes = sorted({1, 2, 15, 16, 17, 60, 127, 128, 455, 456, 512, 913, 914, 1027, 2048, 4096, 8192, 65535, 200000,
                        233016, 233017, 233018, 262144, 524288, 1048576, 2097152, 2200000})
        need = [lib.mqh_moe_prefill_workspace_bytes(T, k, E, H, I, sh) for T in sizes]
        assert need[0] > 0 and all(a <= b for a, b in zip(need, need[1:])), (k, E, H, I, sh)


def workspace_16(T, k, E, H, I, has_shared):
    """Bytes the prefill kernels of 16-token tiles need: flags, per-token gates,
    tile records and their columns, activations and pair outputs, token planes."""
    def up(n):
        return (n + 255) // 256 * 256

    S = k + has_shared
    tiles = max(min(E, T * k) + -(-T * k // 16) + (-(-T // 16) if has_shared else 0), 1)
    return (256 + up(4 * T) + up(16 * tiles) + 256 + 2 * up(64 * tiles) + up(4 * T * S * I) + up(4 * T * S * H)
            + 2 * up(2 * T * H) + up(T * (H // 32) * 4) + up(4 * T))


@pytest.mark.parametrize("k,E,H,I,sh,last", [
    (8, 256, 2048, 512, 1, 913),      # 32 pairs an expert
    (8, 60, 512, 256, 1, 503),        # pairs cbrt(pairs an expert) hidden inter
    (8, 8, 2048, 2048, 0, 511),       # 4096 pairs
    (2, 8, 256, 2048, 0, 5421),       # pairs cbrt(pairs an expert)
    (8, 256, 256, 256, 1, 2868),
])
def test_prefill_workspace_of_prompts_below_the_wide_tiles(lib, k, E, H, I, sh, last):
    """Only prompts that some type takes 64-token tiles for pay for their planes."""
    for T in (1, 3, last // 2, last):
        assert lib.mqh_moe_prefill_workspace_bytes(T, k, E, H, I, sh) == workspace_16(T, k, E, H, I, sh), T
    T, S = last + 1, k + sh
    planes = T * S * (4 * I + 4 * (I // 32) + 4)
    assert lib.mqh_moe_prefill_workspace_bytes(T, k, E, H, I, sh) >= workspace_16(T, k, E, H, I, sh) + planes // 2


def test_prefill_workspace_past_the_wide_tiles(lib):
    """A prompt of 2^32 plane values or more has room for the longest one below."""
    k, E, H, I, sh = 8, 256, 2048, 512, 1
    last = (2 ** 32 - 1) // H // (k + sh)
    need = [lib.mqh_moe_prefill_workspace_bytes(T, k, E, H, I, sh) for T in (last, last + 1, 2 * last)]
    assert need[1] == need[0] > workspace_16(last + 1, k, E, H, I, sh)
    assert need[2] == workspace_16(2 * last, k, E, H, I, sh)


def test_cpu_devices_are_refused():
    """Decode and DeltaNet calls on a CPU device raise before any launch."""
    import torch
    from flash_moe_hip.moe_gpu import MoeRunner
    from flash_moe_hip.native_expert import DeltaState

    state = DeltaState(2, 4, 4, device="cpu")
    q, v, b = torch.zeros(2, 4), torch.zeros(2, 4), torch.zeros(2)
    with pytest.raises(ValueError):
        state.step(q, q, v, b, b)
    runner = MoeRunner(device="cpu")
    with pytest.raises(ValueError):
        runner.decode(None, None, None, None)
    with pytest.raises(ValueError):
        runner.decode_routed(None, None, 1)


def test_current_stream_without_the_private_accessor(monkeypatch):
    """The current stream's handle comes from torch's private accessor where there
    is one, else from the public call."""
    from types import SimpleNamespace

    import torch
    from flash_moe_hip import _lib

    monkeypatch.setattr(torch.cuda, "current_stream", lambda i: SimpleNamespace(cuda_stream=100 + i))
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda i: 200 + i, raising=False)
    assert _lib.stream_accessor()(3) == 203
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream")
    assert _lib.stream_accessor()(3) == 103
