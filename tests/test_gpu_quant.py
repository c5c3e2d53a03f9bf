"""GPU parity: per-tensor fp8 pair (v1 and v2 modules) against the C oracle,
bit-exact for the partials, the scale and every e4m3 byte."""
import ctypes
import json
import os

import numpy as np
import pytest
import torch

import k3h
import oracle as O
from k3data import from_dev, normal_bf16, rng, to_dev

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


@pytest.mark.parametrize("v2", [True, False])
@pytest.mark.parametrize("n,nb", [(16384 * 7168, 2048), (7168 * 40 + 5, 64), (13, 4), (4096, 2048)])
def test_quant_fp8_tensor(ctx, v2, n, nb):
    print(f"[case] quant_fp8_tensor v2={v2} n={n} nb={nb}", flush=True)
    g = rng(1100 + n % 97)
    x = normal_bf16(g, (n,), outlier_p=0.001)
    want_p = O.quant_fp8_amax(x, n, nb, v2=v2)
    want_y, want_s = O.quant_fp8_apply(x, n, want_p, nb)
    xd = to_dev(x)
    y = torch.empty(n + 8, dtype=torch.uint8, device="cuda")
    s = torch.empty(1, dtype=torch.float32, device="cuda")
    p = torch.empty(nb, dtype=torch.float32, device="cuda")
    ctx.quant_fp8_tensor(xd, y, s, p, n, v2=v2)
    torch.cuda.synchronize()
    assert np.array_equal(from_dev(p), want_p)
    assert from_dev(s)[0] == want_s[0]
    assert np.array_equal(from_dev(y)[:n], want_y)


@pytest.mark.parametrize("v2", [True, False])
def test_quant_fp8_tensor_nan(ctx, v2):
    """NaN inputs of either sign: v1 partials ignore them, v2 partials take the
    |bf16| pattern maximum (a NaN partial, compared as bits), the scale comes
    from the non-NaN partials, and each NaN gives the canonical e4m3 NaN 0x7f."""
    n, nb = 7168 * 8 + 3, 64
    print(f"[case] quant_fp8_tensor NaN v2={v2}", flush=True)
    g = rng(1150)
    x = normal_bf16(g, (n,), outlier_p=0.001)
    nan_at = [5, 1000, 30000, n - 1]
    x[nan_at] = [0x7FC0, 0xFFC1, 0x7F81, 0xFFFF]
    want_p = O.quant_fp8_amax(x, n, nb, v2=v2)
    want_y, want_s = O.quant_fp8_apply(x, n, want_p, nb)
    y = torch.empty(n + 8, dtype=torch.uint8, device="cuda")
    s = torch.empty(1, dtype=torch.float32, device="cuda")
    p = torch.empty(nb, dtype=torch.float32, device="cuda")
    ctx.quant_fp8_tensor(to_dev(x), y, s, p, n, v2=v2)
    torch.cuda.synchronize()
    assert np.array_equal(from_dev(p).view(np.uint32), want_p.view(np.uint32))
    assert from_dev(s).view(np.uint32)[0] == want_s.view(np.uint32)[0]
    got_y = from_dev(y)[:n]
    assert np.array_equal(got_y, want_y)
    assert (got_y[nan_at] == 0x7F).all()


def test_quant_fp8_zero_tensor_scale_one(ctx):
    n = 4096
    x = np.zeros(n, np.uint16)
    y = torch.full((n,), 0x55, dtype=torch.uint8, device="cuda")
    s = torch.empty(1, dtype=torch.float32, device="cuda")
    p = torch.empty(16, dtype=torch.float32, device="cuda")
    ctx.quant_fp8_tensor(to_dev(x), y, s, p, n)
    torch.cuda.synchronize()
    assert from_dev(s)[0] == 1.0 and not from_dev(y).any()


def test_quant_fp8_manifest_op(ctx):
    """ops.quant_fp8_tensor of the default manifest (two launches, grid 2048)."""
    ops = json.load(open(os.path.join(GOLDEN, "manifest_hot_ops.json")))
    n = 4096 * 7168
    g = rng(1200)
    x = normal_bf16(g, (n,), outlier_p=0.001)
    y = torch.empty(n, dtype=torch.uint8, device="cuda")
    s = torch.empty(1, dtype=torch.float32, device="cuda")
    p = torch.empty(2048, dtype=torch.float32, device="cuda")
    k3h.ManifestOp(ctx, "quant_fp8_tensor", ops["quant_fp8_tensor"])([to_dev(x), y, s, p, n], {"tokens": 16384})
    torch.cuda.synchronize()
    want_p = O.quant_fp8_amax(x, n, 2048, v2=True)
    want_y, want_s = O.quant_fp8_apply(x, n, want_p, 2048)
    assert np.array_equal(from_dev(p), want_p)
    assert from_dev(s)[0] == want_s[0]
    assert np.array_equal(from_dev(y), want_y)


def _once(ctx, x, n, spin_ticks):
    """k3h_quant_fp8_mark + k3h_quant_fp8_once launched directly: (y, scale, partials)."""
    y = torch.full((n + 8,), 0x5a, dtype=torch.uint8, device="cuda")
    s = torch.zeros(1, dtype=torch.float32, device="cuda")
    p = torch.zeros(2048, dtype=torch.float32, device="cuda")
    key, stream = "k3_quant_fp8_pair_v2", torch.cuda.current_stream().cuda_stream
    for entry, grid, kinds, vals in (
            ("k3h_quant_fp8_mark", 2, ["buffer"], [p]),
            ("k3h_quant_fp8_once", 256, ["buffer", "buffer", "i32", "buffer", "buffer", "i32"],
             [x, y, n, p, s, spin_ticks])):
        buf = k3h.pack_args(kinds, vals)
        cbuf = ctypes.create_string_buffer(buf, len(buf))
        k3h._check(ctx.L.k3h_launch(ctx.function(key, entry), (ctypes.c_uint32 * 3)(grid, 1, 1),
                                    (ctypes.c_uint32 * 3)(1024, 1, 1), 0, stream,
                                    ctypes.cast(cbuf, ctypes.c_void_p), len(buf)), entry)
    torch.cuda.synchronize()
    return y, s, p


@pytest.mark.parametrize("n,spin", [(4096, 20000), (24 << 20, 20000), (12 << 22, 20000),
                                    ((12 << 22) + 7, 20000), ((12 << 22) + 8, 20000),
                                    ((15 << 22) + 4099, 20000), ((30 << 20) + 13, 0)])
def test_quant_fp8_one_launch(ctx, n, spin):
    """The one-launch form against the amax / apply entries, bit for bit: tensors that fit
    the chip, that fill it exactly (24 vectors per thread) and that are partly read again;
    NaN and -inf among the inputs; with no wait at all (spin 0) every workgroup takes the
    maxima it misses itself."""
    print(f"[case] quant_fp8 one launch n={n} spin={spin}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(1300 + n % 97)
    x = torch.empty(n, device="cuda").normal_(0, 2, generator=g).to(torch.bfloat16)
    x[n // 3], x[n - 1], x[n // 2] = float("nan"), -300.0, -0.0
    nb = 2048
    want_y = torch.full((n + 8,), 0x5a, dtype=torch.uint8, device="cuda")
    want_s = torch.zeros(1, dtype=torch.float32, device="cuda")
    want_p = torch.empty(nb, dtype=torch.float32, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    assert ctx.L.k3h_quant_fp8_amax(ctx.h, stream, 1, x.data_ptr(), n, want_p.data_ptr(), nb) == 0
    assert ctx.L.k3h_quant_fp8_apply(ctx.h, stream, 1, x.data_ptr(), want_y.data_ptr(), n,
                                     want_p.data_ptr(), nb, want_s.data_ptr()) == 0
    y, s, p = _once(ctx, x, n, spin)
    assert torch.equal(p.view(torch.int32), want_p.view(torch.int32))
    assert s.view(torch.int32).item() == want_s.view(torch.int32).item()
    assert torch.equal(y, want_y)


@pytest.mark.parametrize("n", [(24 << 20) - 1, 24 << 20, (24 << 20) + 5])
def test_quant_fp8_tensor_route(ctx, n):
    """The typed call on both sides of the size where it changes to the one-launch form."""
    print(f"[case] quant_fp8_tensor route n={n}", flush=True)
    x = normal_bf16(rng(1400), (n,), outlier_p=0.001)
    want_p = O.quant_fp8_amax(x, n, 2048, v2=True)
    want_y, want_s = O.quant_fp8_apply(x, n, want_p, 2048)
    y = torch.empty(n + 8, dtype=torch.uint8, device="cuda")
    s = torch.empty(1, dtype=torch.float32, device="cuda")
    p = torch.empty(2048, dtype=torch.float32, device="cuda")
    ctx.quant_fp8_tensor(to_dev(x), y, s, p, n)
    torch.cuda.synchronize()
    assert np.array_equal(from_dev(p), want_p) and from_dev(s)[0] == want_s[0]
    assert np.array_equal(from_dev(y)[:n], want_y)


@pytest.mark.parametrize("n", [24 << 20, (15 << 22) + 4099])
def test_quant_fp8_tensor_beside_a_waiting_wave(ctx, n):
    """The one-launch form while one wave of another stream (the arrival wait for a rank that
    never arrives, 20 ms) holds a CU, so that one of its workgroups starts only after others
    have ended: the pair's outputs, and no long wait.  The bound is the 200 us that a
    workgroup would once have waited before it took the missing maxima itself (measured:
    713-770 us then; 55 us at 25 M, 75 us at 63 M now)."""
    print(f"[case] quant_fp8_tensor beside a waiting wave n={n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(1500 + n % 97)
    x = torch.empty(n, device="cuda").normal_(0, 2, generator=g).to(torch.bfloat16)
    nb = 2048
    y, want_y = (torch.full((n + 8,), 0x5a, dtype=torch.uint8, device="cuda") for _ in range(2))
    s, want_s = (torch.zeros(1, dtype=torch.float32, device="cuda") for _ in range(2))
    p, want_p = (torch.empty(nb, dtype=torch.float32, device="cuda") for _ in range(2))
    stream = torch.cuda.current_stream().cuda_stream
    assert ctx.L.k3h_quant_fp8_amax(ctx.h, stream, 1, x.data_ptr(), n, want_p.data_ptr(), nb) == 0
    assert ctx.L.k3h_quant_fp8_apply(ctx.h, stream, 1, x.data_ptr(), want_y.data_ptr(), n,
                                     want_p.data_ptr(), nb, want_s.data_ptr()) == 0
    arrive = k3h.ManifestOp(ctx, "arrive", {
        "params": ["out buffer<u64>", "in buffer<u64>", "i32", "i32", "i32", "out buffer<u32>"],
        "impl": {"launches": [{"module": "k3_rs_arrive_v2+K3_SPIN_US=20000",
                               "entry": "k3h_rs_arrive_mask", "block": [64, 1, 1], "grid": [1, 1, 1]}]}})
    own, peer = (torch.zeros(372, dtype=torch.int64, device="cuda") for _ in range(2))
    fpeer = torch.tensor([own.data_ptr(), peer.data_ptr()], dtype=torch.int64, device="cuda")
    missing = torch.full((1,), -1, dtype=torch.int32, device="cuda")
    own[0] = 1 << 20  # an epoch that neither counter reaches
    ctx.quant_fp8_tensor(x, y, s, p, n)  # loads the code object
    torch.cuda.synchronize()
    p.zero_()
    y.fill_(0x5a)
    side, ended = torch.cuda.Stream(), torch.cuda.Event()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        arrive([own, fpeer, 1, 5, 2, missing], {})
        ended.record()
    marks = [torch.cuda.Event(enable_timing=True) for _ in range(9)]
    marks[0].record()
    for i in range(8):
        ctx.quant_fp8_tensor(x, y, s, p, n)
        marks[i + 1].record()
    marks[8].synchronize()
    waiting = not ended.query()
    torch.cuda.synchronize()
    us = sorted(marks[i].elapsed_time(marks[i + 1]) * 1e3 for i in range(8))
    print(f"  the wave was still waiting: {waiting}; median {us[4]:.1f} us", flush=True)
    assert int(missing[0]) == 0b11
    assert torch.equal(p.view(torch.int32), want_p.view(torch.int32))
    assert s.view(torch.int32).item() == want_s.view(torch.int32).item()
    assert torch.equal(y, want_y)
    assert us[4] < 200.0, us


def test_quant_fp8_tensor_one_launch_in_a_graph(ctx):
    """The one-launch form captured: every replay, on new inputs and with eager calls in
    between, gives the pair's outputs (its partials are marked again each time)."""
    n, nb = (24 << 20) + 5, 2048
    print(f"[case] quant_fp8_tensor captured n={n}", flush=True)
    x = torch.empty(n, dtype=torch.bfloat16, device="cuda")
    y, want_y = (torch.empty(n, dtype=torch.uint8, device="cuda") for _ in range(2))
    s, want_s = (torch.empty(1, dtype=torch.float32, device="cuda") for _ in range(2))
    p, want_p = (torch.empty(nb, dtype=torch.float32, device="cuda") for _ in range(2))
    x.fill_(1.0)
    ctx.quant_fp8_tensor(x, y, s, p, n)  # loads the code object before capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ctx.quant_fp8_tensor(x, y, s, p, n)
    stream = torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cuda").manual_seed(1600)
    for r in range(4):
        x.copy_(torch.empty(n, device="cuda").normal_(0, 2.0 / (r + 1), generator=g))
        y.fill_(0x5a)
        graph.replay()
        torch.cuda.synchronize()
        assert ctx.L.k3h_quant_fp8_amax(ctx.h, stream, 1, x.data_ptr(), n, want_p.data_ptr(), nb) == 0
        assert ctx.L.k3h_quant_fp8_apply(ctx.h, stream, 1, x.data_ptr(), want_y.data_ptr(), n,
                                         want_p.data_ptr(), nb, want_s.data_ptr()) == 0
        torch.cuda.synchronize()
        assert torch.equal(p.view(torch.int32), want_p.view(torch.int32)), f"replay {r}"
        assert s.view(torch.int32).item() == want_s.view(torch.int32).item(), f"replay {r}"
        assert torch.equal(y, want_y), f"replay {r}"
    graph.reset()
