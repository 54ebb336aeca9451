"""The native host path (csrc/host.cpp) against the wrappers' general path."""

import shutil
import subprocess
import sys
import threading

import pytest
import torch

import mlx_qsdpa_amd as mq
from conftest import ROOT
from mlx_qsdpa_amd import kernels

pytestmark = pytest.mark.gpu


def _call(L=1, B=2, Hq=8, Hkv=2, N=2000, D=128, bits=4, gs=64, dtype=torch.float16, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q = torch.randn(B, Hq, L, D, generator=g, device="cuda").to(dtype)
    k, v = (kernels.quantize(torch.randn(B, Hkv, N, D, generator=g, device="cuda").to(dtype), gs, bits)
            for _ in range(2))
    return dict(q=q, packed_k=k[0], packed_v=v[0], k_scales=k[1], v_scales=v[1], k_biases=k[2], v_biases=v[2],
                bits=bits, group_size=gs)


def _both(monkeypatch, a):
    """(native path, general path), and whether the native one took the call."""
    took = []
    native = kernels._native_decode
    with monkeypatch.context() as m:
        m.setattr(kernels, "_native_decode", lambda *x: took.append(native(*x)) or took[-1])
        got = mq.quantized_sdpa(**a)
        m.setattr(kernels, "_native_decode", lambda *x: None)
        want = mq.quantized_sdpa(**a)
    torch.cuda.synchronize()
    return got, want, isinstance(took[0], torch.Tensor) if took else False


def _keep(*shape):
    return torch.rand(shape, generator=torch.Generator(device="cuda").manual_seed(7), device="cuda") < 0.8


def _off_by_one(t):
    wide = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    wide[1:] = t.reshape(-1)
    return wide[1:].view(t.shape)


FORMS = {
    "plain": ({}, lambda a: a, True),
    "several": ({"L": 5}, lambda a: dict(a, mask="causal"), True),
    "symmetric": ({}, lambda a: dict(a, k_biases=None), True),
    "padded": ({}, lambda a: dict(a, kv_start=torch.tensor([3, 700], dtype=torch.int32, device="cuda")), True),
    "host_start": ({}, lambda a: dict(a, kv_start=torch.tensor([3, 700])), False),
    "capacity": ({}, lambda a: {n: x[:, :, :1500] if n[0] in "pkv" else x for n, x in a.items()}, True),
    "q_strided": ({"L": 3}, lambda a: dict(a, q=a["q"].transpose(1, 2).contiguous().transpose(1, 2)), True),
    "q_inner": ({}, lambda a: dict(a, q=a["q"].transpose(2, 3).contiguous().transpose(2, 3)), True),
    "q_2_bytes_off": ({}, lambda a: dict(a, q=_off_by_one(a["q"])), True),
    "codes_in_odd_rows": ({}, lambda a: dict(a, packed_k=torch.nn.functional.pad(
        a["packed_k"].view(torch.int32), (1, 0)).view(torch.uint32)[..., 1:]), False),
    "bool": ({}, lambda a: dict(a, mask=_keep(2, 1, 1, 2000)), True),
    "bool_rows": ({"L": 5}, lambda a: dict(a, mask=_keep(2, 8, 5, 2000)), True),
    "bool_2d": ({"L": 5}, lambda a: dict(a, mask=_keep(5, 2000)), True),
    "bool_1d_start": ({}, lambda a: dict(a, mask=_keep(2000), kv_start=torch.tensor([3, 700], dtype=torch.int32,
                                                                                   device="cuda")), True),
    "bool_view": ({}, lambda a: dict(a, mask=_keep(2, 1, 1, 2001)[..., 1:]), True),
    "additive_f16": ({}, lambda a: dict(a, mask=_keep(1, 8, 1, 2000).half()), True),
    "additive_bf16": ({"D": 256}, lambda a: dict(a, mask=_keep(2, 1, 1, 2000).bfloat16()), True),
    "additive_f32": ({"D": 64}, lambda a: dict(a, mask=_keep(2, 1, 1, 2000).float()), True),
    "mask_of_strided_keys": ({}, lambda a: dict(a, mask=_keep(2, 1, 1, 4000)[..., ::2]), False),
    "host_mask": ({}, lambda a: dict(a, mask=_keep(2, 1, 1, 2000).cpu()), True),
    "masked_prefill": ({"L": 700, "B": 12, "Hkv": 4}, lambda a: dict(a, mask=_keep(12, 1, 700, 2000)), True),
    "d256": ({"D": 256, "bits": 8, "dtype": torch.bfloat16}, lambda a: a, True),
}


@pytest.mark.parametrize("form", FORMS)
def test_native_decode_equals_the_general_path(device, monkeypatch, form):
    shape, change, native = FORMS[form]
    print(f"native decode {form}", flush=True)
    got, want, took = _both(monkeypatch, change(_call(**shape)))
    assert took == native
    assert torch.equal(got, want)


@pytest.mark.parametrize("change,error", [
    (lambda a: dict(a, v_scales=a["v_scales"][:, :, :-1]), ValueError),
    (lambda a: dict(a, packed_v=a["packed_v"].view(torch.int32)), ValueError),
    (lambda a: dict(a, k_scales=a["k_scales"].float()), ValueError),
    (lambda a: dict(a, kv_start=torch.zeros(3, dtype=torch.int32, device="cuda")), ValueError),
    (lambda a: dict(a, bits=3), ValueError),
    (lambda a: dict(a, mask=_keep(2, 1, 1, 1999)), ValueError),
    (lambda a: dict(a, mask=_keep(3, 1, 1, 2000)), RuntimeError),
    (lambda a: dict(a, mask=_keep(2, 1, 2, 2000)), ValueError),
    (lambda a: dict(a, mask=_keep(2, 1, 1, 2000).to(torch.int8)), ValueError),
    (lambda a: dict(a, q=a["q"].cpu()), RuntimeError),
    (lambda a: dict(a, packed_k=a["packed_k"][:, :, :0], packed_v=a["packed_v"][:, :, :0],
                    k_scales=a["k_scales"][:, :, :0], v_scales=a["v_scales"][:, :, :0],
                    k_biases=None, v_biases=None), RuntimeError),
], ids=["shape", "codes", "scales", "start", "bits", "mask_keys", "mask_batch", "mask_rows", "mask_type", "host", "empty"])
def test_refusals(device, change, error):
    with pytest.raises(error):
        mq.quantized_sdpa(**change(_call()))


def test_updates_equal_the_general_path(device, monkeypatch):
    """Appends and growth: strided new tokens, odd strides of held buffers."""
    g = torch.Generator(device="cuda").manual_seed(3)
    steps = [torch.randn(2, 3, n, 64, generator=g, device="cuda").half() for n in (300, 1, 213, 256, 5)]

    def fill():
        c = mq.BatchQuantizedSDPACache([0, 7], bits=8, group_size=32)
        for i, x in enumerate(steps):
            if i == 3:
                x = x.transpose(2, 3).contiguous().transpose(2, 3)  # strided rows
            if i == 2:
                c._keys = tuple(torch.cat([t, t], 1)[:, :3] for t in c._keys)
            c.update_and_fetch(x, -x)
        return [t.clone() for t in c._keys + c._values]

    got = fill()
    monkeypatch.setattr(kernels, "grown", lambda *a: None)
    real = kernels._host()
    monkeypatch.setattr(kernels, "_HOST", type("none", (), {"quantize_kv": staticmethod(lambda *a: None),
                                                           "columns": real.columns}))
    for a, b in zip(got, fill()):
        assert a.shape == b.shape and torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_captured_decode_replays(device):
    """A captured call keeps a workspace of its own: replays between eager
    calls that grow and use the shared one give the eager bits."""
    a, big = _call(N=4000), _call(N=60000, seed=1)
    want, want_big = mq.quantized_sdpa(**a), mq.quantized_sdpa(**big)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        mq.quantized_sdpa(**a)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = mq.quantized_sdpa(**a)
    for _ in range(4):
        out.zero_()
        graph.replay()
        assert torch.equal(mq.quantized_sdpa(**big), want_big)
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        kernels._ARGS.d = {}  # the shared workspaces go; the graph's stays


def test_captured_masked_prefill_replays(device):
    """A captured masked prefill of several rounds keeps its key ranges in the
    graph's own workspace."""
    a = _call(B=12, Hkv=4, L=300, N=900)
    a["mask"] = torch.ones(12, 1, 300, 900, dtype=torch.bool, device="cuda").tril(600)
    want = mq.quantized_sdpa(**a)
    other = dict(a, mask=_keep(12, 1, 300, 900))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = mq.quantized_sdpa(**a)
    for _ in range(3):
        out.zero_()
        graph.replay()
        mq.quantized_sdpa(**other)
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        kernels._ARGS.d = {}


def test_threads_on_one_stream(device):
    """Two threads decoding on the same stream share no workspace."""
    calls = [_call(N=9000, B=1, seed=s) for s in (5, 6)]
    want = [mq.quantized_sdpa(**a) for a in calls]
    torch.cuda.synchronize()
    bad = []

    def loop(a, w):
        for _ in range(200):
            if not torch.equal(mq.quantized_sdpa(**a), w):
                bad.append(1)

    ts = [threading.Thread(target=loop, args=x) for x in zip(calls, want)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad


# The library's launches replaced: each returns an error while its thread
# holds the interpreter's lock.
_STUB = """
#include "qsdpa.h"
extern "C" {
int PyGILState_Check(void);
static int held() { return PyGILState_Check() ? QSDPA_ERR_LAUNCH : QSDPA_OK; }
int qsdpa_abi_version(void) { return QSDPA_ABI_VERSION; }
int64_t qsdpa_decode_workspace_size(const qsdpa_decode_args*, int32_t*) { return 0; }
int64_t qsdpa_decode_range_bytes(const qsdpa_decode_args*) { return 0; }
int qsdpa_decode(const qsdpa_decode_args*, void*) { return held(); }
int qsdpa_decode_ranges(const qsdpa_decode_args*, void*, int64_t, void*) { return held(); }
int qsdpa_quantize_batch(const qsdpa_quantize_args*, int32_t, void*) { return held(); }
int qsdpa_move_rows(const qsdpa_row_move*, int32_t, void*) { return held(); }
int qsdpa_causal_mask(const qsdpa_causal_mask_args*, void*) { return held(); }
int qsdpa_rotate(const qsdpa_rotate_args*, void*) { return held(); }
}
"""

_CHILD = """
import sys, torch
torch.zeros(1, device="cuda")
sys.path.insert(0, sys.argv[1])
import _host
x = torch.zeros(1, 2, 4, 64, dtype=torch.float16, device="cuda")
b = tuple(torch.zeros(1, 2, 4, w, dtype=t, device="cuda") for w, t in ((8, torch.uint32), (2, x.dtype), (2, x.dtype)))
out = {"quantize_kv": _host.quantize_kv(x, x, b, b, 0, 4, 32, 0),
       "grown": _host.grown(x, x, None, 0, 8, 4, 32, 0),
       "decode": _host.decode(x, b[0], b[0], b[1], b[1], b[2], b[2], 1.0, 4, 32, None, 0, False, None, 0, None),
       "rotate": _host.rotate(x, x, 3, 1e4, 0),
       "causal_mask": _host.causal_mask(4, 3, None, None, 0, 0)}
for name, got in out.items():
    assert got is not None and (got == 0 if name == "quantize_kv" else type(got) is not int), name
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_launches_release_the_interpreter(device, tmp_path):
    """Every native call gives the interpreter's lock back around its launch
    (a launch waits when the stream's queue is full)."""
    lib, host = tmp_path / "libqsdpa_hip.so", ROOT / "mlx-qsdpa_amd" / "mlx_qsdpa_amd" / "_host.so"
    (tmp_path / "stub.cpp").write_text(_STUB)
    subprocess.run(["g++", "-shared", "-fPIC", f"-I{ROOT / 'include'}", str(tmp_path / "stub.cpp"), "-o", str(lib)],
                   check=True)
    shutil.copy(host, tmp_path / "_host.so")
    subprocess.run([sys.executable, "-c", _CHILD, str(tmp_path)], check=True, timeout=100)
