"""Weights and gradients read into device memory of the caller: bit for bit those read to the host, for packed bf16 matrices at the
edges of the kernel's pieces (a last workgroup of two k steps, of four), fp32 matrices whose experts' parts lie off 16 bytes, odd
lengths, destinations off 16 and off 4 bytes, and nothing written around the destination."""
import ctypes
import importlib

import numpy as np
import pytest

from tests.synth import C, make_inputs, scaled

pytestmark = pytest.mark.gpu
L = importlib.import_module("omega-ai_amd._lib")


@pytest.mark.parametrize("dtype,d,H,E", [("bf16", 256, 384, 2), ("bf16", 768, 256, 3), ("bf16", 512, 640, 17), ("bf16", 2048, 1408, 2),
                                         ("f32", 33, 51, 3), ("f32", 7, 3, 2), ("f32", 64, 128, 2), ("f32", 1024, 1030, 2)])
def test_reads_to_device_equal_reads_to_host(dtype, d, H, E):
    from tests import gpu_util as G
    cfg = scaled(C.CONFIGS["c1_tiny_f32"], T=40, d=d, H=H, E=E, K=2, Es=1, dtype=dtype)
    inp = make_inputs(cfg, 21)
    layer = G.build_layer(cfg, inp)
    x = G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], dtype)
    layer.forward(x)
    layer.back(x)
    shapes = {L.W_GATE: (E, d), L.W_W1: (H, d), L.W_W3: (H, d), L.W_W2: (d, H)}
    lib = layer.lib
    for get, size in ((lib.omega_moe_get_weights, 2 if dtype == "bf16" else 4), (lib.omega_moe_get_grad, 4)):
        for which, shape in shapes.items():
            n = shape[0] * shape[1] * size
            for g in range(1 if which == L.W_GATE else E + 1):
                host = np.empty(n, np.uint8)
                layer.ctx.check(get(layer.handle, which, g, host.ctypes.data, 0))
                assert host.any()
                for off in (0, 4, 8, 2):
                    if off == 2 and size == 4:
                        continue
                    around = np.full(n + 64, 0xA5, np.uint8)
                    buf = G.P.DeviceBuffer.from_numpy(G.ctx(), np.full((n + 64 + 3) // 4, np.uint32(0xA5A5A5A5)).view(np.float32), "f32")
                    layer.ctx.check(get(layer.handle, which, g, ctypes.c_void_p(buf.ptr.value + 32 + off), 1))
                    around[32 + off:32 + off + n] = host
                    assert np.array_equal(buf.to_numpy().view(np.uint8)[:n + 64], around), (which, g, off)
                    buf.free()
    x.free()
    layer.close()
