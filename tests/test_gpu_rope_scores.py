"""The rope/scores chain and the softmax/values chain of attention values cut into slices: positions on
both sides of the scores' 256-row chunks, the last row and past the capacity, head sizes of every vector
layout, softmax rows of every width, q, k and v from buffers and from a split linear's planes; the
graph's results are those of the separate launches bit for bit, and those against a float64 reference."""
import numpy as np
import pytest

import ckl
from ckl.decoder_kernels import multiply
from programs.decoder import Cache, Position, Rotary, Square, attention, qkv

pytestmark = pytest.mark.gpu

_B, _C = ckl.dim("B"), ckl.dim("C")
_Rows = ckl.Buffer[ckl.f32, (_B, _C)]


@ckl.program
def layer(x: _Rows, wq: Square, wk: Square, wv: Square, sincos: Rotary, position: Position, kc: Cache, vc: Cache,
          out: _Rows, one: _Rows, scale: ckl.f32) -> None:
    q, key, value = qkv(x, wq, wk, wv, 0)
    mixed = attention(q, key, value, sincos, position, kc, vc, scale, 0)
    ckl.launch(multiply, mixed, one, out, grid=(ckl.cdiv(_C, 64), _B), block=(64,))


@pytest.mark.parametrize("b, a, t, d", [(1, 2, 1040, 128), (3, 1, 2100, 64), (1, 1, 6200, 20), (2, 2, 1500, 96), (1, 2, 600, 256),
                                        (1, 9, 1030, 128), (1, 1, 8192, 32), (2, 1, 512, 256)])
def test_rope_scores(device, b, a, t, d):
    rng = np.random.default_rng(t + d)
    c = a * d
    angles = np.arange(t)[:, None] * (10000. ** (-np.arange(0, d, 2) / d))[None, :]
    host = {"x": rng.standard_normal((b, c)), "wq": rng.standard_normal((1, c, c)) / np.sqrt(c),
            "wk": rng.standard_normal((1, c, c)) / np.sqrt(c), "wv": rng.standard_normal((1, c, c)) / np.sqrt(c),
            "sincos": np.stack((np.cos(angles), np.sin(angles)), -1), "position": np.zeros(1, np.int32),
            "kc": rng.standard_normal((1, b, a, t, d)), "vc": rng.standard_normal((1, b, a, t, d)),
            "out": np.zeros((b, c)), "one": np.ones((b, c))}
    buffers = {}
    for name, values in host.items():
        kind, dtype = (ckl.i32, np.int32) if name == "position" else (ckl.f32, np.float32)
        host[name] = values.astype(dtype)
        buffers[name] = device.empty(ckl.BufferSpec(values.shape, kind))
        buffers[name].copy_from_host(host[name])
    types = {n: v.spec for n, v in buffers.items()} | {"scale": ckl.f32}
    bound = layer.lower(signature=types).compile(fuse_pointwise=False).bind(*buffers.values(), d ** -0.5)
    assert any(name.startswith("ckl_rope__rope__append_kv__attention_scores") and len(nodes) == 4
               for name, nodes in bound.units())
    assert any(name.startswith("ckl_softmax__attention_values_split") and len(nodes) == 2 for name, nodes in bound.units())
    x = host["x"].astype(np.float64)
    for p in (0, 1, 255, 256, 257, t // 2, t - 1, t):
        results = []
        for mode in ("ordinary", "graph", "graph", "stream"):
            for name in ("kc", "vc", "out"):
                buffers[name].copy_from_host(host[name])
            buffers["position"].copy_from_host(np.array([p], np.int32))
            bound.run(mode=mode, batch_size=2)
            got = {n: np.empty_like(host[n]) for n in ("kc", "vc", "out")}
            for name, values in got.items():
                buffers[name].copy_to_host(values)
            results.append(got)
        if p == t:      # past the capacity nothing is rotated or appended, and q is what its buffer held
            assert all(np.array_equal(got[n], host[n]) for got in results for n in ("kc", "vc"))
            continue
        assert all(np.array_equal(got[n], results[0][n]) for got in results[1:] for n in got), p
        cos, sin = (host["sincos"][p, :, i].astype(np.float64) for i in (0, 1))

        def rotated(w):
            v = (x @ w[0].astype(np.float64)).reshape(b, a, d // 2, 2)
            return np.stack((v[..., 0] * cos - v[..., 1] * sin, v[..., 0] * sin + v[..., 1] * cos), -1).reshape(b, a, d)

        keys, values = host["kc"][0].astype(np.float64), host["vc"][0].astype(np.float64)
        keys[:, :, p], values[:, :, p] = rotated(host["wk"]), (x @ host["wv"][0].astype(np.float64)).reshape(b, a, d)
        logits = (rotated(host["wq"])[:, :, None] * keys[:, :, :p + 1]).sum(-1) * np.float64(np.float32(d ** -0.5))
        weights = np.exp(logits - logits.max(-1, keepdims=True))
        weights /= weights.sum(-1, keepdims=True)
        expected = (weights[..., None] * values[:, :, :p + 1]).sum(2).reshape(b, c)
        # q, k and v are sums of up to 1152 products of N(0, 1/C): ~1e-6 off, so scores and weights by
        # a few 1e-6, of values that are N(0, 1).
        assert np.max(np.abs(results[0]["out"] - expected)) <= 2e-5, p
        assert np.max(np.abs(results[0]["kc"][0] - keys)) <= 1e-5 and np.max(np.abs(results[0]["vc"][0] - values)) <= 1e-5, p
