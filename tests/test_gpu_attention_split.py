"""Attention values cut into slices (few long rows): the sum of every slice, empty slices early in
the context, positions at slice edges, capacities and head sizes with remainders, the counters left
ready for the next launch, and softmax rows long enough for 1024 threads; scores -> softmax -> values
against a float64 reference, every mode and repetition bit for bit the same."""
import numpy as np
import pytest

import ckl
from ckl.decoder_kernels import attention_scores, attention_values, softmax
from ckl.library import _values_slices

pytestmark = pytest.mark.gpu

_B, _C, _L, _A, _T, _D = (ckl.dim(n) for n in ("B", "C", "L", "A", "T", "D"))
_Rows = ckl.Buffer[ckl.f32, (_B, _C)]
_Cache = ckl.Buffer[ckl.f32, (_L, _B, _A, _T, _D)]


@ckl.program
def attend(q: _Rows, kc: _Cache, vc: _Cache, p: ckl.Buffer[ckl.i32, (1,)], out: _Rows, scale: ckl.f32) -> None:
    scores = ckl.empty((_B, _A, _T), dtype=ckl.f32)
    weights = ckl.empty_like(scores)
    ckl.launch(attention_scores, q, kc, p, scores, scale, 1, grid=(ckl.cdiv(_T, 32), _A, _B), block=(32,))
    ckl.launch(softmax, scores, p, weights, grid=(ckl.cdiv(_B, 32), _A), block=(32,))
    ckl.launch(attention_values, weights, vc, p, out, 1, grid=(ckl.cdiv(_D, 32), _A, _B), block=(32,))


@pytest.mark.parametrize("b, a, t, d", [(1, 2, 1024, 128), (1, 1, 6145, 4), (2, 3, 1639, 80), (1, 5, 7001, 20), (3, 11, 600, 256)])
def test_split_values(device, b, a, t, d):
    slices = _values_slices(b * a, t, d)
    assert slices > 1
    rng = np.random.default_rng(t + d)
    host = {"q": rng.standard_normal((b, a * d)), "kc": rng.standard_normal((2, b, a, t, d)),
            "vc": rng.standard_normal((2, b, a, t, d)), "out": np.zeros((b, a * d))}
    buffers = {}
    for name, values in host.items():
        host[name] = values.astype(np.float32)
        buffers[name] = device.empty(ckl.BufferSpec(values.shape, ckl.f32))
        buffers[name].copy_from_host(host[name])
    buffers["p"] = device.empty(ckl.BufferSpec((1,), ckl.i32))
    order = [buffers[n] for n in ("q", "kc", "vc", "p", "out")]
    types = dict(zip(("q", "kc", "vc", "p", "out"), (o.spec for o in order))) | {"scale": ckl.f32}
    compiled = attend.lower(signature=types).compile(fuse_pointwise=False)
    assert '"ckl_attention_values_split"' in compiled.executable_ir
    bound = compiled.bind(*order, d ** -0.5)
    keys, values = host["kc"][1].astype(np.float64), host["vc"][1].astype(np.float64)
    query = host["q"].reshape(b, a, 1, d).astype(np.float64)
    for position in sorted({0, 1, slices - 1, slices, t // 2, t - 2, t - 1}):
        buffers["p"].copy_from_host(np.array([position], np.int32))
        n = position + 1
        logits = (query * keys[:, :, :n]).sum(-1) * np.float64(np.float32(d ** -0.5))
        weights = np.exp(logits - logits.max(-1, keepdims=True))
        weights /= weights.sum(-1, keepdims=True)
        expected = (weights[..., None] * values[:, :, :n]).sum(2).reshape(b, a * d)
        first = None
        for mode in ("ordinary", "graph", "stream", "ordinary"):
            buffers["out"].copy_from_host(np.full((b, a * d), np.nan, np.float32))
            bound.run(mode=mode, batch_size=2)
            got = np.empty((b, a * d), np.float32)
            buffers["out"].copy_to_host(got)
            # Scores of N(0, 1) operands are off by ~1e-6, so weights by ~1e-6 relative; values are N(0, 1).
            assert np.all(np.abs(got - expected) <= 1e-5), (position, mode, float(np.max(np.abs(got - expected))))
            first = got if first is None else first
            assert np.array_equal(got, first), (position, mode)
