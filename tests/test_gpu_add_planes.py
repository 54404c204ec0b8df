"""add as a reader of a split linear's partial planes (the residual sum that no norm follows): the
inferred graph leaves the combine to add, bit for bit what the ordinary launches compute, for rows
taken as float4s and as single elements, planes as either operand or both, and few or many planes."""
import numpy as np
import pytest

import ckl
from ckl.decoder_kernels import add, linear
from ckl.library import linear_tiling

pytestmark = pytest.mark.gpu

_B, _I, _O = (ckl.dim(n) for n in ("B", "I", "O"))
_Y = ckl.Buffer[ckl.f32, (_B, _O)]


@ckl.program
def residual(x: ckl.Buffer[ckl.f32, (_B, _I)], w: ckl.Buffer[ckl.f32, (1, _I, _O)], r: _Y, left: _Y, right: _Y,
             twice: _Y) -> None:
    columns = (ckl.cdiv(_O, 64), _B)
    a = ckl.empty((_B, _O), dtype=ckl.f32)
    b = ckl.empty((_B, _O), dtype=ckl.f32)
    c = ckl.empty((_B, _O), dtype=ckl.f32)
    ckl.launch(linear, x, w, a, 0, grid=columns, block=(64,))
    ckl.launch(add, r, a, right, grid=columns, block=(64,))
    ckl.launch(linear, x, w, b, 0, grid=columns, block=(64,))
    ckl.launch(add, b, r, left, grid=columns, block=(64,))
    ckl.launch(linear, x, w, c, 0, grid=columns, block=(64,))
    ckl.launch(add, c, c, twice, grid=columns, block=(64,))


@pytest.mark.parametrize("shape", [(20, 1024, 1024), (17, 600, 37), (3, 2100, 130), (33, 5632, 260), (16, 4000, 64)],
                         ids=lambda s: "x".join(map(str, s)))
def test_add_reads_partial_planes(device, shape):
    b, i, o = shape
    assert linear_tiling(b, i, o)["split"] > 1
    rng = np.random.default_rng(b + i + o)
    host = {"x": rng.standard_normal((b, i)).astype(np.float32), "w": rng.standard_normal((1, i, o)).astype(np.float32),
            "r": rng.standard_normal((b, o)).astype(np.float32)}
    host.update({name: np.full((b, o), np.nan, np.float32) for name in ("left", "right", "twice")})
    buffers = {}
    for name, values in host.items():
        buffers[name] = device.empty(ckl.BufferSpec(values.shape, ckl.f32))
    bound = residual.lower(signature={n: v.spec for n, v in buffers.items()}).compile(fuse_pointwise=False).bind(*buffers.values())
    results = []
    for mode in ("ordinary", "graph", "stream"):
        for name, values in host.items():
            buffers[name].copy_from_host(values)
        bound.run(mode=mode)
        got = {name: np.empty((b, o), np.float32) for name in ("left", "right", "twice")}
        for name, out in got.items():
            buffers[name].copy_to_host(out)
        results.append(got)
    product = host["x"].astype(np.float64) @ host["w"][0].astype(np.float64)
    for name, expected in (("left", product + host["r"]), ("right", product + host["r"]), ("twice", 2 * product)):
        # f32 accumulation of I products of N(0, 1) values, the bound of test_gpu_linear.py.
        assert np.all(np.abs(results[0][name] - expected) <= np.sqrt(i) * 2e-5 * (1 + np.abs(expected))), name
        assert all(np.array_equal(r[name], results[0][name]) for r in results[1:]), name
