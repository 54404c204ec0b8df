"""Generated elementwise kernels over long vectors (four elements a thread): lengths with and without
an incomplete last group, buffers that start at any element, in-place buffers, several inputs and
outputs, each element type, comparisons ahead of the guard used behind it; and the kernels that stay as
written: short vectors, launches that do not cover the vector, neighbour accesses, loads after a store.
Results are exact (the same operations per element as NumPy's, no contraction)."""
import re

import numpy as np
import pytest

import ckl

N = ckl.dim("N")
F32, F64, I32, I64 = (ckl.Buffer[t, (N,)] for t in (ckl.f32, ckl.f64, ckl.i32, ckl.i64))
LONG = 1 << 20


@ckl.kernel
def blend(a: F32, b: F32, out: F32, flags: F32, w: ckl.f32) -> None:
    i = ckl.global_id(0)
    low = i < 5
    if i < N:
        x = a[i] * w
        y = b[i] - a[i]
        out[i] = x + y
        flags[i] = ckl.select(low, x, y)


@ckl.kernel
def widen(a: F64, k: I32, out: F64, total: I64) -> None:
    i = ckl.global_id(0)
    if i < N:
        tripled = a[i] * 3.0
        total[i] = ckl.cast(k[i], ckl.i64) + 7
        out[i] = tripled


@ckl.kernel
def reread(a: F32, out: F32) -> None:
    i = ckl.global_id(0)
    if i < N:
        out[i] = a[i] + 1.0
        out[i] = out[i] * 2.0


@ckl.kernel
def shift(a: F32, out: F32) -> None:
    i = ckl.global_id(0)
    if i + 1 < N:
        out[i] = a[i + 1]


@ckl.program
def run_blend(a: F32, b: F32, out: F32, flags: F32, w: ckl.f32, groups: ckl.constexpr[ckl.index]) -> None:
    ckl.launch(blend, a, b, out, flags, w, grid=(groups,), block=(256,))


@ckl.program
def run_widen(a: F64, k: I32, out: F64, total: I64) -> None:
    ckl.launch(widen, a, k, out, total, grid=(ckl.cdiv(N, 128),), block=(128,))


@ckl.program
def run_reread(a: F32, out: F32) -> None:
    ckl.launch(reread, a, out, grid=(ckl.cdiv(N, 256),), block=(256,))


@ckl.program
def run_shift(a: F32, out: F32) -> None:
    ckl.launch(shift, a, out, grid=(ckl.cdiv(N, 256),), block=(256,))


def compiled(program, n, **constants):
    types = {name: ckl.BufferSpec((n,), t) for name, t in (("a", ckl.f32), ("b", ckl.f32), ("out", ckl.f32), ("flags", ckl.f32))}
    if program is run_widen:
        types = {name: ckl.BufferSpec((n,), t) for name, t in (("a", ckl.f64), ("k", ckl.i32), ("out", ckl.f64), ("total", ckl.i64))}
    elif program is not run_blend:
        types = {name: types[name] for name in ("a", "out")}
    else:
        types["w"] = ckl.f32
    return program.lower(signature=types, constants=constants).compile(fuse_pointwise=False)


def grid(program):
    return int(re.search(r"\bgrid = array<i64: (\d+)", program.executable_ir).group(1))


def test_which_kernels_are_vectorized():
    covering = -(-LONG // 256)
    assert grid(compiled(run_blend, LONG, groups=covering)) == LONG // 1024
    assert grid(compiled(run_blend, LONG + 1, groups=covering + 1)) == LONG // 1024 + 1
    assert grid(compiled(run_blend, LONG, groups=covering - 1)) == covering - 1          # does not cover N
    assert grid(compiled(run_blend, LONG - 1, groups=covering)) == covering              # short
    assert grid(compiled(run_widen, LONG + 3)) == LONG // 1024 + 1
    assert grid(compiled(run_reread, LONG)) == covering and grid(compiled(run_shift, LONG)) == covering


def buffer(device, values, offset=0):
    kind = {np.float32: ckl.f32, np.float64: ckl.f64, np.int32: ckl.i32, np.int64: ckl.i64}[values.dtype.type]
    whole = device.empty(ckl.BufferSpec((values.size + offset + 5,), kind))
    part = whole.subview(offset=offset, shape=(values.size,))
    part.copy_from_host(values)
    return part


def host(part, like):
    out = np.empty_like(like)
    part.copy_to_host(out)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("n", [LONG, LONG + 1, LONG + 3, (1 << 21) + 2])
@pytest.mark.parametrize("offset", [0, 1])
def test_blend(device, n, offset):
    rng = np.random.default_rng(n)
    a, b = (rng.standard_normal(n).astype(np.float32) for _ in range(2))
    a[:3] = np.inf, -np.inf, np.nan
    zero = np.zeros(n, np.float32)
    program = compiled(run_blend, n, groups=-(-n // 256))
    w = np.float32(0.3)
    with np.errstate(invalid="ignore"):
        x, y = a * w, b - a
        expected = x + y
    flags = np.where(np.arange(n) < 5, x, y)
    da, db, do, df = (buffer(device, v, offset + k) for k, v in enumerate((a, b, zero, zero)))
    for mode in ("ordinary", "graph", "capture"):
        program.bind(da, db, do, df, float(w)).run(mode=mode)
        assert np.array_equal(host(do, zero), expected, equal_nan=True) and np.array_equal(host(df, zero), flags, equal_nan=True)
    program.bind(da, db, db, df, float(w)).run()                     # in place: out is b
    assert np.array_equal(host(db, zero), expected, equal_nan=True) and np.array_equal(host(df, zero), flags, equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [LONG, LONG + 2])
def test_widen(device, n):
    rng = np.random.default_rng(n)
    a, k = rng.standard_normal(n), rng.integers(-2**31, 2**31, n, dtype=np.int32)
    da, dk, do, dt = (buffer(device, v, s) for v, s in ((a, 1), (k, 3), (np.zeros(n), 0), (np.zeros(n, np.int64), 1)))
    compiled(run_widen, n).bind(da, dk, do, dt).run()
    assert np.array_equal(host(do, a), a * 3.0) and np.array_equal(host(dt, np.zeros(n, np.int64)), k.astype(np.int64) + 7)


@pytest.mark.gpu
def test_kernels_that_stay_as_written(device):
    a = np.random.default_rng(1).standard_normal(LONG).astype(np.float32)
    zero = np.zeros_like(a)
    for program, expected in ((run_reread, (a + np.float32(1)) * np.float32(2)), (run_shift, np.append(a[1:], np.float32(0)))):
        da, do = buffer(device, a), buffer(device, zero)
        compiled(program, LONG).bind(da, do).run()
        assert np.array_equal(host(do, zero), expected)
