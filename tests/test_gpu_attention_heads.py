"""Attention over head sizes that are a multiple of 4 but no power of two times the lanes of a row:
the padded layout of the scores and the values' row groups that do not divide the workgroup, alone and
in the rope/attention chain (bit for bit the same, and the oracle's state), rows from one to several
batches of every wave. A key row holding an infinity leaves the other rows' scores alone."""
import numpy as np
import pytest

import ckl
from oracle import decoder as oracle
from ckl.decoder_kernels import attention_scores
from programs.decoder_config import Config
from programs.harness import MUTABLE, DecoderSession

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim, heads, batch, context", [(12, 2, 2, 5), (24, 3, 1, 70), (48, 1, 3, 300), (80, 3, 2, 150),
                                                         (96, 1, 1, 600), (160, 2, 1, 60), (252, 1, 2, 40)])
def test_padded_head_sizes(device, dim, heads, batch, context):
    c = Config(batch=batch, hidden=dim * heads, heads=heads, layers=1, ffn=32, vocab=40, context=context, steps=3)
    initial, _ = oracle.make_inputs(c, 5, init="reference")
    session = DecoderSession(c, device, arrays=initial)
    reference = oracle.expected(initial, c, c.steps)
    for inv in session.invocations.values():
        results = []
        for mode, group in (("ordinary", 1), ("graph", 1), ("stream", c.steps)):
            session.state.reset()
            for _ in range(c.steps // group):
                inv.run(mode=mode, batch_size=group)
            session.state.verify(reference)
            results.append({name: session.state.download(name) for name in MUTABLE})
        for got in results[1:]:
            assert all(np.array_equal(got[name], results[0][name]) for name in MUTABLE)


_B, _C, _L, _A, _T, _D = (ckl.dim(n) for n in ("B", "C", "L", "A", "T", "D"))


@ckl.program
def score(q: ckl.Buffer[ckl.f32, (_B, _C)], kc: ckl.Buffer[ckl.f32, (_L, _B, _A, _T, _D)], p: ckl.Buffer[ckl.i32, (1,)],
          out: ckl.Buffer[ckl.f32, (_B, _A, _T)], scale: ckl.f32) -> None:
    ckl.launch(attention_scores, q, kc, p, out, scale, 0, grid=(ckl.cdiv(_T, 32), _A, _B), block=(32,))


@pytest.mark.parametrize("dim", [20, 80, 96])
def test_infinite_key_stays_in_its_row(device, dim):
    heads, slots, position = 2, 90, 77
    rng = np.random.default_rng(dim)
    q = np.abs(rng.standard_normal((1, heads * dim))).astype(np.float32) + np.float32(0.1)
    keys = rng.standard_normal((1, 1, heads, slots, dim)).astype(np.float32)
    keys[0, 0, 0, 13, 3] = -np.inf
    keys[0, 0, 1, position, dim - 1] = np.inf
    host = {"q": q, "kc": keys, "p": np.array([position], np.int32), "out": np.zeros((1, heads, slots), np.float32)}
    buffers = {}
    for name, values in host.items():
        buffers[name] = device.empty(ckl.BufferSpec(values.shape, ckl.i32 if values.dtype == np.int32 else ckl.f32))
        buffers[name].copy_from_host(values)
    types = {n: b.spec for n, b in buffers.items()} | {"scale": ckl.f32}
    score.lower(signature=types).compile(fuse_pointwise=False).bind(*buffers.values(), 0.125).run()
    got = np.empty_like(host["out"])
    buffers["out"].copy_to_host(got)
    expected = np.einsum("hd,htd->ht", q.reshape(heads, dim).astype(np.float64), keys[0, 0].astype(np.float64)) * 0.125
    n = position + 1
    assert got[0, 0, 13] == -np.inf and got[0, 1, position] == np.inf
    finite = np.isfinite(expected[:, :n])
    assert np.array_equal(finite, np.isfinite(got[0, :, :n]))
    # f32 sums of D products of magnitude about 1.
    assert np.all(np.abs(got[0, :, :n][finite] - expected[:, :n][finite]) <= 1e-6 * dim)
