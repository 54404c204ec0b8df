"""Linears of more than 16 rows whose reduction or output width is no multiple of 4 run on the MFMA
kernels: rows that start at any 4-byte address, a last lane whose columns are moved back into the
row, reductions shorter than one stage. Checked as tests/test_gpu_linear.py checks its shapes
(float64 product, |err| <= 1e-5 * sqrt(I) * (1 + |value|), every mode bit for bit), and inside a
decoder whose split linears leave their combine to the chains (inferred against ordinary launches,
bit for bit, and against the oracle's state)."""
import numpy as np
import pytest

from oracle import decoder as oracle
from ckl.library import linear_tiling
from programs.decoder_config import Config
from programs.harness import MUTABLE, DecoderSession
from test_gpu_linear import test_linear_matches_float64 as matches_float64  # noqa: F401 (called below)

SHAPES = [(17, 1, 1), (17, 5, 3), (33, 18, 2), (32, 37, 65), (64, 130, 131), (61, 1502, 4106), (32, 2047, 2049)]
ODD = Config(batch=20, hidden=42, heads=3, layers=2, ffn=31, vocab=70, context=4, steps=3)
SPLIT = Config(batch=35, hidden=1030, heads=5, layers=1, ffn=1537, vocab=301, context=4, steps=3)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_every_width_takes_a_library_kernel(shape):
    for members in (1, 2, 3):
        t = linear_tiling(*shape, members)
        j = int(t["entry"].removeprefix("ckl_linear_mfma")[0])
        assert j <= shape[2] and t["tiles"] * 32 * j >= shape[2] and t["split"] * t["chunk"] >= shape[1]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_ragged_linear(device, shape):
    matches_float64(device, shape)


@pytest.mark.gpu
@pytest.mark.parametrize("c", [ODD, SPLIT], ids=["odd", "split"])
def test_ragged_decoder_is_bit_identical_to_ordinary(device, c):
    initial, _ = oracle.make_inputs(c, 11, init="reference")
    session = DecoderSession(c, device, arrays=initial)
    reference = oracle.expected(initial, c, c.steps)
    for inv in session.invocations.values():
        results = []
        for mode, group in (("ordinary", 1), ("graph", 1), ("graph", c.steps)):
            session.state.reset()
            for _ in range(c.steps // group):
                inv.run(mode=mode, batch_size=group)
            session.state.verify(reference)
            results.append({name: session.state.download(name) for name in MUTABLE})
        for got in results[1:]:
            assert all(np.array_equal(got[name], results[0][name]) for name in MUTABLE)
