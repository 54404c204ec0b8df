"""Linears of at most 16 rows on the 16-row MFMA kernel: one row and all 16, column tiles and
reduction slices with a remainder, widths no multiple of 4, one and many splits; checked as
tests/test_gpu_linear.py checks its shapes. A decoder whose q/k/v and gate/up run as shared launches
checks the merged launches and the planes its chains read (inferred against ordinary launches, bit
for bit, and against the oracle's state)."""
import numpy as np
import pytest

from oracle import decoder as oracle
from ckl.library import linear_tiling
from programs.decoder_config import Config
from programs.harness import MUTABLE, DecoderSession
from test_gpu_linear import test_linear_matches_float64 as matches_float64

SHAPES = [(1, 32800, 16), (16, 31000, 17), (5, 7900, 67), (16, 2049, 1031), (8, 5632, 2048), (13, 1027, 4097), (2, 1024, 12002)]
SHARED = Config(batch=7, hidden=2048, heads=8, layers=1, ffn=2902, vocab=301, context=4, steps=3)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_linear_of_few_rows(device, shape):
    assert linear_tiling(*shape)["entry"].startswith("ckl_linear_mfma16_")
    matches_float64(device, shape)


@pytest.mark.gpu
def test_decoder_of_few_rows_is_bit_identical_to_ordinary(device):
    c = SHARED
    initial, _ = oracle.make_inputs(c, 13, init="reference")
    session = DecoderSession(c, device, arrays=initial)
    reference = oracle.expected(initial, c, c.steps)
    for inv in session.invocations.values():
        names = [name for name, _ in inv.units()]
        assert any(n.startswith("ckl_linear_mfma16_") and n.endswith("_shared3") for n in names)
        assert any(n.startswith("ckl_linear_mfma16_") and n.endswith("_shared2") for n in names)
        results = []
        for mode, group in (("ordinary", 1), ("graph", 1), ("graph", c.steps)):
            session.state.reset()
            for _ in range(c.steps // group):
                inv.run(mode=mode, batch_size=group)
            session.state.verify(reference)
            results.append({name: session.state.download(name) for name in MUTABLE})
        for got in results[1:]:
            assert all(np.array_equal(got[name], results[0][name]) for name in MUTABLE)
