"""GPU parity of the fused FFN's 16-row blocks (few rows): row counts at the
block edges and on both sides of one block per CU, the last block with one to
sixteen live rows, requant directions of every block of the seeded model, and
the next LayerNorm through the model; against the CPU oracle, bit for bit."""

import numpy as np
import pytest

from heatvit_amd import synth

pytestmark = pytest.mark.gpu


def _check(oracle, bp, lens, seed):
    from heatvit_amd.transformer import transformer_block_batch
    rng = np.random.default_rng(seed)
    xs = [rng.integers(-128, 128, (n, 192)).astype(np.int8) for n in lens]
    zs = transformer_block_batch(xs, bp)
    for i, x in enumerate(xs):
        want, _ = oracle.transformer_block(x, bp, checkpoints=False)
        assert np.array_equal(zs[i], want), (lens, i)


@pytest.mark.parametrize("rows", (1, 15, 16, 17, 31, 33, 197, 4081, 4095, 4096, 4097, 4112))
def test_block_row_counts(oracle, rows):
    """4,096 rows are one 16-row block per CU of a 256-CU device."""
    lens = [197] * (rows // 197) + ([rows % 197] if rows % 197 else [])
    _check(oracle, synth.block_workload()[1], lens, rows)


@pytest.mark.parametrize("index", range(12))
def test_requant_directions(oracle, index):
    bp = synth.pruned_params().blocks[index]
    _check(oracle, bp, [197, 64, 5], 50 + index)


@pytest.mark.parametrize("batch", (2, 20, 21, 41, 42))
def test_model_chains_the_next_layernorm(oracle, batch):
    from heatvit_amd.model import HeatViTModel
    images, params = synth.pruned_workload(batch)
    res = HeatViTModel().infer_batch(images, params)
    logits, counts, status, warnings = oracle.model_infer_batch(images, params, threads=8)
    assert not status.any()
    assert np.array_equal(res.logits, logits)
    assert np.array_equal(res.token_counts, counts)
    assert np.array_equal(res.warnings, warnings)
