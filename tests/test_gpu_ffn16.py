"""GPU parity of the fused FFN's 16-row blocks (few rows): row counts at the
block edges and on both sides of one block per CU, the last block with one to
sixteen live rows, requant directions of every block of the seeded model, and
the next LayerNorm through the model; and, after selectors that keep most
rows, the same blocks over 32 rows; against the CPU oracle, bit for bit."""

import dataclasses

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


# Selectors that keep every token: after them 21 to 41 images still hold more
# live rows than one 16-row block per CU, so the blocks take 32 rows.
KEEP_ALL = ((1 << 20),) * 3


@pytest.mark.parametrize("batch", (20, 21, 23, 32, 41))
@pytest.mark.parametrize("wide", (False, True))
def test_selectors_that_keep_everything(oracle, batch, wide):
    """The last block of 4 (20 images, 16-row blocks), 9, 19, 32 and 13 live
    rows; wide: block 5's projection and FFN biases beyond the int32
    epilogues."""
    from heatvit_amd.model import HeatViTModel
    params = synth.pruned_params(keep_biases=KEEP_ALL)
    if wide:
        blocks = list(params.blocks)
        bp = blocks[4]
        far = lambda v, at: np.where(np.isin(np.arange(len(v)), at), (1 << 31) - 1, np.asarray(v))
        blocks[4] = dataclasses.replace(
            bp, mhsa=dataclasses.replace(bp.mhsa, bproj=far(bp.mhsa.bproj, [3, 191])),
            ffn=dataclasses.replace(bp.ffn, b1=far(bp.ffn.b1, [5, 300, 767]),
                                    b2=far(bp.ffn.b2, [0, 100])))
        params = dataclasses.replace(params, blocks=tuple(blocks))
    images = synth.pruned_workload(batch)[0]
    res = HeatViTModel().infer_batch(images, params)
    logits, counts, status, warnings = oracle.model_infer_batch(images, params, threads=8)
    assert not status.any() and (counts == 197).all()
    assert np.array_equal(res.logits, logits)
    assert np.array_equal(res.token_counts, counts)
    assert np.array_equal(res.warnings, warnings)


@pytest.mark.parametrize("batch", (21, 32, 41))
def test_kept_tokens_do_not_take_a_second_round(batch):
    """The FFN launches of a forward whose selectors keep every token against
    those of the unpruned model (32-row blocks at these sizes, the same rows):
    a second round of 16-row blocks took 1.3 times as long."""
    import torch

    from heatvit_amd import _lib
    from heatvit_amd.model import Engine
    L = _lib.lib()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert 16 * cus < 197 * batch <= 32 * cus
    keep = synth.pruned_params(keep_biases=KEEP_ALL)
    images = torch.randint(-128, 128, (batch, 224 * 224 * 3), dtype=torch.int8, device="cuda")

    def ffn_ms(params):
        engine = Engine(params, batch)
        times = []
        for _ in range(12):
            L.hv_profile_enable(1)
            try:
                engine.forward(images)
                ms = np.zeros(len(_lib.PROF_CLASSES), np.float32)
                n = np.zeros(len(_lib.PROF_CLASSES), np.int32)
                _lib.check(L.hv_profile_read(ms.ctypes.data, n.ctypes.data, len(ms)), "profile")
            finally:
                L.hv_profile_enable(0)
            assert n[_lib.PROF_CLASSES.index("ffn")] == 12
            times.append(float(ms[_lib.PROF_CLASSES.index("ffn")]))
        return min(times)

    kept, unpruned = ffn_ms(keep), ffn_ms(synth.unpruned_control(keep))
    print(f"FFN of a forward: {kept:.4f} ms kept, {unpruned:.4f} ms unpruned")
    assert kept < 1.15 * unpruned, (kept, unpruned)
