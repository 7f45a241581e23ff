"""GPU parity of the attention kernel's work splits: four or eight wavefronts
per workgroup and one to four workgroups per (image, head), chosen from the
image count and from whether other batches are in flight.  The batches sit on both sides of each change of split on a
256-CU device and their images at the edges of the 16-query and 32-row tiles
(images with fewer query tiles than workgroups among them); every output is
compared with the CPU oracle, bit for bit."""

import numpy as np
import pytest

from heatvit_amd import synth

pytestmark = pytest.mark.gpu

EDGES = (197, 1, 16, 17, 32, 33, 48, 63, 64, 65, 96, 128, 129, 192, 193)


def _lengths(batch):
    return [EDGES[i % len(EDGES)] for i in range(batch)]


@pytest.mark.parametrize("batch", (1, 21, 22, 128, 129))
def test_attention_over_given_qkv(oracle, batch):
    from heatvit_amd.ops import attention
    from test_gpu_attention import peaky_qkv
    rng = np.random.default_rng(batch)
    m = synth.block_workload()[1].mhsa
    exps = (m.qkv_out_scale_exp, m.score_scale_exp, m.prob_scale_exp, m.context_out_scale_exp)
    qkvs = [peaky_qkv(rng, n) for n in _lengths(batch)]
    got = _context(qkvs, exps)
    for i, q in enumerate(qkvs):
        want = oracle.attention(q, *exps)[2]
        assert np.array_equal(got[i], want), (batch, i, len(q))


@pytest.mark.parametrize("exponents", range(6))
@pytest.mark.parametrize("batch", (15, 30, 129))
def test_attention_exponents_over_given_qkv(oracle, batch, exponents):
    """The score and context exponents of test_gpu_attention's sweep, whose
    launches with score and prob outputs keep four wavefronts, on four parts of
    eight, two parts, and four wavefronts without those outputs."""
    from test_gpu_attention import EXPS, peaky_qkv
    assert len(EXPS) == 6
    rng = np.random.default_rng(7 * batch + exponents)
    qkvs = [peaky_qkv(rng, n) for n in _lengths(batch)]
    got = _context(qkvs, EXPS[exponents])
    for i, q in enumerate(qkvs):
        assert np.array_equal(got[i], oracle.attention(q, *EXPS[exponents])[2]), (i, len(q))


def _context(qkvs, exps):
    """The context rows of hv_attention_i8 without score and prob outputs
    (whose launches keep four wavefronts), and its status."""
    import torch

    from heatvit_amd import _lib
    lens = [len(q) for q in qkvs]
    offsets = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    qkv = torch.from_numpy(np.concatenate(qkvs)).cuda()
    off = torch.from_numpy(offsets).cuda()
    ctx = torch.empty((int(offsets[-1]), 192), dtype=torch.int8, device="cuda")
    status = torch.full((len(qkvs),), -1, dtype=torch.int32, device="cuda")
    _lib.check(_lib.lib().hv_attention_i8(
        qkv.data_ptr(), off.data_ptr(), len(qkvs), int(offsets[-1]), ctx.data_ptr(), None, None,
        *exps, status.data_ptr(), torch.cuda.current_stream().cuda_stream), "attention")
    assert not status.cpu().numpy().any()
    host = ctx.cpu().numpy()
    return [host[offsets[i]:offsets[i + 1]] for i in range(len(qkvs))]


@pytest.mark.parametrize("batch", (32, 42, 43, 85, 86))
def test_block_with_qkv_in_the_attention_kernel(oracle, batch):
    from heatvit_amd.transformer import transformer_block_batch
    rng = np.random.default_rng(100 + batch)
    bp = synth.block_workload()[1]
    xs = [rng.integers(-128, 128, (n, 192)).astype(np.int8) for n in _lengths(batch)]
    zs = transformer_block_batch(xs, bp)
    for i, x in enumerate(xs):
        want, _ = oracle.transformer_block(x, bp, checkpoints=False)
        assert np.array_equal(zs[i], want), (batch, i, len(x))


@pytest.mark.parametrize("batch", (1, 3, 22, 43))
def test_model_of_few_images(oracle, batch):
    from heatvit_amd.model import HeatViTModel
    images, params = synth.pruned_workload(batch)
    res = HeatViTModel().infer_batch(images, params)
    logits, counts, status, warnings = oracle.model_infer_batch(images, params, threads=8)
    assert not status.any()
    assert np.array_equal(res.logits, logits)
    assert np.array_equal(res.token_counts, counts)
    assert np.array_equal(res.warnings, warnings)


@pytest.mark.parametrize("batch", (42, 85))
def test_pipelined_forwards_do_not_repeat_keys_and_values(batch):
    """Three unpruned batches in flight: with HV_FWD_PIPELINED the attention
    splits as if it had half the CUs, since the other batches fill them.  Split
    by the batch alone, Pipeline's forwards took 1.13 and 1.10 times as long as
    those of three engines without the option on streams of their own; now
    1.02 and 0.99."""
    import time

    import torch

    from heatvit_amd.model import Engine, Pipeline
    params = synth.unpruned_control(synth.pruned_params())
    images = [torch.randint(-128, 128, (batch, 224 * 224 * 3), dtype=torch.int8, device="cuda")
              for _ in range(3)]
    pipe = Pipeline(params, batch, depth=3)
    engines = [Engine(pipe.engines[0].model, batch) for _ in range(3)]
    streams = [torch.cuda.Stream() for _ in range(3)]

    def plain():
        for e, s, x in zip(engines, streams, images):
            with torch.cuda.stream(s):
                e.forward(x)

    def pipelined():
        for x in images:
            pipe.submit(x)

    def best(fn):
        times = []
        for i in range(8):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(10):
                fn()
            torch.cuda.synchronize()
            times.append(time.perf_counter() - t0)
        return min(times)

    best(plain), best(pipelined)
    a, b = best(plain), best(pipelined)
    print(f"{batch} images: {a * 1e5:.1f} us per round plain, {b * 1e5:.1f} pipelined")
    for e, p in zip(engines, pipe.engines):
        assert torch.equal(e.logits[:batch], p.logits[:batch])
    assert b < 1.06 * a, (a, b)
