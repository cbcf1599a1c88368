"""Results and prompts of every size through the pinned staging of a model.

Downloads travel in chunks of 1 MiB, two in flight, and are checked for
non-finite values on the host (up to 98304 values) or on the device; uploads up
to 1 MiB are staged.  The sizes around those lines against the same rows asked
for in small calls, and the error path of both checks.
"""
import ctypes

import numpy as np
import pytest

import grokking_abmod_amd as G
import oracle_lib as O

pytestmark = pytest.mark.gpu

SHAPE = dict(vocab_size=256, context=4, width=64, heads=4, layers=1, attention_mesh_depth=2, ffn_mesh_depth=2)


# rows of 256 logits: 98304 values and four rows more, one chunk, a row either
# side of it, two chunks and more than two, whole and ragged
@pytest.mark.parametrize("rows", [4, 128, 132, 384, 388, 1020, 1024, 1028, 2048, 2052, 5000])
def test_downloads_of_every_size(rows):
    tokens = np.random.default_rng(rows).integers(0, 256, rows).astype(np.uint32)
    with G.MeshGpt(0, G.GptConfig(**SHAPE), 7) as model:
        whole = model.logits(tokens, 4)
        hidden = model.hidden_states(tokens, 4)
        for at in (0, rows // 8 * 4, rows - 4):
            assert np.array_equal(whole[at:at + 4], model.logits(tokens[at:at + 4], 4))
            assert np.array_equal(hidden[at:at + 4], model.hidden_states(tokens[at:at + 4], 4))


@pytest.mark.parametrize("batch,n", [(1, 1), (3, 5), (256, 1024), (300, 1000)])
def test_prompts_and_tokens_of_every_size(batch, n):
    """Up to more than the 1 MiB that is staged: the prompts come back as they went."""
    cfg = G.GptConfig(**dict(SHAPE, context=1024, width=16, heads=2))
    prompts = np.random.default_rng(n).integers(0, 256, (batch, n)).astype(np.uint32)
    with G.MeshGpt(0, cfg, 7, max_batch=batch) as model:
        got = model.generate_tokens(prompts, 0, 0.0, 7)
        assert np.array_equal(got, prompts)
        got = model.generate_tokens(prompts, 1, 0.5, 3)
        assert np.array_equal(got[:, :n], prompts)
        alone = model.generate_tokens(prompts[-1:], 1, 0.5, 3 + batch - 1)
        assert np.array_equal(got[-1:], alone)


@pytest.mark.parametrize("rows", [8, 4000])
def test_nonfinite_results_leave_the_output_alone(rows):
    """Either check refuses the result before anything is written, and the model goes on."""
    cfg = G.GptConfig(**SHAPE)
    tokens = np.random.default_rng(1).integers(0, 256, rows).astype(np.uint32)
    with G.MeshGpt(0, cfg, 7) as model:
        good = model.logits(tokens, 4)
        weights = model.parameters()
        bad = weights.copy()
        start = O.group_offsets(O.config(**SHAPE))[3]
        bad[start:start + 2 * 64 * 2] = 3e38
        model.set_parameters(bad)
        out = np.full((rows, 256), 7.0, np.float32)
        status = G.lib().mg_logits(model._h, tokens.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), rows, 4, 0,
                                   out.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), out.size)
        assert status == G.MG_NONFINITE and (out == 7.0).all()
        model.set_parameters(weights)
        assert np.array_equal(model.logits(tokens, 4), good)
        status = G.lib().mg_logits(model._h, tokens.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), rows, 4, 0,
                                   out.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), out.size - 1)
        assert status == G.MG_INVALID_ARGUMENT
