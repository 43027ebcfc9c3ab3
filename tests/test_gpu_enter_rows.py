"""The launch a pass starts with (look-up, first norm, schedule): every embedding format, rows of one workgroup's width and of more
than it takes in one walk, a row beyond its LDS (which goes through the general operators), and a token outside the vocabulary."""
from dataclasses import replace

import numpy as np
import pytest

from test_gpu_forward import dev, hip, rel_rms  # noqa: F401  (a fixture among them)

pytestmark = pytest.mark.gpu


def one_block(hidden, dtype):
    from guffin_amd import model, synth
    return replace(model.GEMMA3_12B, layers=1, hidden=hidden, ffn=512, q_heads=2, kv_heads=1, vocab=1024, ring_global=1024,
                   dtypes=(synth.Q8_0,) * 7, embed_dtype=dtype)


@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("hidden,fmt", [(256, "Q8_0"), (320, "Q8_0"), (256, "Q6_K"), (1280, "Q4_K"), (4352, "Q6_K"), (16128, "Q8_0"), (16384, "Q8_0")])
def test_one_block_matches_the_oracle(hip, gfo, hidden, fmt, rows):  # noqa: F811
    from guffin_amd import model, synth
    host = model.HostModel(one_block(hidden, getattr(synth, fmt)), seed=hidden + rows, position=9)
    devm = model.DeviceModel.from_host(host)
    tokens = np.array([1023, 4][:rows], np.uint32)
    want, _, _ = gfo.forward(host, tokens, 9, threads=8)
    hidden_rows, _, _, _, status = devm.forward(dev(tokens), 9)
    assert int(status.item()) == 0
    assert rel_rms(hidden_rows.cpu().numpy(), want) <= 1e-3


def test_a_token_outside_the_vocabulary_is_flagged(hip):  # noqa: F811
    from guffin_amd import model, synth
    devm = model.DeviceModel.from_host(model.HostModel(one_block(256, synth.Q8_0), seed=1, position=9))
    good = devm.forward(dev(np.array([0], np.uint32)), 9)
    bad = devm.forward(dev(np.array([1024], np.uint32)), 9)
    assert int(good[4].item()) == 0 and int(bad[4].item()) != 0
    assert np.array_equal(good[0].cpu().numpy(), bad[0].cpu().numpy())   # read as token 0
