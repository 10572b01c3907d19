"""Qwen3.5's recurrence over batches: prompts whose lengths are not multiples of the conv kernel's
four-token groups or that are shorter than the conv, then continued (the conv's first inputs come
from the ring, the state from either half), against the oracle bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from brisk_hip import HipSession, model, synth  # noqa: E402
import pyoracle  # noqa: E402


# tiny-qwen35: 64-wide states, 4 taps; tiny-qwen35w: 128-wide, 3 taps
@pytest.mark.parametrize("name", ["tiny-qwen35", "tiny-qwen35w"])
@pytest.mark.parametrize("lengths", [(2, 2, 1, 3), (3, 5, 2), (515, 6)], ids=lambda v: "+".join(map(str, v)))
def test_recurrence_batches(name, lengths):
    f, cfg, table = model.load(synth.model_path(name))
    total = sum(lengths)
    print(f"[recurrence] {name}: {lengths}", flush=True)
    prompt = synth.prompt_ids(total, cfg.vocab, seed=17)
    o = pyoracle.Oracle(cfg, table, total + 8)
    with HipSession((f, cfg, table), max_context=total + 8) as s:
        at = 0
        for n in lengths:
            got, want = s.eval(prompt[at:at + n]), o.eval(prompt[at:at + n])
            np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32), err_msg=f"at {at}")
            at += n
    o.close()
