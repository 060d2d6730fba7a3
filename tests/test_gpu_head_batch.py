"""The batched head (one pass over the table for up to 16 sequences, the
products on the 4x4x1 MFMA) at the edges of its vector groups (1..16
sequences in fours) and table sizes, f16 and f32 tables: every sequence's
logits as its own single-sequence call gives them, bit for bit."""
import json

import numpy as np
import pytest

from fieldrun_amd import Bundle, Gemma, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("embed,vocab,d", [("f16", 63, 128), ("f16", 1030, 96), ("f32", 517, 64), ("f32", 64, 160)])
def test_head_batch_matches_single(ctx, tmp_path, embed, vocab, d):
    stem = str(tmp_path / "g")
    synth.write_gemma2_bundle(stem, 3, n_layer=1, n_head=2, n_kv=1, hd=32, d=d, ffn=64, vocab=vocab, std=0.2,
                              embed=embed)
    b = Bundle(stem, ctx)
    g = Gemma(b)
    prompts = np.stack([synth.gpt2_prompt(4, vocab, 7 + i) for i in range(16)])
    one = [g.generate(p, 3, with_logits=True) for p in prompts]
    for nb in (2, 3, 4, 5, 8, 9, 12, 13, 16):
        toks, lg = g.generate_batch(prompts[:nb], 3, with_logits=True)
        for i in range(nb):
            assert np.array_equal(toks[i], one[i][0]), (nb, i)
            assert np.array_equal(lg[i].view(np.uint32), one[i][1].view(np.uint32)), (nb, i)
    g.free()
    b.close()


def test_head_batch_subnormal_products(ctx, tmp_path):
    """Table rows of subnormal values: their products are subnormal too, and
    the matrix cores keep them as the single-sequence head's multiplies do."""
    vocab, d = 200, 64
    stem = str(tmp_path / "s")
    synth.write_gemma2_bundle(stem, 5, n_layer=1, n_head=2, n_kv=1, hd=32, d=d, ffn=64, vocab=vocab, std=0.2,
                              embed="f32")
    at = next(e["offset"] for e in json.load(open(stem + ".fieldrun.json"))["arrays"] if e["name"] == "embed")
    blob = np.memmap(stem + ".fieldrun.bin", np.uint8, "r+")
    embed = blob[at:at + vocab * d * 4].view(np.float32).reshape(vocab, d)
    embed[100:150] *= np.float32(1e-38)
    embed[150:] *= np.float32(1e-42)
    blob.flush()
    b = Bundle(stem, ctx)
    g = Gemma(b)
    prompts = np.stack([(np.arange(4) * 7 + i) % 100 for i in range(5)])
    toks, lg = g.generate_batch(prompts, 1, with_logits=True)
    tiny = np.abs(lg[:, 0, 100:])
    assert ((tiny > 0) & (tiny < np.finfo(np.float32).tiny)).mean() > 0.5
    for i in range(5):
        t1, l1 = g.generate(prompts[i], 1, with_logits=True)
        assert np.array_equal(toks[i], t1) and np.array_equal(lg[i].view(np.uint32), l1.view(np.uint32)), i
    g.free()
    b.close()
