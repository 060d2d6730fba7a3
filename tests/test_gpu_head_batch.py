"""The batched head (one pass over the table for up to 16 sequences, the
products on the 4x4x1 MFMA) at the edges of its vector groups (1..16
sequences in fours) and table sizes, f16 and f32 tables: every sequence's
logits as its own single-sequence call gives them, bit for bit."""
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
