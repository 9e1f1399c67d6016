"""GPU: the decoder's LM head on both sides of the vocabulary from which batches of at most 8 rows stream
the matrix (three quarters of the CUs' worth of row tiles): logits and greedy tokens against the decoder oracle, with
runs that cut row tiles and a last tile of 9 rows."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = 5e-4  # as the decoder tests with f32 cache rows


@pytest.mark.parametrize("vocab,B", [(16393, 3), (49127, 1), (49127, 8), (49161, 1), (49161, 8), (70009, 5)])
def test_lm_head_vocabulary_rule(oracle, vocab, B):
    from burnext_amd import decoder as D
    cfg = D.GptOssConfig(vocab_size=vocab, d_model=256, n_layers=1, n_heads=8, head_dim=32, kv_heads=2, ffn_hidden=64, num_experts=4,
                         experts_per_token=2, cache_len=40, window=8, max_seq_len=128)
    data = D.make_decoder(cfg, seed=19, sinks_std=0.8, norm_std=0.1, moe_dtype="f32")
    print(f"[lm head] vocab={vocab} B={B}", flush=True)
    dev, orc = D.GptOssDecoder(data, max_batch=B), oracle.DecoderOracle(data, B)
    tok = np.random.default_rng(4).integers(0, vocab, B).astype(np.int32)
    for pos in range(2):
        nxt, lg = dev.decode(torch.from_numpy(tok).cuda(), pos, logits=True)
        o_nxt, o_lg, _ = orc.step(tok, pos)
        got = lg.cpu().numpy()
        assert oracle.max_abs_rel(got, o_lg) <= TOL
        assert np.array_equal(nxt.cpu().numpy(), got.argmax(1))  # lowest index on ties
        tok = o_nxt
    dev.close()
