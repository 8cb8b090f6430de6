"""Prompts of a batch that share prompt passes: every row's ids equal a run of its own, where prompts
of one token, of a chunk of 64, of 63 and 65, more prompts than one pass takes (32), and prompts longer
than a pass (1024 tokens, then a rest that shares a pass with the next rows) meet; a second turn
continues the rows' caches at different positions.  4 rows and 5 are the two sides of the choice
between the decode step's launch sequences, 40 a second row group of 8.  Both of those runs share kernels,
so rows of shared passes are also compared with the oracle."""
import numpy as np
import pytest

import oracle as O
import q35

pytestmark = pytest.mark.gpu


def dims():
    return q35.make_dims(hidden=512, ffn=1536, vocab=8192, n_layers=4, lin_heads=4, attn_heads=4, kv_heads=2)


@pytest.mark.parametrize("lens", [[9, 4, 30, 2], [1, 64, 63, 65, 2, 3, 17], [5] * 40, [1100, 3, 70, 1025, 30]])
def test_batch_prompts_share_passes(lens):
    print(f"[batch prompts] {len(lens)} rows, longest {max(lens)}", flush=True)
    d, n_new, second = dims(), 6, 9
    rng = np.random.default_rng(len(lens))
    prompts = [rng.integers(0, d.vocab, n).astype(np.int32) for n in lens]
    turn2 = [rng.integers(0, d.vocab, second + r % 3).astype(np.int32) for r in range(len(lens))]
    tmax = max(lens) + 2 * n_new + second + 8
    m = q35.TextForCausalLM(d, seed=3, tmax=tmax)
    bt = q35.BatchDecoder(m, len(lens), tmax)
    toks, _ = bt.generate(prompts, n_new, prefill=True)
    toks2, _ = bt.generate(turn2, n_new, prefill=True)
    for r in range(len(lens)):
        m.reset()
        want, _ = m.generate(prompts[r], n_new, mode="persistent", prefill=True)
        want2, _ = m.generate(turn2[r], n_new, mode="persistent", prefill=True)
        np.testing.assert_array_equal(toks[r], want, err_msg=f"row {r}")
        np.testing.assert_array_equal(toks2[r], want2, err_msg=f"row {r}, second turn")
    bt.close()
    m.close()


@pytest.mark.parametrize("lens", [[9, 4, 30, 2], [1, 64, 63, 65, 2, 3, 17]])
def test_batch_prompts_match_oracle(lens):
    """Rows of a shared prompt pass, then decoded: each the oracle's ids for its own prompt."""
    print(f"[batch prompts oracle] {len(lens)} rows", flush=True)
    d, n_new, seed = dims(), 8, 3
    rng = np.random.default_rng(60 + len(lens))
    prompts = [rng.integers(0, d.vocab, n).astype(np.int32) for n in lens]
    tmax = max(lens) + n_new + 8
    m = q35.TextForCausalLM(d, seed=seed, tmax=tmax)
    bt = q35.BatchDecoder(m, len(lens), tmax)
    toks, _ = bt.generate(prompts, n_new, prefill=True)
    for r, p in enumerate(prompts):
        ref = O.Model(O.cfg_from_dims(d), lambda name, n: q35.synth_model_tensor(d, seed, name, n), tmax)
        want, margins = ref.generate(p, n_new)
        np.testing.assert_array_equal(toks[r], want, err_msg=f"row {r}, smallest oracle margin {margins.min():.3g}")
    bt.close()
    m.close()
