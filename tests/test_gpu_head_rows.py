"""The head's launch reads the last tokens' rows where they lie (no gather ahead of it): a prompt step's logits against the oracle's."""
import numpy as np
import pytest

from oracle import model as om
from tests.test_gpu_engine import check_logits, prefill_inputs, simple_tables, small_cfg
from vllm_rs_amd.engine import Engine

pytestmark = pytest.mark.gpu


# rows of kernel A (1..3; small heads: up to 7), of the dense kernel W (two row tiles from 17) and of the general product behind a gather (33)
@pytest.mark.parametrize("vocab", [512, 4096])
@pytest.mark.parametrize("seqs", [1, 3, 4, 16, 17, 32, 33])
def test_last_rows_against_the_oracle(seqs, vocab):
    cfg = small_cfg(vocab_size=vocab)
    w = om.make_random_checkpoint(cfg, 3)
    r = np.random.default_rng(seqs)
    prompts = [r.integers(1, vocab - 1, size=int(n)).tolist() for n in r.integers(1, 9, seqs)]
    bt = simple_tables([len(p) for p in prompts])
    eng = Engine(cfg, num_gpu_blocks=64, max_num_seqs=64, max_model_len=512, use_graph=False).load_weights(w)
    args = prefill_inputs(prompts, bt)
    ids, pos, slots, ctx, cu = args
    ref = om.OracleModel(cfg, w, num_blocks=64).forward(ids, pos, slots, bt, ctx, cu)
    check_logits(eng.forward_raw(ids, pos, slots, bt, ctx, cu), ref, f"{seqs} last rows, {vocab} columns")
    eng.close()
