"""The final norm of layer stacks adds the last layer's parts itself, to the rows whose logits are wanted (csrc/stack_ops.hip, StkNormArgs::rows): the bits of the
sum over all rows, the gather and the norm behind them, which a step with the layer trace on still runs.  Parallel blocks with a dense, a mixed and no
feed-forward in the last layer, sequential blocks, rows of whole quads and others, wider than what stays in registers; all rows, some in any order, one."""
import numpy as np
import pytest

from tests import gaperax_oracle as go
from tests import stack_oracle as so
from tests import test_gpu_gaperax as gx
from tests import test_gpu_stack as st

pytestmark = pytest.mark.gpu


def parallel(width, last, groups=1):
    layers = [dict(type="attention", mixer=st.mixer(), mlp=dict(kind="dense", ff=40)), dict(type="attention", mixer=st.mixer(), mlp=last)]
    return dict(architecture="Ditilix", width=width, vocab=90, residual_mult=0.4, logit_scale=0.7, norm=dict(eps=1e-5, groups=groups), layers=layers)


MODELS = {"dense": (so, lambda: parallel(96, dict(kind="dense", ff=72), 3)), "mixture": (so, lambda: parallel(96, st.moe())), "mixture alone": (so, lambda: parallel(50, st.moe(shared=None))),
          "none": (so, lambda: parallel(50, None)), "wide": (so, lambda: parallel(2560, dict(kind="dense", ff=64))), "sequential": (go, gx.config_a), "sequential odd": (go, gx.config_b)}


@pytest.mark.parametrize("dt", [st.F32, st.BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("name", MODELS)
def test_chosen_rows_have_the_bits_of_all_rows(name, dt):
    oracle, cfg = MODELS[name][0], MODELS[name][1]()
    eng = st.build(cfg, oracle.random_tensors(cfg, 5), dt, blocks=12, max_model_len=256)
    r = np.random.default_rng(len(name))
    toks = [r.integers(0, cfg["vocab"], n).tolist() for n in (37, 1, 70)]
    try:
        for want in ([list(range(len(t))) for t in toks], [[36, 0, 5], [0], [69]], [[len(t) - 1] for t in toks]):
            runs = []
            for traced in (True, False):
                eng.layer_trace(traced)
                first = eng.replay_step([(i, t, w) for i, (t, w) in enumerate(zip(toks, want))])
                one = eng.replay_step([(i, [3 + i], [0]) for i in range(3)], [0, 1, 2])  # (a decode step behind it)
                runs.append(np.concatenate([first, one]).view(np.uint32))
            assert np.array_equal(*runs) and runs[0].any(axis=1).all()
    finally:
        eng.layer_trace(False)
        eng.close()
