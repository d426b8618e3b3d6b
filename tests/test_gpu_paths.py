"""GPU parity at the edges of kernels that are picked by size: each case sits
where a variant's tiles, remainders or limits can go wrong, and is checked
against the CPU oracle or a float64 product, at the bars of the tests of the
same path."""
import numpy as np
import pytest

from rustane_amd.engine import ModelWeights

from helpers import random_gammas, small_cfg
from test_gpu_backward import _run

pytestmark = pytest.mark.gpu


def test_embedding_gradient_of_repeated_tokens(orc):
    """Ids that occur 1, 3, 4, 5, 15, 16, 17 and 67 times (the embedding
    backward sums a token's positions 16, 4 and 1 at a time), at a width whose
    columns end inside a block (640 = 512 + 128)."""
    cfg = small_cfg(dim=640, hidden=512, heads=5, hd=128, nlayers=1, vocab=256, seq=64)
    w = random_gammas(ModelWeights.normal(cfg, seed=301, std=0.05), 302)
    rng = np.random.default_rng(303)
    ids = np.repeat(np.array([0, 7, 19, 33, 90, 128, 200, 255], np.uint32), [1, 3, 4, 5, 15, 16, 17, 67])
    tok = rng.permutation(ids).reshape(2, 64).astype(np.uint32)
    tgt = rng.integers(0, cfg.vocab, size=tok.shape).astype(np.uint32)
    _run(orc, cfg, w, np.ascontiguousarray(tok), tgt)
