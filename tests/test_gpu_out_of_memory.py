"""A call whose buffers do not fit the device fails with RH_ENOMEM and leaves the
context usable: the next call of an ordinary size allocates what it needs again
and gives the same bits as before."""
import numpy as np
import pytest

from rustane_amd import hip_bridge as hb

from helpers import small_cfg, tokens_uniform

pytestmark = pytest.mark.gpu


def test_forward_after_a_workspace_that_does_not_fit():
    # 360000 tokens x 262144 logits x 4 bytes = 377 GB, more than the device holds
    cfg = small_cfg(dim=128, hidden=128, heads=2, hd=64, nlayers=1, vocab=262144, seq=300)
    tok, tgt = tokens_uniform(400, cfg.vocab, 1, 64)
    with hb.Context(cfg.to_rh(), 0, 1200, 0) as c:
        want = c.forward(tok, tgt)
        for n in (1, 2):  # the second failure finds the first one's leftovers
            with pytest.raises(hb.HipBridgeError) as e:
                c.forward(np.zeros((1200, 300), np.uint32), want_logits=False)
            assert e.value.code == hb.RH_ENOMEM
            got = c.forward(tok, tgt)
            assert np.array_equal(got.logits, want.logits) and np.array_equal(got.token_losses, want.token_losses), n


def test_gradients_after_training_buffers_that_do_not_fit():
    # 1.2 million tokens x 65536: the forward's gate is 157 GB and fits, the two kept pre-activations, 315 GB, do not
    cfg = small_cfg(dim=128, hidden=65536, heads=2, hd=64, nlayers=1, vocab=512, seq=300)
    tok, tgt = tokens_uniform(401, cfg.vocab, 1, 70)
    big = np.zeros((4000, 300), np.uint32)
    with hb.Context(cfg.to_rh(), 0, 4000, 0) as c:
        c.forward_backward(tok, tgt, 256.0)
        want = c.read_grads()
        for n in (1, 2):
            with pytest.raises(hb.HipBridgeError) as e:
                c.forward_backward(big, big, 256.0)
            assert e.value.code == hb.RH_ENOMEM
            c.zero_grads()
            c.forward_backward(tok, tgt, 256.0)
            got = c.read_grads()
            flat = [[g[0], g[1], *g[2][0]] for g in (got, want)]
            assert all(np.array_equal(a, b) for a, b in zip(*flat)), n
