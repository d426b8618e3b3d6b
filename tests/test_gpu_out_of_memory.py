"""A call whose buffers do not fit the device fails with RH_ENOMEM and leaves
the context usable: the next call of an ordinary size allocates what it needs
again and gives the same bits as before."""
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
