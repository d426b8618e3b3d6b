"""GPU parity at the edges of kernels that are picked by size: each case sits
where a variant's tiles, remainders or limits can go wrong, and is checked
against the CPU oracle or a float64 product, at the bars of the tests of the
same path."""
import ctypes

import numpy as np
import pytest

from rustane_amd import hip_bridge as hb
from rustane_amd import hip_rt
from rustane_amd.engine import ModelWeights

from helpers import LOGIT_ATOL, random_gammas, small_cfg, tokens_uniform
from test_gpu_backward import _run
from test_gpu_gemm_tiles import (CFGS, EPI_F32, EPI_QKV, EPI_SWIGLU, close, frag_pack, frag_unpack, lib,  # noqa: F401
                                 operands, ptr, run, swiglu_ref, up16)

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


@pytest.mark.parametrize("vocab,ids", [(128, [0, 127]), (2048, [0, 1, 1024, 2047]), (2052, [3, 2047, 2048, 2051]),
                                       (6152, [0, 1, 2047, 2048, 2049, 4095, 4096, 4097, 6144, 6151])])
def test_embedding_gradient_index(orc, vocab, ids):
    """Ids on either side of the index's 11-bit sort digits, equal in one digit
    and not in the other, and a vocabulary that one pass covers."""
    cfg = small_cfg(dim=128, hidden=128, heads=1, hd=128, nlayers=1, vocab=vocab, seq=40)
    w = random_gammas(ModelWeights.normal(cfg, seed=304, std=0.05), 305)
    rng = np.random.default_rng(306)
    tok = rng.choice(np.array(ids, np.uint32), size=(2, 40))
    _run(orc, cfg, w, tok, rng.integers(0, vocab, size=tok.shape).astype(np.uint32))


@pytest.mark.parametrize("K", [128, 256, 384, 640, 1152])
@pytest.mark.parametrize("name", ["D8_256x256", "D8_256x256_SK", "D8_256x128", "D8_256x128_SK"])
def test_ping_pong_step_counts(lib, name, K):  # noqa: F811
    """k loops shorter than the stage ring, ending on each of its buffers."""
    x, w, y = operands(21, 270, 520, K)
    out = np.zeros((270, 520), np.float32)
    run(lib, EPI_F32, CFGS[name], x, w, io=out)
    close(out, y, 1e-5, f"{name} K {K}")


# The 256x128 tile without ping-pong, which short k loops take: plain and SwiGLU
# stores with ragged rows and columns and 4 - 32 k steps, and picked by size (one
# round of 252 tiles) at the last K that takes it and the first that does not.
@pytest.mark.parametrize("cfg,M,N,K", [(28, 270, 520, 128), (28, 129, 1000, 640), (28, 128, 256, 1024),
                                       (0, 192, 32004, 1024), (0, 192, 32004, 1152)])
def test_short_k_tile(lib, cfg, M, N, K):  # noqa: F811
    x, w, y = operands(28, M, N, K)
    out = np.full((M, N), np.nan, np.float32)
    run(lib, EPI_F32, cfg, x, w, io=out)
    close(out, y, 1e-5, f"store {M} {N} {K}")
    F = N // 256 * 128
    if F:
        out16 = np.zeros(up16(M) * F, np.float16)
        run(lib, EPI_SWIGLU, cfg, x, np.ascontiguousarray(w[:2 * F]), out16=out16)
        close(frag_unpack(out16, M, F), swiglu_ref(y[:, :2 * F])[0], 2e-3, "swiglu")


# Few tokens: token tiles of 16 full and ragged, 64 and the first count past
# it; every choice of row tiles per block (by N), ragged in N; fewer k chunks
# than waves, more, and a remainder.  fp32 sums of K <= 1408 products: 1e-5 of
# max|Y|; fp16 outputs one rounding: 2e-3.
@pytest.mark.parametrize("M", [1, 16, 17, 45, 64, 65])
@pytest.mark.parametrize("N,K", [(996, 128), (1000, 1152), (8204, 384)])
def test_few_tokens_fp32(lib, M, N, K):  # noqa: F811
    x, w, y = operands(22, M, N, K)
    out = np.full((M, N), np.nan, np.float32)
    run(lib, EPI_F32, 0, x, w, alpha=0.5, softcap=30.0, io=out)
    close(out, 30.0 * np.tanh(0.5 * y / 30.0), 1e-5, f"M {M}")


@pytest.mark.parametrize("M", [1, 33, 64])
@pytest.mark.parametrize("F,K", [(128, 128), (4224, 256), (8320, 1408)])
def test_few_tokens_swiglu(lib, M, F, K):  # noqa: F811
    x, w, y = operands(23, M, 2 * F, K)
    out16 = np.zeros(up16(M) * F, np.float16)
    run(lib, EPI_SWIGLU, 0, x, w, out16=out16)
    close(frag_unpack(out16, M, F), swiglu_ref(y)[0], 2e-3, f"M {M} F {F}")


@pytest.mark.parametrize("B,S,H,hd", [(1, 5, 3, 64), (3, 16, 22, 128), (2, 31, 33, 128)])
def test_few_tokens_qkv(lib, B, S, H, hd):  # noqa: F811
    ctx, pos0, K, D = S + 9, 4, 256, H * hd
    x, w, y = operands(24, B * S, 3 * D, K)
    ang = np.random.default_rng(25).uniform(-np.pi, np.pi, (ctx, hd // 2))
    rope = np.stack([np.cos(ang), np.sin(ang)], -1).astype(np.float32)
    q, k, v = (np.zeros((B, H, n, hd), np.float16) for n in (S, ctx, ctx))
    run(lib, EPI_QKV, 0, x, w, qkv=(B, S, H, hd, ctx, pos0, rope, q, k, v))
    y = y.reshape(B, S, 3, H, hd).transpose(2, 0, 3, 1, 4)
    c, s = (rope[pos0:pos0 + S, :, i].astype(np.float64) for i in (0, 1))

    def rot(t):
        e, o = t[..., 0::2], t[..., 1::2]
        return np.stack([e * c - o * s, o * c + e * s], -1).reshape(t.shape)

    close(q, rot(y[0]), 2e-3, "q")
    close(k[:, :, pos0:pos0 + S], rot(y[1]), 2e-3, "k cache")
    close(v[:, :, pos0:pos0 + S], y[2], 2e-3, "v cache")
    assert not k[:, :, :pos0].any() and not k[:, :, pos0 + S:].any()


@pytest.mark.parametrize("M", [1, 45, 64])
@pytest.mark.parametrize("N,K", [(1024, 128), (1024, 1152), (2688, 1408), (8192, 640)])
def test_few_tokens_residual_then_rmsnorm(lib, M, N, K):  # noqa: F811
    eps, alpha = 1e-5, 0.25
    x, w, y = operands(26, M, N, K)
    rng = np.random.default_rng(27)
    x0 = rng.standard_normal((M, N)).astype(np.float32)
    gamma = rng.uniform(0.5, 1.5, N).astype(np.float32)
    io, xn = x0.copy(), np.zeros(up16(M) * N, np.float16)
    rc = lib.rhh_gemm_resid_norm(0, ptr(frag_pack(w)), ptr(frag_pack(x)), M, N, K, alpha, None, ptr(io), ptr(gamma),
                                 eps, ptr(xn))
    assert rc == 0
    x1 = x0.astype(np.float64) + alpha * y
    close(io, x1, 1e-5, "residual")
    close(frag_unpack(xn, M, N), x1 / np.sqrt((x1 * x1).mean(1, keepdims=True) + eps) * gamma, 2e-3, "rmsnorm")


# The row tiles per block of wide models: QKV 5 and 6, W1 | W3 8 (up to 32
# tokens; past them the tile kernel), 6 past 2048 row tiles, the split form 3.
@pytest.mark.parametrize("B,S,H", [(1, 64, 43), (1, 7, 43), (2, 24, 53), (1, 33, 54), (1, 64, 64)])
def test_few_tokens_qkv_wide(lib, B, S, H):  # noqa: F811
    test_few_tokens_qkv(lib, B, S, H, 128)


@pytest.mark.parametrize("M", [1, 17, 32, 33, 64])
@pytest.mark.parametrize("F", [12416, 16384, 16512])
def test_few_tokens_swiglu_wide(lib, M, F):  # noqa: F811
    test_few_tokens_swiglu(lib, M, F, 384)


@pytest.mark.parametrize("M", [1, 33, 64])
@pytest.mark.parametrize("N,K", [(5504, 256), (6144, 1408), (6272, 256)])
def test_few_tokens_residual_then_rmsnorm_wide(lib, M, N, K):  # noqa: F811
    test_few_tokens_residual_then_rmsnorm(lib, M, N, K)


def _decode_matches_forward(cfg, B, p0, steps, seed, max_ctx=0):
    """Teacher-forced decode logits equal the forward's at every position."""
    w = random_gammas(ModelWeights.normal(cfg, seed=seed), seed + 1)
    tok, _ = tokens_uniform(seed + 2, cfg.vocab, B, p0 + steps)
    with hb.Context(cfg.to_rh(), 0, B, max_ctx or p0 + steps) as c:
        c.load_weights(w.embed, w.gamma_final, [lw.tensors() for lw in w.layers])
        want = c.forward(tok).logits
        c.prefill(tok[:, :p0])
        for p in range(p0, p0 + steps):
            got = c.decode_step(tok[:, p], want_logits=True)[1]
            assert np.abs(got - want[:, p]).max() <= LOGIT_ATOL, (B, p)


# RMSNorm inside the decode GEMVs, a wave per token or the block for each:
# rows shorter than a wave's 256 columns, ending inside and on one; fewer
# tokens than waves, as many, more, and a ragged last round.
@pytest.mark.parametrize("heads,B", [(2, 2), (2, 16), (6, 5), (10, 3), (10, 9), (16, 16), (42, 2), (42, 3), (42, 5)])
def test_decode_norm_waves(heads, B):
    cfg = small_cfg(dim=64 * heads, hidden=256, heads=heads, hd=64, nlayers=2, vocab=512, seq=24)
    _decode_matches_forward(cfg, B, 5, 4, 310 + heads + B)


# Decode attention over one chunk (caches up to 512 positions) and several, at
# the first and last positions of each.
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("max_ctx,p0", [(129, 127), (512, 1), (512, 509), (513, 3), (513, 510)])
def test_decode_attention_chunks(hd, max_ctx, p0):
    cfg = small_cfg(dim=2 * hd if hd == 64 else hd, hidden=256, heads=2 if hd == 64 else 1, hd=hd, nlayers=2,
                    vocab=512, seq=64)
    _decode_matches_forward(cfg, 2, p0, min(3, max_ctx - p0), 330 + p0, max_ctx)


# Weight gradients of one input as one product with two or three outputs
# (narrow models), stored and accumulated: 128-wide tiles, whose edges fall on
# the outputs' edges, and dW1 | dW3 of 1024 x 2816 on 192-wide tiles, which
# straddle the two outputs.
@pytest.mark.parametrize("heads,hidden", [(1, 128), (3, 640), (5, 1408), (8, 2816)])
@pytest.mark.parametrize("calls", [1, 2])
def test_joint_weight_gradients(orc, heads, hidden, calls):
    cfg = small_cfg(dim=128 * heads, hidden=hidden, heads=heads, hd=128, nlayers=1, vocab=512, seq=70)
    w = random_gammas(ModelWeights.normal(cfg, seed=340 + heads, std=0.05), 341)
    tok, tgt = tokens_uniform(342, cfg.vocab, 2, cfg.seq)
    _run(orc, cfg, w, tok, tgt, calls=calls)


# 2560 x 6912: up to 512 tokens the first dW1 and dW3 are two products of the
# store-wave kernel on transposed copies, later ones (and longer first ones) one
# product with two outputs, in place.  All sum the tokens in order, and with
# powers of two for the loss scale and the length every scaling is exact: a
# second call on the same batch doubles the gradients to the bit, and a zero
# between a forward and its backward gives the first ones again.
@pytest.mark.parametrize("seq", [128, 256, 512, 1024])
def test_first_and_joint_weight_gradients_agree(seq):
    cfg = small_cfg(dim=2560, hidden=6912, heads=20, hd=128, nlayers=1, vocab=512, seq=seq)
    tok, tgt = tokens_uniform(343, cfg.vocab, 1, seq)
    with hb.Context(cfg.to_rh(), 0, 1, 0) as c:
        c.init_normal(344, 0.02)
        c.forward_backward(tok, tgt, 256.0)
        first = c.read_grads()[2][0]
        c.forward_backward(tok, tgt, 256.0)
        second = c.read_grads()[2][0]
        fwd, _ = c.forward_train(tok, tgt)
        c.zero_grads()
        c.backward(fwd, loss_scale=256.0)
        third = c.read_grads()[2][0]
    for j in range(7):
        assert first[j].any() and np.array_equal(second[j], 2 * first[j]) and np.array_equal(third[j], first[j]), j


def grads_product(lib, cfg, accumulate, x, w, M, N, alpha, outs, part_cols=0, w_off=0, tokens=False):  # noqa: F811
    """x, w: [K][features] with tokens, else [M][K] and [N][K]; outs: one to three output arrays."""
    f, i, p = ctypes.c_float, ctypes.c_int, ctypes.c_void_p
    lib.rhh_gemm_grads.argtypes = [i, i, p, p, i, i, i, i, i, i, f, i, p, p, p]
    K = x.shape[0] if tokens else x.shape[1]
    io = list(outs) + [None] * (3 - len(outs))
    xf, wf = frag_pack(x), frag_pack(w)
    rc = lib.rhh_gemm_grads(cfg, accumulate, ptr(wf), ptr(xf), M, N, K, x.shape[1] if tokens else 0,
                            w.shape[1] if tokens else 0, w_off, alpha, part_cols, *[ptr(o) for o in io])
    assert rc == 0, f"rhh_gemm_grads cfg {cfg}: error {rc}"


PICKED = ["D8_256x256", "D8_256x128", "D8_192x256", "D8_192x128", "D8_128x128"]  # the tile model's choices


# Products over tokens with both operands token-major, every tile the model can
# pick: outputs that end inside a tile and inside a 32-feature block, operand
# rows wider than the product and a W that starts inside its rows (dW3's), k
# loops shorter than the stage rings and ending on each of their buffers, and
# more tiles than CUs or groups of 8 M-tiles.
# fp32 sums of K <= 640 products: 1e-5 of max|Y|.
@pytest.mark.parametrize("M,N,K,trx,trw,w_off", [(4, 4, 128, 128, 128, 0), (600, 700, 128, 640, 768, 32),
                                                 (300, 1000, 256, 384, 1152, 96), (600, 700, 384, 640, 768, 64),
                                                 (300, 516, 640, 384, 640, 0), (2100, 2200, 128, 2176, 2304, 0)])
@pytest.mark.parametrize("name", PICKED)
def test_products_over_tokens(lib, name, M, N, K, trx, trw, w_off):  # noqa: F811
    rng = np.random.default_rng(28)
    x, w = (rng.standard_normal((K, n)).astype(np.float16) for n in (trx, trw))
    y = x[:, :M].T.astype(np.float64) @ w[:, w_off:w_off + N].astype(np.float64)
    cfg = CFGS[name]
    out = np.full((M, N), np.nan, np.float32)
    grads_product(lib, cfg, 0, x, w, M, N, 0.5, [out], w_off=w_off, tokens=True)
    close(out, 0.5 * y, 1e-5, f"{name} store")
    x0 = rng.standard_normal((M, N)).astype(np.float32)
    io = x0.copy()
    grads_product(lib, cfg, 1, x, w, M, N, 0.25, [io], w_off=w_off, tokens=True)
    close(io, x0.astype(np.float64) + 0.25 * y, 1e-5, f"{name} accumulate")


# One product with two or three outputs: output widths below, at and past a
# tile's, so that tiles hold features of two or three outputs, and a last one
# cut short, whose remaining columns stay as they are.
@pytest.mark.parametrize("tokens", [False, True])
@pytest.mark.parametrize("part_cols,N", [(128, 384), (132, 264), (132, 396), (320, 640), (320, 900), (68, 204)])
@pytest.mark.parametrize("name", PICKED)
def test_products_with_several_outputs(lib, name, part_cols, N, tokens):  # noqa: F811
    M, K = 300, 256
    rng = np.random.default_rng(29)
    x = rng.standard_normal((K, 384) if tokens else (M, K)).astype(np.float16)
    w = rng.standard_normal((K, (N + 127) // 128 * 128) if tokens else (N, K)).astype(np.float16)
    xd, wd = (x[:, :M].T, w[:, :N].T) if tokens else (x, w)
    y = xd.astype(np.float64) @ wd.astype(np.float64).T
    n = (N + part_cols - 1) // part_cols
    old = rng.standard_normal((n, M, part_cols)).astype(np.float32)
    for accumulate in (0, 1):
        outs = [o.copy() for o in old]
        grads_product(lib, CFGS[name], accumulate, x, w, M, N, 0.5, outs, part_cols=part_cols, tokens=tokens)
        got = np.concatenate(outs, 1)
        before = np.concatenate(list(old), 1)
        assert np.array_equal(got[:, N:], before[:, N:])
        want = before[:, :N].astype(np.float64) * accumulate + 0.5 * y
        close(got[:, :N], want, 1e-5, f"{name} accumulate {accumulate}")


# Attention backward at head dim 128: lengths that end inside and on a 64-row
# tile, and one, two and several tiles (both stages and the odd last one); six
# heads' tiles do not share out evenly over the XCDs.
@pytest.mark.parametrize("seq", [2, 63, 64, 65, 130, 320])
def test_attention_backward_lengths(orc, seq):
    cfg = small_cfg(dim=384, hidden=256, heads=3, hd=128, nlayers=1, vocab=512, seq=seq)
    w = random_gammas(ModelWeights.normal(cfg, seed=350, std=0.05), 351)
    tok, tgt = tokens_uniform(352 + seq, cfg.vocab, 2, cfg.seq)
    _run(orc, cfg, w, tok, tgt)


# RMSNorm backward with 64, 128 and 256 threads a row: widths ending inside a
# row's groups and on one, and token counts that leave the last block's rows
# partly empty.
@pytest.mark.parametrize("heads,hd,seq", [(2, 64, 9), (4, 128, 13), (5, 128, 9), (8, 128, 15), (9, 128, 7)])
def test_rmsnorm_backward_widths(orc, heads, hd, seq):
    cfg = small_cfg(dim=heads * hd, hidden=256, heads=heads, hd=hd, nlayers=1, vocab=256, seq=seq)
    w = random_gammas(ModelWeights.normal(cfg, seed=360, std=0.05), 361)
    tok, tgt = tokens_uniform(362 + heads, cfg.vocab, 1, cfg.seq)
    _run(orc, cfg, w, tok, tgt)


# Weight gradients of whole 128-token blocks read the token-major operands in
# place (at these sizes), others take transposed copies: token counts on both
# sides, one and several layers (each buffer rewritten a layer after its product
# read it), a vocabulary that ends inside a tile, and (8, 2816), whose dW1 | dW3
# runs on 192-wide tiles that straddle the outputs.
@pytest.mark.parametrize("heads,hidden,nlayers", [(1, 128, 1), (3, 640, 2), (5, 1408, 3), (8, 2816, 1)])
@pytest.mark.parametrize("batch,seq", [(1, 128), (2, 64), (3, 128), (2, 96)])
@pytest.mark.parametrize("calls", [1, 2])
def test_weight_gradients_of_whole_blocks(orc, heads, hidden, nlayers, batch, seq, calls):
    cfg = small_cfg(dim=128 * heads, hidden=hidden, heads=heads, hd=128, nlayers=nlayers, vocab=520, seq=seq)
    w = random_gammas(ModelWeights.normal(cfg, seed=370 + heads, std=0.05), 371)
    tok, tgt = tokens_uniform(372 + seq, cfg.vocab, batch, cfg.seq)
    _run(orc, cfg, w, tok, tgt, calls=calls)


def test_operand_copies_come_with_the_first_ragged_call():
    """The transposed operand copies are allocated by the first token count
    that is no multiple of 128, once, for the largest count seen; calls before
    and after it give the same bits as in a context of their own."""
    cfg = small_cfg(dim=512, hidden=1408, heads=8, hd=64, nlayers=1, vocab=32000, seq=1024)
    copies = (32000 + 8 * 512 + 3 * 1408) * 2048 * 2
    whole, ragged = tokens_uniform(380, cfg.vocab, 2, 1024), tokens_uniform(381, cfg.vocab, 2, 1000)

    def free():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip_rt.rt().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    def grads(c, batch):
        c.zero_grads()
        c.forward_backward(*batch, 256.0)
        g = c.read_grads()
        return [g[0], g[1], *g[2][0]]

    def same(a, b):
        return all(np.array_equal(x, y) for x, y in zip(a, b))

    with hb.Context(cfg.to_rh(), 0, 2, 0) as c:
        c.init_normal(382, 0.02)
        want_ragged = grads(c, ragged)
    with hb.Context(cfg.to_rh(), 0, 2, 0) as c:
        c.init_normal(382, 0.02)
        want_whole = grads(c, whole)
        before = free()
        assert same(grads(c, whole), want_whole) and free() == before
        assert same(grads(c, ragged), want_ragged)
        after = free()
        assert before - after >= copies
        assert same(grads(c, ragged), want_ragged) and same(grads(c, whole), want_whole) and free() == after
