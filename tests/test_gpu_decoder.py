"""GPU parity of the decoder pieces around the MoE block (config 5's prefill):
RoPE, causal attention, the residual / bias adds and the embedding gather,
each through the C ABI against the CPU oracle on the same seeded inputs.

Bar: RoPE, the adds and the gather bit-exact (same table, same roundings);
attention within REL_TOL = 1e-4 normwise relative error (its two products
run on MFMA in another summation order than the oracle's serial loops).
"""
import numpy as np
import pytest

from helpers import assert_close, load_pkg, normal

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as _t
    assert _t.cuda.is_available(), "GPU tests need the MI355X"
    return _t


@pytest.fixture(scope="module")
def pkg():
    return load_pkg()


@pytest.fixture(scope="module")
def ctx(pkg, torch):
    c = pkg.Context(0)
    yield c
    c.close()


def dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def host(t):
    return t.detach().cpu().numpy()


# ------------------------------------------------------------------ RoPE
@pytest.mark.parametrize("B,S,H,KVH,hd,theta", [
    (1, 1, 1, 1, 2, 10000.0), (2, 9, 4, 2, 16, 10000.0), (3, 37, 3, 1, 6, 500000.0),
    (2, 100, 2, 0, 8, 10000.0), (8, 512, 16, 16, 64, 10000.0)])
def test_rope_bit_exact(ctx, torch, orc, B, S, H, KVH, hd, theta):
    print(f"rope B={B} S={S} H={H} KVH={KVH} hd={hd}", flush=True)
    rng = np.random.default_rng(B * 131 + S * 7 + hd)
    q = normal(rng, (B * S, H * hd))
    k = normal(rng, (B * S, max(KVH, 1) * hd))
    qd, kd = dev(torch, q), dev(torch, k)
    ctx.rope(qd, kd, B, S, H, KVH, hd, theta)
    rq, rk = orc.rope(q, k, B, S, H, KVH, hd, theta)
    assert np.array_equal(host(qd), rq)
    assert np.array_equal(host(kd), rk)


def test_rope_longer_table_and_errors(ctx, pkg, torch, orc):
    rng = np.random.default_rng(11)
    B, S, H, hd = 2, 12, 2, 8
    q, k = normal(rng, (B * S, H * hd)), normal(rng, (B * S, H * hd))
    qd, kd = dev(torch, q), dev(torch, k)
    table = ctx.rope_table(10000.0, hd, 64)  # rows past seq_len are never read
    ctx.rope(qd, kd, B, S, H, H, hd, table=table)
    rq, rk = orc.rope(q, k, B, S, H, H, hd)
    assert np.array_equal(host(qd), rq) and np.array_equal(host(kd), rk)
    short = ctx.rope_table(10000.0, hd, S - 1)
    with pytest.raises(pkg.MoeInvalidArgument):
        ctx.rope(qd, kd, B, S, H, H, hd, table=short)
    with pytest.raises(pkg.MoeInvalidArgument):
        ctx.rope(qd, kd, B, S, H, H, 7)


# ------------------------------------------------------------- attention
# (B, S, Hq, Hkv, hd, window): one tile; grouped query heads; a window inside
# one tile and across tiles; several 128-row tiles of a 64-wide head; a
# window of exactly S (unlimited); config 5's full prefill shape.  head_dim
# 64 and 128 take the fused kernel (any S: 1, 37, 200, 300 below), the
# others the batched-GEMM path.
ATTN_CASES = [(1, 16, 1, 1, 16, None), (2, 48, 4, 2, 16, None), (2, 48, 4, 2, 16, 5),
              (1, 160, 2, 1, 64, None), (1, 160, 2, 1, 64, 130), (2, 272, 3, 3, 32, 20),
              (1, 144, 4, 1, 48, 144), (8, 512, 16, 16, 64, None), (3, 1, 2, 1, 64, None),
              (2, 37, 4, 2, 64, None), (1, 300, 2, 2, 128, None), (2, 200, 4, 1, 128, 50),
              (1, 129, 16, 4, 128, 33),
              # the bf16 pieces' eight waves (512 tiles of 128 queries and more
              # at head_dim 128, 1,024 at 64): sequences off their 256-query
              # tiles, grouped heads, windows inside a key block and across them
              (4, 449, 32, 4, 128, None), (4, 400, 32, 32, 128, 21), (16, 31, 32, 2, 128, None),
              (8, 385, 32, 4, 64, 300), (16, 129, 32, 8, 64, None),
              # head_dim 64 about the line to eight waves: 1,536 keys and 1,537, and a
              # window of each in a longer sequence
              (1, 1536, 86, 43, 64, None), (1, 1537, 86, 43, 64, None),
              (1, 1800, 74, 37, 64, 1536), (1, 1800, 74, 37, 64, 1537)]


@pytest.mark.parametrize("B,S,H,KVH,hd,window", ATTN_CASES)
def test_attention_vs_oracle(ctx, torch, orc, B, S, H, KVH, hd, window):
    print(f"attention B={B} S={S} H={H} KVH={KVH} hd={hd} window={window}", flush=True)
    rng = np.random.default_rng(B * 17 + S + H * 5 + hd + (window or 0))
    q = normal(rng, (B * S, H * hd))
    k = normal(rng, (B * S, KVH * hd))
    v = normal(rng, (B * S, KVH * hd))
    out = torch.full((B * S, H * hd), float("nan"), device="cuda")
    ctx.attention(dev(torch, q), dev(torch, k), dev(torch, v), out, B, S, H, KVH, hd,
                  window or 0)
    ref = orc.attention(q, k, v, B, S, H, KVH, hd, window)
    assert_close(host(out), ref, what="attention")


@pytest.mark.parametrize("B,S,H,KVH,hd", [(2, 70, 2, 1, 64), (4, 385, 32, 4, 128),
                                          (8, 385, 32, 4, 64)])
def test_attention_values_the_pieces_do_not_hold(ctx, torch, orc, B, S, H, KVH, hd):
    """One tile's infinities, NaN, huge and tiny values leave every other
    sequence and head as it was, and give what the fp32 loop gives."""
    rng = np.random.default_rng(hd + S)
    q = normal(rng, (B * S, H * hd))
    k = normal(rng, (B * S, KVH * hd))
    v = normal(rng, (B * S, KVH * hd))
    v[S // 2, 0] = np.nan                        # sequence 0, key head 0
    v[S + 5, 1] = np.inf                         # sequence 1: huge values and tiny ones
    v[S + 9, hd - 1] = 3.4028e38
    if KVH > 1:
        v[:, hd:2 * hd] *= np.float32(1e-37)     # key head 1: pieces would keep 8 bits of it
        k[:, hd:2 * hd] *= np.float32(1e-36)
        q[:, (H // KVH) * hd:2 * (H // KVH) * hd] *= np.float32(1e36)
    out = torch.full((B * S, H * hd), 7.0, device="cuda")
    ctx.attention(dev(torch, q), dev(torch, k), dev(torch, v), out, B, S, H, KVH, hd, 0)
    got, ref = host(out), orc.attention(q, k, v, B, S, H, KVH, hd, None)
    # a masked key's infinity or NaN times a zero weight within its key block
    # is NaN here and skipped in the loop: rows from those keys on, and before
    # their blocks (sequence 1's keys 5 and 9: rows past its first 32)
    pos, seq = np.arange(B * S) % S, np.arange(B * S) // S
    rows = (seq >= 2) | ((seq == 0) & (pos >= S // 2)) | ((seq == 1) & (pos >= 32))
    assert np.array_equal(np.isnan(got[rows]), np.isnan(ref[rows]))
    assert np.array_equal(np.isfinite(got[rows]), np.isfinite(ref[rows]))
    # each output to the weighted magnitudes of its own values: a score of up to
    # 128 products, some 8 in magnitude, moves its weight by 1e-5, the sums less
    with np.errstate(all="ignore"):
        mag = orc.attention(q, k, np.abs(v), B, S, H, KVH, hd, None)[rows].astype(np.float64)
        diff = np.abs(got[rows].astype(np.float64) - ref[rows])
    ok = np.isfinite(ref[rows])
    assert np.all(diff[ok] <= 2e-5 * mag[ok] + 1e-44)
    huge = ok[:, hd - 1] & (seq[rows] == 1)     # 3.4e38 under a weight: a finite output
    assert huge.any() and np.max(np.abs(got[rows][huge, hd - 1])) > 1e30


@pytest.mark.parametrize("B,S,H,KVH,hd,gap", [
    (1, 70, 2, 1, 64, 122), (8, 385, 32, 4, 64, 118), (4, 385, 32, 4, 128, 124),
    (2, 70, 2, 1, 128, 120)])
def test_attention_small_weights_keep_their_bits(ctx, torch, B, S, H, KVH, hd, gap):
    """The first key dominates and its value is zero, so the outputs are the
    other keys' values under weights of about 2^-gap.  The scores are exact here
    (two non-zero columns of few bits).  A weight's exponent, up to 128 and so
    rounded by at most 2^-18, and the logarithm's constant in it, another 2^-18, leave
    a relative error of 2^-17 ln 2 = 5.3e-6; the sums and the quotient some 1e-6."""
    rng = np.random.default_rng(S + hd + gap)
    scale = np.sqrt(hd)
    q = np.zeros((B, S, H, hd), np.float32)
    k = np.zeros((B, S, KVH, hd), np.float32)
    v = rng.uniform(0.5, 1.5, (B, S, KVH, hd)).astype(np.float32)
    q[..., 0], q[..., 1] = 16.0, 1.0
    # the first key's exponent is above the others' by gap, an exact score
    k[:, 0, :, 0] = np.round(gap * scale / 1.4426950408889634 / 16 * 256) / 256
    k[:, 1:, :, 1] = np.round(rng.uniform(-1, 1, (B, S - 1, KVH)) * 256) / 256
    v[:, 0] = 0.0
    out = torch.empty((B * S, H * hd), device="cuda")
    ctx.attention(dev(torch, q.reshape(B * S, -1)), dev(torch, k.reshape(B * S, -1)),
                  dev(torch, v.reshape(B * S, -1)), out, B, S, H, KVH, hd, 0)
    got = host(out).reshape(B, S, H, hd)
    for h in range(H):
        s = np.einsum("bik,bjk->bij", q[:, :, h].astype(np.float64),
                      k[:, :, h // (H // KVH)].astype(np.float64)) / scale
        s = np.where(np.tril(np.ones((S, S), bool)), s, -np.inf)
        w = np.exp(s - s.max(axis=2, keepdims=True))
        ref = (w / w.sum(axis=2, keepdims=True)) @ v[:, :, h // (H // KVH)].astype(np.float64)
        assert np.all(got[:, 0, h] == 0)
        rel = np.abs(got[:, 1:, h] / ref[:, 1:] - 1)
        assert np.max(rel) <= 8e-6, (h, np.max(rel))


def test_attention_after_rope_matches_the_oracle_chain(ctx, torch, orc):
    # the order the decoder runs them in: RoPE on q, k, then attention
    rng = np.random.default_rng(21)
    B, S, H, hd = 2, 64, 4, 32
    q, k, v = (normal(rng, (B * S, H * hd)) for _ in range(3))
    qd, kd = dev(torch, q), dev(torch, k)
    ctx.rope(qd, kd, B, S, H, H, hd)
    out = torch.empty((B * S, H * hd), device="cuda")
    ctx.attention(qd, kd, dev(torch, v), out, B, S, H, H, hd)
    rq, rk = orc.rope(q, k, B, S, H, H, hd)
    assert_close(host(out), orc.attention(rq, rk, v, B, S, H, H, hd), what="rope+attention")


def test_attention_unsupported_and_invalid_shapes(ctx, pkg, torch):
    z = torch.zeros(4096, device="cuda")
    with pytest.raises(pkg.MoeRuntimeError):  # seq_len not a multiple of 16 (head_dim 16)
        ctx.attention(z, z, z, z, 1, 20, 2, 2, 16)
    with pytest.raises(pkg.MoeRuntimeError):  # head_dim not a multiple of 16
        ctx.attention(z, z, z, z, 1, 16, 2, 2, 8)
    with pytest.raises(pkg.MoeInvalidArgument):  # q heads not a multiple of kv heads
        ctx.attention(z, z, z, z, 1, 16, 3, 2, 16)
    with pytest.raises(pkg.MoeInvalidArgument):
        ctx.attention(z, z, z, z, 1, 16, 2, 2, 16, window=-1)
    ctx.attention(z, z, z, z, 0, 16, 2, 2, 16)  # no sequences: nothing to do


# ------------------------------------------------ adds and the embedding
@pytest.mark.parametrize("rows,cols", [(1, 1), (7, 33), (4096, 1024)])
def test_add_and_add_bias_bit_exact(ctx, torch, rows, cols):
    rng = np.random.default_rng(rows + cols)
    a, b = normal(rng, (rows, cols)), normal(rng, (rows, cols))
    bias = normal(rng, (cols,))
    ad = dev(torch, a)
    ctx.add(ad, dev(torch, b))
    assert np.array_equal(host(ad), a + b)
    ctx.add_bias(ad, dev(torch, bias))
    assert np.array_equal(host(ad), (a + b) + bias[None, :])


def test_embed_gathers_rows_and_zeroes_out_of_range_tokens(ctx, torch):
    rng = np.random.default_rng(4)
    vocab, d, n = 1000, 96, 777
    table = normal(rng, (vocab, d))
    tokens = rng.integers(0, vocab, n).astype(np.int32)
    tokens[[3, 10]] = [-1, vocab]
    out = torch.full((n, d), float("nan"), device="cuda")
    ctx.embed(dev(torch, table), dev(torch, tokens), out)
    ref = table[np.clip(tokens, 0, vocab - 1)]
    ref[[3, 10]] = 0.0
    assert np.array_equal(host(out), ref)


# ------------------------------------------------------- the decoder model
def _host_weights(W):
    np_ = lambda t: None if t is None else t.detach().cpu().numpy()
    out = {k: np_(v) for k, v in W.items() if k != "layers"}
    out["layers"] = [{k: np_(v) for k, v in L.items()} for L in W["layers"]]
    return out


def _rows_of(idx_ref, got, batch, seq_len):
    """The oracle's routing rows matching a GPU routing tensor: all rows, or
    the last row of every sequence for the pruned last layer."""
    if got.shape[0] == idx_ref.shape[0]:
        return idx_ref
    return idx_ref[np.arange(1, batch + 1) * seq_len - 1]


def _topk_margin(orc, h, L, cfg):
    """The oracle's gate logits of the MoE input h: the gap between the k-th
    and (k+1)-th largest logit of every row (a near tie flips on 1e-7 noise)."""
    from oracle import decoder as od
    logits = orc.matmul_nt(od.norm(h, L["post_norm_w"], L["post_norm_b"], cfg), L["gate_w"],
                           cfg.contract)
    s = -np.sort(-logits, axis=1)
    k = cfg.top_k
    return (s[:, k - 1] - s[:, k]) if k < s.shape[1] else np.full(len(s), np.inf)


def _per_layer_check(ctx, pkg, torch, orc, model, cfg, Wh, trace, x_last, batch, seq_len):
    """Multi-layer drift: each GPU layer runs on the oracle's input of that
    layer; routing must match except on rows whose oracle top-k margin is
    within float noise, and the output within REL_TOL elsewhere."""
    T = batch * seq_len
    flips = 0
    for li, (x, h, idx_ref) in enumerate(trace):
        y_ref = trace[li + 1][0] if li + 1 < len(trace) else x_last
        y = torch.empty((T, cfg.d), device="cuda")
        idx = torch.empty((T, cfg.top_k), dtype=torch.int32, device="cuda")
        model.layer_forward(li, dev(torch, x), y, batch, seq_len, topk_idx=idx)
        idx = host(idx)
        bad = np.any(idx != idx_ref, axis=1)
        if bad.any():
            margin = _topk_margin(orc, h, Wh["layers"][li], cfg)
            scale = float(np.max(np.abs(h)))
            assert np.all(margin[bad] <= 1e-5 * max(scale, 1.0)), \
                f"layer {li}: routing differs on rows with clear margins"
            flips += int(bad.sum())
        assert_close(host(y)[~bad], y_ref[~bad], what=f"layer {li}")
    return flips


def test_decoder_small_end_to_end_and_per_layer(ctx, pkg, torch, orc):
    from oracle import decoder as od
    cfg = pkg.DecoderConfig(layers=2, d=64, heads=4, kv_heads=2, head_dim=16, experts=4,
                            top_k=2, d_ff=96, vocab=300)
    W = pkg.random_weights(cfg, "cuda", seed=3)
    model = pkg.DecoderModel(ctx, cfg, W)
    B, S = 2, 48
    tokens = np.random.default_rng(2).integers(0, cfg.vocab, (B, S)).astype(np.int32)
    model.reserve(B, S)
    routing = []
    logits = model.generate(dev(torch, tokens), routing=routing)
    Wh = _host_weights(W)
    ref, x_last, trace = od.generate(tokens, Wh, cfg)
    for li, (_, _, idx_ref) in enumerate(trace):
        assert np.array_equal(host(routing[li]), _rows_of(idx_ref, routing[li], B, S)), \
            f"routing of layer {li}"
    assert_close(host(logits), ref, what="logits")
    full = pkg.DecoderModel(ctx, cfg, W, prune_last=False)
    assert_close(host(full.generate(dev(torch, tokens))), ref, what="unpruned logits")
    assert _per_layer_check(ctx, pkg, torch, orc, model, cfg, Wh, trace, x_last, B, S) == 0
    # a second call on the warmed-up buffers gives the same logits bit for bit
    again = model.generate(dev(torch, tokens))
    assert np.array_equal(host(again), host(logits))


def test_decoder_config5_one_sequence(ctx, pkg, torch, orc):
    # config 5's shapes (4 layers, d 1024, 16 heads, 8 SwiGLU experts d_ff
    # 2816 top-2, vocab 32000) on one of its 8 sequences of 512 tokens: the
    # oracle covers every layer in seconds
    from oracle import decoder as od
    print("decoder config 5, 1 x 512", flush=True)
    cfg = pkg.DecoderConfig()
    W = pkg.random_weights(cfg, "cuda", seed=0)
    model = pkg.DecoderModel(ctx, cfg, W)
    B, S = 1, 512
    tokens = np.random.default_rng(5).integers(0, cfg.vocab, (B, S)).astype(np.int32)
    model.reserve(B, S)
    routing = []
    logits = host(model.generate(dev(torch, tokens), routing=routing))
    Wh = _host_weights(W)
    ref, x_last, trace = od.generate(tokens, Wh, cfg)
    flips = _per_layer_check(ctx, pkg, torch, orc, model, cfg, Wh, trace, x_last, B, S)
    e2e = sum(int(np.any(host(r) != _rows_of(t[2], r, B, S), axis=1).sum())
              for r, t in zip(routing, trace))
    print(f"per-layer flips {flips}, end-to-end routing rows differing {e2e}", flush=True)
    # with N(0, 0.02) weights no top-k margin of this input lies within float
    # noise: the routing of every layer must match end to end, and the logits
    assert e2e == 0, f"end-to-end routing differs on {e2e} rows"
    assert_close(logits, ref, what="logits")


def test_decoder_config5_batch_of_8(ctx, pkg, torch, orc):
    """Config 5's whole batch (8 x 512 tokens) on the GPU; the oracle runs two
    whole sequences, the first and the last (attention is per sequence and
    causal, so they are exact rows of the batched prefill): routing of every
    layer bit-exact on their rows, their logits within 1e-4."""
    from oracle import decoder as od
    print("decoder config 5, 8 x 512 (oracle on sequences 0 and 7)", flush=True)
    cfg = pkg.DecoderConfig()
    W = pkg.random_weights(cfg, "cuda", seed=1)
    model = pkg.DecoderModel(ctx, cfg, W)
    B, S = 8, 512
    tokens = np.random.default_rng(8).integers(0, cfg.vocab, (B, S)).astype(np.int32)
    model.reserve(B, S)
    routing = []
    logits = host(model.generate(dev(torch, tokens), routing=routing))
    seqs = [0, B - 1]
    ref, _, trace = od.generate(tokens[seqs], _host_weights(W), cfg)
    rows = np.concatenate([np.arange(b * S, (b + 1) * S) for b in seqs])
    for li, (r, t) in enumerate(zip(routing, trace)):
        got = host(r)
        if got.shape[0] == B * S:
            got, want = got[rows], t[2]
        else:  # the pruned last layer: the last row of every sequence
            got, want = got[seqs], t[2][np.arange(1, len(seqs) + 1) * S - 1]
        assert np.array_equal(got, want), f"routing of layer {li}"
    assert_close(logits[seqs], ref, what="logits of sequences 0 and 7")


def test_captured_prefill_replays_match_eager(ctx, pkg, torch):
    # several replays with eager work and synchronisations between them,
    # each against the eager result; new tokens written in place between
    cfg = pkg.DecoderConfig(layers=2, d=64, heads=4, kv_heads=4, head_dim=16, experts=4,
                            top_k=2, d_ff=96, vocab=300)
    W = pkg.random_weights(cfg, "cuda", seed=8)
    model = pkg.DecoderModel(ctx, cfg, W)
    B, S = 2, 32
    rng = np.random.default_rng(9)
    toks = [dev(torch, rng.integers(0, cfg.vocab, (B, S)).astype(np.int32)) for _ in range(3)]
    eager = [host(model.generate(t)) for t in toks]
    from moe_amd.decoder import CapturedPrefill
    cap = CapturedPrefill(model, B, S)
    try:
        for rep in range(6):
            i = rep % 3
            got = host(cap.replay(toks[i]))
            assert np.array_equal(got, eager[i]), f"replay {rep}"
            # eager work on the shared model's context between replays
            other = host(model.generate(toks[(i + 1) % 3]))
            assert np.array_equal(other, eager[(i + 1) % 3])
            torch.cuda.synchronize()
    finally:
        cap.close()


# the last case's row (8200 scores) is past the LDS row limit: scores in HBM
@pytest.mark.parametrize("B,S,H,KVH,hd,window", [(1, 1, 1, 1, 1, None), (2, 37, 4, 2, 6, None),
                                                 (3, 300, 4, 1, 64, 100),
                                                 (8, 512, 16, 16, 64, None),
                                                 (1, 8200, 1, 1, 16, None)])
def test_attention_last_bit_exact(ctx, torch, orc, B, S, H, KVH, hd, window):
    # the last position of every sequence against the oracle's full attention
    print(f"attention_last B={B} S={S} H={H} KVH={KVH} hd={hd} window={window}", flush=True)
    rng = np.random.default_rng(B + S + H + hd)
    q = normal(rng, (B * S, H * hd))
    k, v = normal(rng, (B * S, KVH * hd)), normal(rng, (B * S, KVH * hd))
    last = np.arange(1, B + 1) * S - 1
    out = torch.full((B, H * hd), float("nan"), device="cuda")
    ctx.attention_last(dev(torch, q[last]), dev(torch, k), dev(torch, v), out, B, S, H, KVH, hd,
                       window or 0)
    ref = orc.attention(q, k, v, B, S, H, KVH, hd, window)[last]
    assert np.array_equal(host(out), ref)


def test_rope_first_pos_rotates_rows_at_their_position(ctx, pkg, torch, orc):
    rng = np.random.default_rng(12)
    B, S, H, hd = 3, 20, 2, 8
    q = normal(rng, (B * S, H * hd))
    last = np.arange(1, B + 1) * S - 1
    ql = dev(torch, q[last])
    ctx.rope(ql, None, B, 1, H, 0, hd, first_pos=S - 1, table=ctx.rope_table(1e4, hd, S))
    rq, _ = orc.rope(q, q.copy(), B, S, H, H, hd)
    assert np.array_equal(host(ql), rq[last])
    with pytest.raises(pkg.MoeInvalidArgument):  # the table has no position S
        ctx.rope(ql, None, B, 1, H, 0, hd, first_pos=S, table=ctx.rope_table(1e4, hd, S))


# ------------------------------------------- prefix-trie rows (key lists)
def _trie(seqs):
    """One node per distinct prefix, in order of first appearance, as the
    reference builds it (src/model.cu:1624-1680): node tokens, depths,
    root paths flattened (CSR), the last node of every sequence."""
    child, tok, depth, parent, last = {}, [], [], [], []
    for seq in seqs:
        p = -1
        for pos, t in enumerate(seq):
            key = (p, int(t))
            if key not in child:
                child[key] = len(tok)
                tok.append(int(t))
                depth.append(pos)
                parent.append(p)
            p = child[key]
        last.append(p)
    off, anc = [0], []
    for n in range(len(tok)):
        path = (anc[off[parent[n]]:off[parent[n] + 1]] if parent[n] >= 0 else []) + [n]
        anc += path
        off.append(len(anc))
    return (np.array(tok, np.int32), np.array(depth, np.int32), np.array(anc, np.int32),
            np.array(off, np.int32), np.array(last, np.int32))


def test_rope_rows_at_explicit_positions(ctx, torch, orc):
    rng = np.random.default_rng(31)
    rows, H, KVH, hd = 50, 3, 1, 16
    pos = rng.integers(0, 200, rows).astype(np.int32)
    q, k = normal(rng, (rows, H * hd)), normal(rng, (rows, KVH * hd))
    qd, kd = dev(torch, q), dev(torch, k)
    ctx.rope_rows(qd, kd, ctx.rope_table(1e4, hd, 200), dev(torch, pos), rows, H, KVH, hd)
    # the oracle with a table whose row r is the position of row r
    t = orc.rope_table(1e4, hd, 200)[pos]
    rq, rk = orc.rope(q, k, 1, rows, H, KVH, hd, table=t)
    assert np.array_equal(host(qd), rq) and np.array_equal(host(kd), rk)


@pytest.mark.parametrize("window", [None, 4])
@pytest.mark.parametrize("H,KVH,hd", [(4, 2, 32), (16, 4, 128), (2, 2, 64)])
def test_attention_paths_over_a_trie_bit_exact(ctx, torch, orc, window, H, KVH, hd):
    # sequences with shared prefixes (and one that is a prefix of another):
    # every node's result equals the oracle's attention over its sequence;
    # (16, 4, 128) is Phi-tiny-MoE's head layout, (2, 2, 64) another
    # compile-time head_dim
    rng = np.random.default_rng(32)
    base = rng.integers(0, 50, 30)
    seqs = [base[:30], base[:12], np.concatenate([base[:12], [7, 8, 9]]), base[:5],
            rng.integers(0, 50, 21), np.concatenate([base[:20], rng.integers(0, 50, 9)])]
    tok, depth, anc, off, last = _trie(seqs)
    n = len(tok)
    assert n < sum(len(s) for s in seqs)  # prefixes are shared
    q = normal(rng, (n, H * hd))
    k, v = normal(rng, (n, KVH * hd)), normal(rng, (n, KVH * hd))
    out = torch.full((n, H * hd), float("nan"), device="cuda")
    offd = dev(torch, off)
    ctx.attention_paths(dev(torch, q), dev(torch, k), dev(torch, v), out, dev(torch, anc),
                        offd[:-1], offd[1:], int(np.max(np.diff(off))), H, KVH, hd,
                        window or 0)
    got = host(out)
    for b, seq in enumerate(seqs):
        path = anc[off[last[b]]:off[last[b] + 1]]  # the sequence's nodes, by position
        ref = orc.attention(q[path], k[path], v[path], 1, len(seq), H, KVH, hd, window)
        assert np.array_equal(got[path], ref), f"sequence {b}"
    # the last rows alone (the pruned layer's queries), key lists by begin/end
    beg, end = off[last], off[last + 1]
    out_l = torch.empty((len(seqs), H * hd), device="cuda")
    ctx.attention_paths(dev(torch, q[last]), dev(torch, k), dev(torch, v), out_l,
                        dev(torch, anc), dev(torch, beg), dev(torch, end),
                        int(np.max(end - beg)), H, KVH, hd, window or 0)
    assert np.array_equal(host(out_l), got[last])


def test_attention_paths_refuses_lists_past_its_bounds(ctx, torch):
    # a list longer than the stated max_len, or past key_rows: NaN rows, no
    # access outside the buffers
    H, hd = 2, 16
    q = torch.ones((2, H * hd), device="cuda")
    kv = torch.ones((40, H * hd), device="cuda")
    rows = torch.arange(40, dtype=torch.int32, device="cuda")
    beg = torch.tensor([0, 5], dtype=torch.int32, device="cuda")  # disjoint lists
    end = torch.tensor([5, 40], dtype=torch.int32, device="cuda")
    out = torch.zeros((2, H * hd), device="cuda")
    ctx.attention_paths(q, kv, kv, out, rows, beg, end, 8200, H, H, hd)  # global-score path
    got = host(out)
    assert np.all(np.isfinite(got))
    end2 = torch.tensor([5, 41], dtype=torch.int32, device="cuda")  # past key_rows
    ctx.attention_paths(q, kv, kv, out, rows, beg, end2, 64, H, H, hd)
    got = host(out)
    assert np.all(np.isfinite(got[0])) and np.all(np.isnan(got[1]))
