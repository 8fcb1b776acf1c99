"""Multi-token prefill: the TL1 contraction on int8 MFMA against the
per-token GEMV and the CPU oracle (the int32 accumulators are exact, so the
batched results equal the sequential per-token ones bit for bit: fp32 outputs
are one multiply of them), and the engine's batched prefill against one
prefill_token call per token (KV cache, hidden state and the following
decode steps bit for bit: every stage runs the same arithmetic)."""
import numpy as np
import pytest

import oracle
from tenzo_amd import formats

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available(), "GPU test needs a visible GPU"
    from tenzo_amd import _lib
    _lib.load()
    return torch


def to_dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _setup(torch, N, K, M, seed):
    from tenzo_amd import ops
    rng = np.random.default_rng(seed)
    w = formats.tl1_random(N, K, rng)
    x = (rng.standard_normal((M, K)) * rng.uniform(0.1, 10, (M, 1))).astype(np.float32)
    wp = ops.tl1_repack(to_dev(torch, w), N, K)
    codes, q, _ = ops.rmsnorm_quant31(to_dev(torch, x), None)
    return w, x, wp, codes, q


@pytest.mark.parametrize("N,K", [(64, 64), (128, 130), (192, 1000), (3840, 2560),
                                 (2560, 6912), (13824, 2560)])
@pytest.mark.parametrize("M", [1, 7, 16, 33, 64, 100])
def test_batch_equals_per_token_gemv(torch_dev, N, K, M):
    from tenzo_amd import ops
    torch = torch_dev
    print(f"tl1_batch N={N} K={K} M={M}", flush=True)
    w, x, wp, codes, q = _setup(torch, N, K, M, N + 3 * K + 7 * M)
    yb, ab = ops.bitlinear_tl1_batch(codes, q, wp, 0.0173, N, K, want_acc=True)
    yg, ag = ops.bitlinear_tl1(codes, q, wp, 0.0173, N, K, want_acc=True)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(ab.cpu().numpy(), ag.cpu().numpy())
    np.testing.assert_array_equal(yb.cpu().numpy().view(np.uint32),
                                  yg.cpu().numpy().view(np.uint32))
    # the first and last token against the oracle, from the CPU quantization
    for m in sorted({0, M - 1}):
        yo, acco, _ = oracle.tl1_gemv(x[m], w, N, 0.0173)
        np.testing.assert_array_equal(ab[m].cpu().numpy(), acco)
        np.testing.assert_array_equal(yb[m].cpu().numpy(), yo)


@pytest.mark.parametrize("M,N,K", [
    (33, 4194368, 130),                                    # N above 2^22: tl1_mfma_kernel
    (5, 64, 64), (31, 320, 130), (64, 320, 1030),          # 64 x 32 tiles, four K groups
    (600, 1088, 200), (97, 8256, 64), (545, 1920, 320),    # 128 x 32, two K groups
    (1999, 1088, 130), (1030, 2112, 70), (260, 13824, 64),  # 128 x 64
    (3400, 1344, 70), (1285, 3840, 2500), (500, 13824, 190)])  # 256 x 128
def test_batch_shapes_against_whole_sums(torch_dev, M, N, K):
    """Every shape that the plan picks, with ragged tokens, rows that end inside a
    tile and odd and even counts of 64-column chunks, against the whole-number sums
    in float64 (exact: |sum| < 2^53) and the one fp32 product of each."""
    from tenzo_amd import ops
    torch = torch_dev
    print(f"tl1_batch shapes M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N + K)
    w = torch.randint(-1, 2, (N, K), dtype=torch.int8, device="cuda", generator=g)
    u = (w + 1).to(torch.uint8).reshape(N // 64, 2, 32, K // 2, 2)
    nib = u[..., 0] | (u[..., 1] << 2)
    packed = (nib[:, 0] | (nib[:, 1] << 4)).transpose(1, 2).contiguous().reshape(-1)
    wp = ops.tl1_repack(packed, N, K)
    codes, q, _ = ops.rmsnorm_quant31(torch.randn((M, K), device="cuda", generator=g))
    yb, ab = ops.bitlinear_tl1_batch(codes, q, wp, 0.0173, N, K, want_acc=True)
    del u, nib, packed
    acc = codes[:, :K].double() @ w.double().T
    assert torch.equal(ab.double(), acc)
    scale = ops.actq_inv_scale(q) * torch.tensor(0.0173, device="cuda")
    assert torch.equal(yb, acc.float() * scale[:, None])


@pytest.mark.parametrize("tile", [142, 242, 442, 222, 422, 221, 421, 412, 411, 811])
def test_batch_every_tile_shape(torch_dev, tile):
    """Every workgroup tile shape gives the same exact sums, with a ragged
    token count and a K that is not a multiple of the chunk (64) or of the
    K groups' runs."""
    from tenzo_amd import ops
    torch = torch_dev
    N, K, M = 1280, 2600, 70
    print(f"tl1_batch tile={tile}", flush=True)
    w, x, wp, codes, q = _setup(torch, N, K, M, 11)
    ref, _ = ops.bitlinear_tl1(codes, q, wp, 0.5, N, K)
    for _ in range(2):
        yb, _ = ops.bitlinear_tl1_batch(codes, q, wp, 0.5, N, K, tile=tile)
        np.testing.assert_array_equal(yb.cpu().numpy(), ref.cpu().numpy())


def test_batch_prompt_sized(torch_dev):
    """A 512-token prompt at the largest projection: every row against the
    per-token GEMV, a sample against the oracle's integer contraction."""
    from tenzo_amd import ops
    torch = torch_dev
    N, K, M = 13824, 2560, 512
    w, x, wp, codes, q = _setup(torch, N, K, M, 5)
    yb, ab = ops.bitlinear_tl1_batch(codes, q, wp, 1.0, N, K, want_acc=True)
    _, ag = ops.bitlinear_tl1(codes, q, wp, 1.0, N, K, want_acc=True)
    assert torch.equal(ab, ag)
    c = codes.cpu().numpy()
    for m in (0, 255, 511):
        acc = oracle.tl1_gemv_i32(w, c[m, :K], N, K)
        np.testing.assert_array_equal(ab[m].cpu().numpy(), acc)


def test_batch_zero_and_extreme_codes(torch_dev):
    """All-zero rows (absmax floor) and rows at the code range limits."""
    from tenzo_amd import ops
    torch = torch_dev
    N, K, M = 256, 640, 20
    rng = np.random.default_rng(2)
    w = formats.tl1_random(N, K, rng)
    x = np.zeros((M, K), np.float32)
    x[1] = 1e30
    x[2] = -3.0
    x[3, ::2] = 7.0
    x[3, 1::2] = -7.0
    x[4:] = rng.standard_normal((M - 4, K))
    wp = ops.tl1_repack(to_dev(torch, w), N, K)
    codes, q, _ = ops.rmsnorm_quant31(to_dev(torch, x), None)
    yb, ab = ops.bitlinear_tl1_batch(codes, q, wp, 0.25, N, K, want_acc=True)
    for m in range(M):
        yo, acco, _ = oracle.tl1_gemv(x[m], w, N, 0.25)
        np.testing.assert_array_equal(ab[m].cpu().numpy(), acco)
        np.testing.assert_array_equal(yb[m].cpu().numpy(), yo)


def _engine_pair(eng_mod, cfg, sm):
    a, b = eng_mod.Engine(cfg), eng_mod.Engine(cfg)
    for e in (a, b):
        e.set_model(sm)
        e.set_mode("eager")
    return a, b


@pytest.mark.parametrize("ctx,n", [(0, 1), (0, 5), (0, 40), (5, 23), (17, 30)])
def test_engine_prefill_equals_token_by_token(torch_dev, ctx, n):
    """exact=True: one pass of the batched pipeline equals n prefill_token
    calls of the per-stage (eager) path bit for bit."""
    from tenzo_amd import engine as eng_mod, synth
    cfg = synth.DecodeConfig(hidden=512, n_q_heads=4, n_kv_heads=1, n_layers=3, ffn=1024,
                             vocab=2048, max_seq=64, theta=10000.0)
    sm = synth.make_model(cfg, seed=61 + n, ctx=ctx)
    rng = np.random.default_rng(n)
    toks = rng.integers(0, cfg.vocab, n).astype(np.int32)
    print(f"engine prefill ctx={ctx} n={n}", flush=True)
    a, b = _engine_pair(eng_mod, cfg, sm)
    with a, b:
        for t in toks:
            a.prefill(int(t))
        b.prefill_batch(toks, exact=True)
        assert a.seq_len == b.seq_len == ctx + n
        for x, y in zip(a.get_kv(ctx + n), b.get_kv(ctx + n)):
            np.testing.assert_array_equal(x, y)
        np.testing.assert_array_equal(a.buffer("x"), b.buffer("x"))
        for t in (7, 11, 13):
            assert a.step(t) == b.step(t)
            np.testing.assert_array_equal(a.logits(), b.logits())


@pytest.mark.parametrize("n,F", [(20, 6912), (100, 6912), (140, 6912), (600, 4160)])
def test_engine_prefill_gate_up_shapes(torch_dev, n, F):
    """The gate | up product with the activation in its epilogue, in each of its
    shapes (20: 128 x 32 tiles, 100: 128 x 64 with two K groups, 140: 128 x 64,
    600: 256 x 128, whose last tile is half empty at 65 row blocks): bit for bit
    the per-token path's gate, up and activation."""
    from tenzo_amd import engine as eng_mod, synth
    cfg = synth.DecodeConfig(hidden=512, n_q_heads=4, n_kv_heads=1, n_layers=1, ffn=F,
                             vocab=512, max_seq=640, theta=10000.0)
    sm = synth.make_model(cfg, seed=n, ctx=0)
    toks = np.random.default_rng(n).integers(0, cfg.vocab, n).astype(np.int32)
    print(f"engine prefill gate|up n={n} F={F}", flush=True)
    a, b = _engine_pair(eng_mod, cfg, sm)
    with a, b:
        rows = []
        for t in toks:
            a.prefill(int(t))
            rows.append(a.buffer("x"))
        b.prefill_batch(toks, exact=True)
        np.testing.assert_array_equal(rows[-1], b.buffer("x"))
        for i in (n // 3, n // 2):  # other tokens' rows, as the last of a shorter prompt
            b.reset()
            b.prefill_batch(toks[:i], exact=True)
            np.testing.assert_array_equal(rows[i - 1], b.buffer("x"))


def test_engine_prefill_passes(torch_dev):
    """2100 tokens in two passes (2048 + 52 rows) equal the same tokens as two
    prompts of 300 (small buffers) and 1800 rows (buffers grown)."""
    from tenzo_amd import engine as eng_mod, synth
    cfg = synth.DecodeConfig(hidden=512, n_q_heads=4, n_kv_heads=1, n_layers=2, ffn=512,
                             vocab=1024, max_seq=2200, theta=10000.0)
    sm = synth.make_model(cfg, seed=72, ctx=0)
    toks = np.random.default_rng(4).integers(0, cfg.vocab, 2100).astype(np.int32)
    a, b = _engine_pair(eng_mod, cfg, sm)
    with a, b:
        a.prefill_batch(toks, exact=True)
        b.prefill_batch(toks[:300], exact=True)
        b.prefill_batch(toks[300:], exact=True)
        for x, y in zip(a.get_kv(2100), b.get_kv(2100)):
            np.testing.assert_array_equal(x, y)
        np.testing.assert_array_equal(a.buffer("x"), b.buffer("x"))


def test_engine_prefill_longer_than_one_pass(torch_dev):
    """600 tokens: more than one step of 512 buffer rows, attention over up to 19
    chunks per query, G = 4 query heads per kv head."""
    from tenzo_amd import engine as eng_mod, synth
    cfg = synth.DecodeConfig(hidden=512, n_q_heads=4, n_kv_heads=1, n_layers=2, ffn=512,
                             vocab=1024, max_seq=640, theta=10000.0)
    sm = synth.make_model(cfg, seed=71, ctx=0)
    toks = np.random.default_rng(3).integers(0, cfg.vocab, 600).astype(np.int32)
    a, b = _engine_pair(eng_mod, cfg, sm)
    with a, b:
        for t in toks:
            a.prefill(int(t))
        b.prefill_batch(toks, exact=True)
        for x, y in zip(a.get_kv(600), b.get_kv(600)):
            np.testing.assert_array_equal(x, y)
        np.testing.assert_array_equal(a.buffer("x"), b.buffer("x"))
        assert a.step(5) == b.step(5)
        np.testing.assert_array_equal(a.logits(), b.logits())


def test_engine_prefill_chunk_size_changes(torch_dev):
    """16 kv heads: decode aims at 512 / 16 = 32 chunks per head, so its chunk
    size is 32 tokens up to a context of 1024 and 64 past it (ceil(ctx / 32)
    rounded up to a multiple of 32); a prompt from position 1000 mixes both
    in one launch (rows with 32-token chunks run in the kernel built for 64),
    G = 1."""
    from tenzo_amd import engine as eng_mod, synth
    cfg = synth.DecodeConfig(hidden=2048, n_q_heads=16, n_kv_heads=16, n_layers=1, ffn=512,
                             vocab=512, max_seq=1100, theta=10000.0)
    sm = synth.make_model(cfg, seed=29, ctx=1000)
    toks = np.random.default_rng(4).integers(0, cfg.vocab, 60).astype(np.int32)
    print("engine prefill ctx=1000 n=60 Hkv=16", flush=True)
    a, b = _engine_pair(eng_mod, cfg, sm)
    with a, b:
        for t in toks:
            a.prefill(int(t))
        b.prefill_batch(toks, exact=True)
        for x, y in zip(a.get_kv(1060), b.get_kv(1060)):
            np.testing.assert_array_equal(x, y)
        np.testing.assert_array_equal(a.buffer("x"), b.buffer("x"))
        assert a.step(9) == b.step(9)
        np.testing.assert_array_equal(a.logits(), b.logits())


@pytest.mark.parametrize("ctx", [2020, 3180])
def test_engine_prefill_wide_merge(torch_dev, ctx):
    """One kv head: decode aims at 512 chunks per head, so its chunks stay 32
    tokens long; past a chunk count the merge moves to the four-group kernel
    (attn_combine_wide_kernel). A prompt of 60 tokens from position 2020 (64 ->
    65 chunks) puts rows on both sides of that line in one launch, one from
    3180 (100 -> 102) only past it; the exact prefill must still equal
    token-by-token decode bit for bit."""
    from tenzo_amd import engine as eng_mod, synth
    cfg = synth.DecodeConfig(hidden=512, n_q_heads=4, n_kv_heads=1, n_layers=1, ffn=512,
                             vocab=512, max_seq=3300, theta=10000.0)
    sm = synth.make_model(cfg, seed=37, ctx=ctx)
    toks = np.random.default_rng(6).integers(0, cfg.vocab, 60).astype(np.int32)
    print(f"engine prefill ctx={ctx} n=60 Hkv=1", flush=True)
    a, b = _engine_pair(eng_mod, cfg, sm)
    with a, b:
        for t in toks:
            a.prefill(int(t))
        b.prefill_batch(toks, exact=True)
        for x, y in zip(a.get_kv(ctx + 60), b.get_kv(ctx + 60)):
            np.testing.assert_array_equal(x, y)
        np.testing.assert_array_equal(a.buffer("x"), b.buffer("x"))
        assert a.step(9) == b.step(9)
        np.testing.assert_array_equal(a.logits(), b.logits())


def test_engine_prefill_then_persistent_decode(torch_dev):
    """A batched prefill followed by persistent-kernel decode steps gives the
    tokens of token-by-token prefill + decode (fp32 logits to 1e-5: the
    persistent kernel sums attention in its own order)."""
    from tenzo_amd import engine as eng_mod, synth
    cfg = synth.DecodeConfig(hidden=512, n_q_heads=4, n_kv_heads=1, n_layers=3, ffn=1024,
                             vocab=2048, max_seq=64, theta=10000.0)
    sm = synth.make_model(cfg, seed=83, ctx=0)
    toks = np.arange(1, 20, dtype=np.int32) * 37 % cfg.vocab
    with eng_mod.Engine(cfg) as a, eng_mod.Engine(cfg) as b:
        a.set_model(sm)
        b.set_model(sm)
        for t in toks:
            a.prefill(int(t))
        b.prefill_batch(toks, exact=True)
        ta, tb = a.decode(3, 6)[0], b.decode(3, 6)[0]
        assert list(ta) == list(tb)
        la, lb = a.logits(), b.logits()
        assert np.abs(la - lb).max() <= 1e-5 * max(np.abs(la).max(), 1e-30)


def test_engine_prefill_errors(torch_dev):
    from tenzo_amd import engine as eng_mod, synth
    cfg = synth.DecodeConfig(hidden=512, n_q_heads=4, n_kv_heads=1, n_layers=1, ffn=512,
                             vocab=256, max_seq=16, theta=10000.0)
    sm = synth.make_model(cfg, seed=5, ctx=0)
    with eng_mod.Engine(cfg) as e:
        e.set_model(sm)
        with pytest.raises(RuntimeError, match="outside"):
            e.prefill_batch(np.array([1, 256], np.int32))
        with pytest.raises(RuntimeError, match="full"):
            e.prefill_batch(np.zeros(17, np.int32))
        assert e.seq_len == 0
        assert not e.prefill_rows("prefill_attn", 3).any()  # (no pass yet: nothing is copied)
        e.prefill_batch(np.zeros(16, np.int32))
        assert e.seq_len == 16


@pytest.mark.parametrize("ctx,n,G", [(0, 40, 4), (17, 47, 4), (0, 600, 4), (3, 130, 1),
                                     (0, 70, 2)])
def test_engine_prefill_streaming_attention(torch_dev, ctx, n, G):
    """The default (streaming attention) prefill against the exact one: the
    attention differs only in how the softmax sums are grouped, so the hidden
    state agrees to 1e-4 and almost every KV code is identical (a code can flip
    where a value sits on a rounding boundary). The next decode step (on the
    persistent kernel, whose per-layer int32 sums are read back) attends over
    those caches: when every layer's activation codes are the same in both
    engines (every TL1 sum equal) the new hidden states agree to 1e-4; a +-31
    code can flip at a rounding tie, which moves them by ~1e-3, and only then
    -- exactly one GEMV whose sums differ, each by at most one weight (a
    single code moved by one) -- are they held to 1e-2. Each engine's logits
    must equal, bit for bit, the oracle's LM head applied to its own hidden
    state (the head's +-127 codes may flip at ties between the two engines,
    but never between an engine and the oracle). The greedy token must agree."""
    from tenzo_amd import engine as eng_mod, synth
    cfg = synth.DecodeConfig(hidden=512, n_q_heads=4, n_kv_heads=4 // G, n_layers=2, ffn=512,
                             vocab=1024, max_seq=ctx + n + 8, theta=10000.0)
    sm = synth.make_model(cfg, seed=97 + n, ctx=ctx)
    toks = np.random.default_rng(n).integers(0, cfg.vocab, n).astype(np.int32)
    print(f"streaming prefill ctx={ctx} n={n} G={G}", flush=True)
    a, b = _engine_pair(eng_mod, cfg, sm)
    with a, b:
        a.prefill_batch(toks, exact=True)
        b.prefill_batch(toks)
        xa, xb = a.buffer("x"), b.buffer("x")
        assert rel(xb, xa) < 1e-4
        for u, v in zip(a.get_kv(ctx + n), b.get_kv(ctx + n)):
            u, v = np.asarray(u, np.float64), np.asarray(v, np.float64)
            assert (u != v).mean() < 0.01
        a.set_mode("persistent")
        b.set_mode("persistent")
        ta, tb = a.step(5), b.step(5)
        la, lb = a.logits(), b.logits()
        moved = []
        for l in range(cfg.n_layers):
            for name in ("acc_qkv", "acc_o", "acc_gu", "acc_down"):
                d = a.layer_state(l, name).astype(np.int64) - b.layer_state(l, name)
                if d.any():
                    moved.append((l, name, int(np.abs(d).max())))
        # the head is exact given its input: each engine's logits equal the
        # oracle's LM head (bit-exact rms_norm, +-127 codes, int8 rows) applied
        # to that engine's own final hidden state
        xa2, xb2 = a.buffer("x"), b.buffer("x")
        for x, lg in ((xa2, la), (xb2, lb)):
            ref_lg = oracle.lm_head(oracle.rms_norm(x, sm.final_norm), sm.embed,
                                    sm.embed_scales)[0]
            np.testing.assert_array_equal(lg, ref_lg)
        print(f"GEMVs whose sums differ: {moved}; hidden rel {rel(xb2, xa2):.2e}", flush=True)
        if not moved:
            assert rel(xb2, xa2) < 1e-4
        else:
            assert len(moved) == 1 and moved[0][2] == 1, moved
            assert rel(xb2, xa2) < 1e-2
        assert ta == tb


@pytest.mark.parametrize("ctx,n,Hq,Hkv", [(200, 60, 4, 4), (0, 256, 4, 2), (250, 77, 4, 1),
                                          (255, 1, 4, 1), (0, 300, 8, 1), (0, 2100, 16, 4),
                                          (31, 2200, 16, 16), (455, 60, 4, 4), (256, 256, 4, 2),
                                          (450, 77, 4, 1), (767, 1, 4, 1), (0, 600, 8, 1)])
def test_engine_prefill_streaming_64_rows(torch_dev, ctx, n, Hq, Hkv):
    """The streaming attention at and around the prefixes from which the 64-row kernel takes
    over (512 keys; 768 for fewer than 16 rows a kv head, as the row of (767, 1); 384 and 256 where
    the rows are many, as in the two prompts of over 2000 tokens, which have two key groups to a
    workgroup, the others four) against the exact form, for every count of heads per kv head, ragged ends of rows and of key tiles, and rows whose
    prefix ends inside the first tiles. Each token's second-layer K and V codes come
    from its own first-layer attention: rounded codes may flip on a tie (a flip moves a
    few of a row's codes by one), a row with a key too many or too few differs
    throughout."""
    from tenzo_amd import engine as eng_mod, synth
    cfg = synth.DecodeConfig(hidden=128 * Hq, n_q_heads=Hq, n_kv_heads=Hkv, n_layers=2, ffn=512,
                             vocab=512, max_seq=ctx + n + 8, theta=10000.0)
    sm = synth.make_model(cfg, seed=n, ctx=ctx)
    toks = np.random.default_rng(n).integers(0, cfg.vocab, n).astype(np.int32)
    print(f"streaming 64 rows ctx={ctx} n={n} Hq={Hq} Hkv={Hkv}", flush=True)
    a, b = _engine_pair(eng_mod, cfg, sm)
    with a, b:
        a.prefill_batch(toks, exact=True)
        b.prefill_batch(toks)
        ka, va, *_ = a.get_kv(ctx + n)
        kb, vb, *_ = b.get_kv(ctx + n)
        for u, v in ((ka, kb), (va, vb)):
            np.testing.assert_array_equal(u[0], v[0])
            d = np.abs(u[1].astype(np.int32) - v[1])  # [Hkv][token][128]
            print("codes that differ", (d > 0).mean(), "largest share of a row",
                  (d > 0).mean(axis=(0, 2)).max(), flush=True)
            assert (d > 0).mean() < 0.01
            assert np.sqrt((d.astype(np.float64) ** 2).mean(axis=(0, 2))).max() < 4.0


def test_engine_prefill_little_memory(torch_dev):
    """A prompt of 2200 tokens where memory holds the buffers of one step of 512 rows only, and
    scratch for a part of the queries: passes of as many rows as fit, bit for bit the same state,
    and a longer prompt later takes no more either."""
    from tenzo_amd import engine as eng_mod, synth
    torch = torch_dev
    cfg = synth.DecodeConfig(hidden=512, n_q_heads=4, n_kv_heads=1, n_layers=1, ffn=32768,
                             vocab=512, max_seq=2304, theta=10000.0)
    sm = synth.make_model(cfg, seed=3, ctx=0)
    toks = np.random.default_rng(3).integers(0, cfg.vocab, 2200).astype(np.int32)
    a, b = _engine_pair(eng_mod, cfg, sm)
    hold = []
    with a, b:
        a.prefill_batch(toks, exact=True)  # 340 MiB for 2048 rows (512: 85), scratch up to 142
        eng_mod.lib().tenzo_hip_release_scratch()
        torch.cuda.empty_cache()
        try:
            for _ in range(8):
                torch.cuda.synchronize()
                free = torch.cuda.mem_get_info()[0]
                if free < 122 << 20:
                    break
                hold.append(torch.empty(free - (112 << 20), dtype=torch.uint8, device="cuda"))
            print("little memory: bytes left", free, flush=True)
            assert free < 122 << 20
            b.prefill_batch(toks[:600], exact=True)
            b.prefill_batch(toks[600:], exact=True)
        finally:
            hold.clear()
            torch.cuda.empty_cache()
            eng_mod.lib().tenzo_hip_release_scratch()
        for x, y in zip(a.get_kv(2200), b.get_kv(2200)):
            np.testing.assert_array_equal(x, y)
        np.testing.assert_array_equal(a.buffer("x"), b.buffer("x"))


def _one_layer(eng_mod, synth, Hq, Hkv, ctx, n, loud, seed):
    """A one-layer engine and its model. loud: embeddings with a common part, which rows 5 and 69
    of each query head sum up while its other rows take differences of four values; the keys
    hold zeros there."""
    cfg = synth.DecodeConfig(hidden=128 * Hq, n_q_heads=Hq, n_kv_heads=Hkv, n_layers=1, ffn=512,
                             vocab=1024, max_seq=ctx + n + 8, theta=10000.0)
    sm = synth.make_model(cfg, seed=seed, ctx=ctx)
    if loud:
        rng = np.random.default_rng(seed)
        sm.embed[:] = np.clip(np.rint(60 + 18 * rng.standard_normal(sm.embed.shape)), -127, 127)
        lw, H = sm.layers[0], cfg.hidden
        lw.in_norm[:] = 1.0
        wq = np.zeros((Hq * 128, H), np.int8)
        for r in wq:
            r[rng.choice(H, 4, replace=False)] = [1, 1, -1, -1]
        wk = formats.tl1_unpack(lw.tl1["k"], Hkv * 128, H).copy()
        for d in (5, 69):
            wq[d::128], wk[d::128] = 1, 0
        sm.kc[:, :, :, [5, 69]] = 0
        lw.tl1["q"], lw.tl1["k"] = formats.tl1_pack(wq), formats.tl1_pack(wk)
        lw.scale["q"] = np.float32(8.0)
    e = eng_mod.Engine(cfg)
    e.set_model(sm)
    return cfg, e


def _attention64(torch, cfg, qkv, kv, pos0, table):
    """softmax(q k / sqrt(128)) v of the rows' rotated queries (fp32, as the append and decode
    rotate them) over the cached rows in float64: (output, largest |score|)."""
    n, Hq, Hkv = len(qkv), cfg.n_q_heads, cfg.n_kv_heads
    q = qkv[:, :Hq * 128].reshape(n, Hq, 128)
    cs, sn = (t[pos0:pos0 + n, None] for t in (table[:, :64], table[:, 64:]))
    lo, hi = q[..., :64], q[..., 64:]
    d = np.float64
    q = np.concatenate([(lo.astype(d) * cs - (hi * sn).astype(d)).astype(np.float32),
                        (lo.astype(d) * sn + (hi * cs).astype(d)).astype(np.float32)], -1)
    q = torch.from_numpy(q.astype(d)).cuda()
    k, v = (torch.from_numpy(c[0].astype(d) * s[0, :, :, None].astype(d)).cuda()
            for c, s in ((kv[0], kv[2]), (kv[1], kv[3])))
    late = torch.arange(k.shape[1], device="cuda")[None] > pos0 + torch.arange(n, device="cuda")[:, None]
    out, top = torch.empty((n, Hq, 128), dtype=torch.float64, device="cuda"), 0.0
    for h in range(Hq):
        s = (q[:, h] @ k[h * Hkv // Hq].T / 128 ** 0.5).masked_fill(late, -float("inf"))
        top = max(top, s[~late].abs().max().item())
        out[:, h] = torch.softmax(s, -1) @ v[h * Hkv // Hq]
    return out.reshape(n, -1).cpu().numpy(), top


@pytest.mark.parametrize("ctx,n,Hq,Hkv", [(0, 700, 4, 1), (900, 60, 4, 4), (1500, 200, 8, 1),
                                          (0, 2048, 20, 5), (100, 60, 4, 2)])
@pytest.mark.parametrize("loud", [False, True])
def test_engine_prefill_streaming_error(torch_dev, ctx, n, Hq, Hkv, loud):
    """Streaming attention outputs of a pass against float64 (the 64-row kernel with four and two
    key groups, and the 16-row kernel), for ordinary queries and for rows whose largest elements, a
    few hundred times the others, meet zero keys. A query element's hi and lo parts hold 22 bits
    of it, a score of at most 32 is wrong by at most 32 (2^-22 + 2^-21 for its sums), so a
    weight by 2.3e-5 of itself; over hundreds of keys with independent signs that is below
    2e-6 of the output's norm."""
    from tenzo_amd import _lib, engine as eng_mod, synth
    cfg, e = _one_layer(eng_mod, synth, Hq, Hkv, ctx, n, loud, 31 + n)
    toks = np.random.default_rng(n).integers(0, cfg.vocab, n).astype(np.int32)
    table = np.empty((cfg.max_seq, 128), np.float32)
    _lib.load().tenzo_hip_rope_table(10000.0, 128, 0, cfg.max_seq, table.ctypes.data)
    print(f"streaming error ctx={ctx} n={n} Hq={Hq} Hkv={Hkv} loud={loud}", flush=True)
    with e:
        e.prefill_batch(toks)
        qkv, out = e.prefill_rows("prefill_qkv", n), e.prefill_rows("prefill_attn", n)
        ref, top = _attention64(torch_dev, cfg, qkv, e.get_kv(ctx + n), ctx, table)
    q = np.abs(qkv[:, :Hq * 128]).reshape(n, Hq, 128)
    spread = q.max() / np.median(q[q > 0])
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    print(f"error {err:.2e}, largest score {top:.1f}, largest |q| over the median {spread:.0f}", flush=True)
    assert top < 32 and (spread > 200) == loud
    assert err < 2e-6


@pytest.mark.parametrize("scale", [np.nan, np.inf])
@pytest.mark.parametrize("ctx,n,Hq,Hkv", [(0, 40, 4, 1), (900, 30, 4, 2), (0, 2048, 20, 5)])
def test_engine_prefill_streaming_queries_not_finite(torch_dev, ctx, n, Hq, Hkv, scale):
    """Queries of NaN (or of infinities and NaN) over finite keys and values: NaN outputs, as the
    exact form gives, from the 16-row and the 64-row kernel alike."""
    from tenzo_amd import engine as eng_mod, synth
    cfg, e = _one_layer(eng_mod, synth, Hq, Hkv, ctx, n, False, 7)
    sm = synth.make_model(cfg, seed=7, ctx=ctx)
    sm.layers[0].scale["q"] = np.float32(scale)
    e.set_layer(0, sm.layers[0])
    toks = np.random.default_rng(n).integers(0, cfg.vocab, n).astype(np.int32)
    with e:
        for exact in (True, False):
            e.rewind(ctx)
            e.prefill_batch(toks, exact=exact)
            assert np.isfinite(e.prefill_rows("prefill_qkv", n)[:, Hq * 128:]).all()
            assert np.isnan(e.prefill_rows("prefill_attn", n)).all(), exact


@pytest.mark.parametrize("n,Hq,Hkv", [(700, 4, 1), (2048, 20, 5), (1100, 8, 8)])
def test_engine_prefill_streaming_infinite_scale(torch_dev, n, Hq, Hkv):
    """A few tokens' value scales overflow fp16: the rows before such a token, also those of its
    workgroup and those that share a key tile with it, have their ordinary outputs (against float64
    as above), and the rows from it on are not finite, as in the exact form."""
    from tenzo_amd import _lib, engine as eng_mod, synth
    cfg, e = _one_layer(eng_mod, synth, Hq, Hkv, 0, n, False, 9)
    sm = synth.make_model(cfg, seed=9, ctx=0)
    toks = np.random.default_rng(n).permutation(max(n, cfg.vocab))[:n].astype(np.int32) % cfg.vocab
    table = np.empty((cfg.max_seq, 128), np.float32)
    _lib.load().tenzo_hip_rope_table(10000.0, 128, 0, cfg.max_seq, table.ctypes.data)
    with e:
        e.prefill_batch(toks)
        top = np.sort(e.get_kv(n)[3].reshape(-1))[-3]
        sm.layers[0].scale["v"] *= np.float32(66000.0 / top)  # (65520 and more round to infinity)
        e.set_layer(0, sm.layers[0])
        for exact in (True, False):
            e.reset()
            e.prefill_batch(toks, exact=exact)
            out = e.prefill_rows("prefill_attn", n).reshape(n, Hkv, -1)
            kv = e.get_kv(n)
            far = np.isinf(kv[3][0])  # [Hkv][token]
            assert 2 < far.sum() < 32
            first = [int(f.argmax()) if f.any() else n for f in far]
            print(f"n={n} exact={exact} first infinite scales {first}", flush=True)
            kv = kv[:3] + (np.where(np.isinf(kv[3]), 0, kv[3]),)
            ref, _ = _attention64(torch_dev, cfg, e.prefill_rows("prefill_qkv", n), kv, 0, table)
            for h, p in enumerate(first):
                assert not np.isfinite(out[p:, h]).any()
                r = ref.reshape(n, Hkv, -1)[:p, h]
                assert np.linalg.norm(out[:p, h] - r) < 2e-6 * np.linalg.norm(r), (exact, h)


def rel(a, b):
    return np.abs(np.asarray(a, np.float64) - b).max() / max(np.abs(b).max(), 1e-30)
