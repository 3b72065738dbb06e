"""Per-kernel parity of the HIP kernels against the CPU oracle, called through
the C ABI.  Bar (north star): max abs error <= 2e-2 on fp16 activations; the
reference's own cosine bars (tests/test_*.cu) are checked alongside."""

import numpy as np
import pytest

from conftest import cosine_rows, to_dev
from oracle import bert_oracle as O

pytestmark = pytest.mark.gpu

TOL = 2e-2  # max abs error on activations (north star)


def _h(rng, shape, scale=1.0):
    return (rng.standard_normal(shape) * scale).astype(np.float16)


def _np(t):
    return t.float().cpu().numpy()


# ---- Linear ------------------------------------------------------------------

GEMM_SHAPES = [
    # (M, N, K, gelu): the four Linears of the path at small / ragged / large M
    (16, 1152, 384, False), (1000, 1152, 384, False), (48, 384, 384, False),
    (1040, 1536, 384, True),
    (1024, 384, 1536, False), (3072, 1152, 384, False), (8192, 1536, 384, True),
    (4096, 384, 1536, False), (100, 128, 64, False), (7, 64, 128, True),
    # the batch-64 buckets' tiles, ragged: 128x128 for FFN1, 64x128 for FFN2
    (2500, 1536, 384, True), (3000, 384, 1536, False),
    # odd slice counts (3, 1)
    (3000, 384, 192, False), (2100, 384, 64, True),
    # large-M tiles (cfg5 runs M = 131072 end to end), one shape per tile bucket
    (12288, 1152, 384, False), (16384, 384, 1536, False),
    (32768, 1152, 384, False), (32768, 1536, 384, True), (32768, 384, 384, False),
    (32768, 384, 1536, False),
    (40000, 1152, 384, False), (40000, 1536, 384, True), (40000, 384, 1536, False),
    # the weight-resident K = 384 kernel (QKV from M = 49152, FFN1 from 24576), ragged last tile
    (50000, 1152, 384, False),
]


@pytest.mark.parametrize("M,N,K,gelu", GEMM_SHAPES)
def test_linear(torch_cuda, M, N, K, gelu):
    torch = torch_cuda
    from bbh import engine

    rng = np.random.default_rng(M * 7 + N + K)
    A, W, b = _h(rng, (M, K)), _h(rng, (N, K), 1.0 / np.sqrt(K)), _h(rng, (N,), 0.1)
    C = torch.empty((M, N), dtype=torch.float16, device="cuda")
    engine.launch_matmul(to_dev(torch, A), to_dev(torch, W), C, M, N, K, bias=to_dev(torch, b),
                         gelu=gelu)
    want = O.linear(A.astype(np.float32), W.astype(np.float32), b.astype(np.float32), act_gelu=gelu)
    got = _np(C)
    assert np.abs(got - want).max() <= TOL
    assert cosine_rows(got.ravel(), want.ravel()) >= 0.9999


@pytest.mark.parametrize("N,gelu", [(1152, False), (1536, True), (384, False)])
def test_linear_rows_identical_across_kernels(torch_cuda, N, gelu):
    # The first rows of a large-M GEMM equal the same rows computed alone:
    # every kernel accumulates in the same k order and rounds the same way.
    # M = 50000 runs all three on the weight-resident kernel, M = 2048 on 64x64
    # tiles; M = 3000 QKV on a 128x128, FFN1 on a 64x64, N = 384 on a 96x64 tile.
    torch = torch_cuda
    from bbh import engine

    M, K = 50000, 384
    rng = np.random.default_rng(N + 11)
    A, W, b = _h(rng, (M, K)), _h(rng, (N, K), 1.0 / np.sqrt(K)), _h(rng, (N,), 0.1)
    dA, dW, db = to_dev(torch, A), to_dev(torch, W), to_dev(torch, b)
    big = torch.empty((M, N), dtype=torch.float16, device="cuda")
    engine.launch_matmul(dA, dW, big, M, N, K, bias=db, gelu=gelu)
    for m in (2048, 3000):
        small = torch.empty((m, N), dtype=torch.float16, device="cuda")
        engine.launch_matmul(dA[:m], dW, small, m, N, K, bias=db, gelu=gelu)
        torch.cuda.synchronize()
        assert np.array_equal(_np(big[:m]), _np(small)), m


@pytest.mark.parametrize("M", [4096, 32768])
def test_gelu_epilogue_accuracy(torch_cuda, M):
    # The GELU of the FFN1 epilogue against x Phi(x) in float64 over x in
    # [-14, 14]: W is one-hot (W[n, 0] = 1, exact in fp32 accumulation), so
    # column n of row m is GELU(x_m + b_n).  M = 4096 runs a tiled kernel,
    # M = 32768 the weight-resident one.  Bars: the epilogue's own error plus
    # one fp16 rounding step: 1.1e-5 + half a unit in the last place for
    # |x| < 3, 2e-4 + half an ulp everywhere.
    torch = torch_cuda
    from math import erf, sqrt
    from bbh import engine

    N, K = 1536, 384
    x = np.linspace(-14, 14, M).astype(np.float16)
    A = np.zeros((M, K), np.float16)
    A[:, 0] = x
    W = np.zeros((N, K), np.float16)
    W[:, 0] = 1
    b = np.zeros(N, np.float16)
    b[1::2] = 0.25  # half the columns see x + 0.25
    C = torch.empty((M, N), dtype=torch.float16, device="cuda")
    engine.launch_matmul(to_dev(torch, A), to_dev(torch, W), C, M, N, K, bias=to_dev(torch, b),
                         gelu=True)
    got = _np(C).astype(np.float64)
    for col, shift in ((0, 0.0), (1, 0.25)):
        v = x.astype(np.float64) + shift
        want = np.array([0.5 * t * (1 + erf(t / sqrt(2))) for t in v])
        half_ulp = np.abs(want).astype(np.float16).astype(np.float64)
        half_ulp = np.spacing(half_ulp.astype(np.float16)).astype(np.float64) / 2
        err = np.abs(got[:, col] - want)
        small = np.abs(v) < 3
        assert np.all(err[small] <= 1.1e-5 + half_ulp[small] + 1e-12)
        assert np.all(err <= 2e-4 + half_ulp)
    # every column of a row holds the same value as its column of equal bias
    assert np.array_equal(got[:, 0::2], np.repeat(got[:, :1], N // 2, axis=1))


@pytest.mark.parametrize("tag", ["small", "real"])
def test_linear_reference_kat(torch_cuda, kats, tag):
    # tests/test_matmul.cu: 4x16x8 (any-shape kernel) and 128x384x384 (MFMA)
    torch = torch_cuda
    from bbh import engine

    A, B, C = kats[f"matmul_{tag}_A"], kats[f"matmul_{tag}_B"], kats[f"matmul_{tag}_C"]
    M, K = A.shape
    N = B.shape[0]
    out = torch.empty((M, N), dtype=torch.float16, device="cuda")
    engine.launch_matmul(to_dev(torch, A), to_dev(torch, B), out, M, N, K)
    got = _np(out)
    assert cosine_rows(got.ravel(), C.ravel()) >= 0.9995
    assert np.abs(got - C).max() <= TOL


@pytest.mark.parametrize("M,K", [(16, 384), (33, 384), (1024, 1536), (8192, 1536), (3000, 384),
                                 (2100, 1536), (3000, 1536),  # the 64x128 tile, ragged
                                 (12288, 384), (16384, 1536), (32768, 384), (32768, 1536),
                                 (70001, 384)])  # the weight-resident kernel, ragged last tile
def test_linear_residual_layernorm(torch_cuda, M, K):
    torch = torch_cuda
    from bbh import engine

    rng = np.random.default_rng(M + K)
    A, W = _h(rng, (M, K)), _h(rng, (384, K), 1.0 / np.sqrt(K))
    b, r = _h(rng, (384,), 0.1), _h(rng, (M, 384))
    g, be = (1 + rng.standard_normal(384) * 0.1).astype(np.float16), _h(rng, (384,), 0.1)
    y = torch.empty((M, 384), dtype=torch.float16, device="cuda")
    engine.launch_linear_residual_layernorm(to_dev(torch, A), to_dev(torch, W), to_dev(torch, b),
                                            to_dev(torch, r), to_dev(torch, g), to_dev(torch, be),
                                            y, M, K)
    f = lambda a: a.astype(np.float32)  # noqa: E731
    want = O.layer_norm(O.linear(f(A), f(W), f(b)), f(g), f(be), residual=f(r))
    assert np.abs(_np(y) - want).max() <= TOL


@pytest.mark.parametrize("M,K", [(200, 1536), (66000, 384)])
def test_linear_residual_layernorm_in_place(torch_cuda, M, K):
    # y aliasing the residual is how the last layer writes the workspace's
    # final hidden (M = 66000, K = 384: the weight-resident kernel)
    torch = torch_cuda
    from bbh import engine

    rng = np.random.default_rng(3)
    A, W = _h(rng, (M, K)), _h(rng, (384, K), 1.0 / np.sqrt(K))
    b, r = _h(rng, (384,), 0.1), _h(rng, (M, 384))
    g, be = np.ones(384, np.float16), np.zeros(384, np.float16)
    rt = to_dev(torch, r)
    engine.launch_linear_residual_layernorm(to_dev(torch, A), to_dev(torch, W), to_dev(torch, b), rt,
                                            to_dev(torch, g), to_dev(torch, be), rt, M, K)
    f = lambda a: a.astype(np.float32)  # noqa: E731
    want = O.layer_norm(O.linear(f(A), f(W), f(b)), f(g), f(be), residual=f(r))
    assert np.abs(_np(rt) - want).max() <= TOL


def test_linear_residual_layernorm_row_chunks(torch_cuda):
    # M * K * 2 bytes of A above 2^30: the launcher splits the rows into
    # chunks of 349440 (K = 1536), each addressed through its own 32-bit
    # buffer range.  Rows either side of the chunk boundary and the ragged
    # tail match the oracle, and a call over a row window that starts
    # mid-chunk reproduces the same rows bit for bit.
    torch = torch_cuda
    from bbh import engine

    M, K, edge = 360001, 1536, 349440
    g = torch.Generator(device="cuda").manual_seed(11)
    A = torch.randn((M, K), device="cuda", generator=g).half()
    W = (torch.randn((384, K), device="cuda", generator=g) / np.sqrt(K)).half()
    b = (torch.randn(384, device="cuda", generator=g) * 0.1).half()
    r = torch.randn((M, 384), device="cuda", generator=g).half()
    gm = (1 + 0.1 * torch.randn(384, device="cuda", generator=g)).half()
    be = (0.1 * torch.randn(384, device="cuda", generator=g)).half()
    y = torch.empty((M, 384), dtype=torch.float16, device="cuda")
    engine.launch_linear_residual_layernorm(A, W, b, r, gm, be, y, M, K)
    w0 = 330000  # window rows 330000 .. M-1, M = 30001: the same tile, one chunk
    yw = torch.empty((M - w0, 384), dtype=torch.float16, device="cuda")
    engine.launch_linear_residual_layernorm(A[w0:], W, b, r[w0:], gm, be, yw, M - w0, K)
    torch.cuda.synchronize()
    assert torch.equal(y[w0:], yw)
    rows = torch.from_numpy(np.r_[0:64, edge - 64:edge + 64, M - 64:M]).cuda()
    want = O.layer_norm(O.linear(_np(A[rows]), _np(W), _np(b)), _np(gm), _np(be),
                        residual=_np(r[rows]))
    assert np.abs(_np(y[rows]) - want).max() <= TOL


# ---- LayerNorm ---------------------------------------------------------------

def test_layernorm_reference_kat(torch_cuda, kats):
    torch = torch_cuda
    from bbh import engine

    x, g, b, y = kats["ln_x"], kats["ln_gamma"], kats["ln_beta"], kats["ln_y"]
    out = torch.empty(x.shape, dtype=torch.float16, device="cuda")
    engine.launch_layernorm(to_dev(torch, x), to_dev(torch, g), to_dev(torch, b), out, 128, 384)
    got = _np(out)
    assert cosine_rows(got.ravel(), y.ravel()) >= 0.9995
    assert np.abs(got - y).max() <= TOL


@pytest.mark.parametrize("D,res", [(384, True), (384, False), (100, True), (1536, False)])
def test_layernorm(torch_cuda, D, res):
    torch = torch_cuda
    from bbh import engine

    rng = np.random.default_rng(D)
    M = 77
    x, r = _h(rng, (M, D), 2.0), _h(rng, (M, D))
    g, b = (1 + rng.standard_normal(D) * 0.1).astype(np.float16), _h(rng, (D,), 0.1)
    out = torch.empty((M, D), dtype=torch.float16, device="cuda")
    engine.launch_layernorm(to_dev(torch, x), to_dev(torch, g), to_dev(torch, b), out, M, D,
                            residual=to_dev(torch, r) if res else None)
    f = lambda a: a.astype(np.float32)  # noqa: E731
    want = O.layer_norm(f(x), f(g), f(b), residual=f(r) if res else None)
    assert np.abs(_np(out) - want).max() <= TOL


# ---- embedding -----------------------------------------------------------------

def test_embedding_and_fused_layernorm(torch_cuda, weights16):
    torch = torch_cuda
    from bbh import engine, synth

    rows = [synth.sentence(np.random.default_rng(i), L) for i, L in enumerate([9, 30, 2, 48])]
    ids, types, mask = synth.pack(rows, 48)
    types[1, 5:] = 1
    ids[3, 0] = 30521  # last vocabulary row
    w = weights16
    dw = {k: to_dev(torch, w[k].astype(np.float16)) for k in (
        "embeddings.word_embeddings.weight", "embeddings.position_embeddings.weight",
        "embeddings.token_type_embeddings.weight", "embeddings.LayerNorm.weight",
        "embeddings.LayerNorm.bias")}
    B, S = ids.shape
    ti, tt = to_dev(torch, ids), to_dev(torch, types)
    summed = torch.empty((B * S, 384), dtype=torch.float16, device="cuda")
    engine.launch_embedding(ti, tt, dw["embeddings.word_embeddings.weight"],
                            dw["embeddings.position_embeddings.weight"],
                            dw["embeddings.token_type_embeddings.weight"], summed, S, 384, B)
    want_sum = O.embedding_sum(ids, types, w["embeddings.word_embeddings.weight"],
                               w["embeddings.position_embeddings.weight"],
                               w["embeddings.token_type_embeddings.weight"]).reshape(B * S, 384)
    assert np.abs(_np(summed) - want_sum).max() <= 1e-3
    out = torch.empty((B * S, 384), dtype=torch.float16, device="cuda")
    engine.launch_embedding_layernorm(ti, tt, dw["embeddings.word_embeddings.weight"],
                                      dw["embeddings.position_embeddings.weight"],
                                      dw["embeddings.token_type_embeddings.weight"],
                                      dw["embeddings.LayerNorm.weight"], dw["embeddings.LayerNorm.bias"],
                                      out, S, B)
    want = O.embeddings(w, ids, types).reshape(B * S, 384)
    assert np.abs(_np(out) - want).max() <= TOL


# ---- attention -----------------------------------------------------------------

def _masks(rng, B, S, kind):
    m = np.zeros((B, S), np.int32)
    if kind == "prefix":
        for b in range(B):
            m[b, :rng.integers(1, S + 1)] = 1
    elif kind == "random":
        m = (rng.random((B, S)) > 0.3).astype(np.int32)
        m[:, 0] = 1
    elif kind == "full":
        m[:] = 1
    elif kind == "empty_row":
        for b in range(B):
            m[b, :rng.integers(1, S + 1)] = 1
        m[1] = 0  # every key of sequence 1 masked -> zero context (softmax.cu:57-62)
    return m


@pytest.mark.parametrize("S,kind", [(16, "prefix"), (32, "random"), (48, "empty_row"), (64, "full"),
                                    (80, "prefix"), (128, "random"), (512, "prefix"),
                                    (512, "empty_row"), (256, "rising"), (512, "rising"),
                                    (224, "prefix"), (320, "random")])
def test_fused_attention(torch_cuda, S, kind):
    torch = torch_cuda
    from bbh import engine

    rng = np.random.default_rng(S)
    B = 3
    qkv = _h(rng, (B, S, 1152), 1.5)
    if kind == "rising":
        # Keys whose scores climb along the sequence, by about 10 raw units
        # per 32-key chunk for sequence 0 (the row max moves a little at every
        # chunk) and about 100 for sequence 1 (it jumps at every chunk).
        ramp = np.arange(S, dtype=np.float32)[:, None] * np.array([0.01, 0.1, 0.0])[:, None, None]
        qkv[..., :384] = np.abs(qkv[..., :384])
        qkv[..., 384:768] = (qkv[..., 384:768] * 0.1 + ramp).astype(np.float16)
    mask = _masks(rng, B, S, "full" if kind == "rising" else kind)
    out = torch.empty((B * S, 384), dtype=torch.float16, device="cuda")
    engine.launch_attention(to_dev(torch, qkv.reshape(B * S, 1152)), to_dev(torch, mask), out, B, S)
    want = O.attention(qkv.astype(np.float32), mask).reshape(B * S, 384)
    got = _np(out)
    assert np.abs(got - want).max() <= TOL
    if kind == "empty_row":
        assert np.all(got[S:2 * S] == 0.0)


def test_attention_bits_do_not_depend_on_the_padding(torch_cuda):
    # Every workgroup shape with one query tile a wavefront takes the same
    # rescale decisions per tile and the same key order: a sentence's rows are,
    # bit for bit, the same at every padded length, scores rising along the keys
    # included.  (8 and 16 tiles, two to a wavefront, are close only.)
    torch = torch_cuda
    from bbh import engine

    rng = np.random.default_rng(7)
    for n in (32, 45, 100, 130, 250, 300):
        qkv = _h(rng, (2, 512, 1152), 2.0)
        qkv[0, :, 384:768] += (np.arange(512)[:, None] * 0.02).astype(np.float16)
        ref = None
        lengths = {-(-n // 16) * 16} | {x for x in (64, 112, 128, 144, 176, 208, 256, 288, 400, 496, 512)
                                        if x >= n}
        two = lambda S: -(-S // 32) in (8, 16)  # noqa: E731
        for S in sorted(lengths, key=lambda S: (two(S), S)):
            mask = np.zeros((2, S), np.int32)
            mask[:, :n] = 1
            out = torch.empty((2 * S, 384), dtype=torch.float16, device="cuda")
            x = to_dev(torch, qkv[:, :S].reshape(2 * S, 1152))
            engine.launch_attention(x, to_dev(torch, mask), out, 2, S)
            got = out.cpu().numpy().reshape(2, S, 384)[:, :n]
            ref = got if ref is None else ref
            # rows of a part-filled 32-query tile share its rescale decisions
            # with the rows past the sentence: compare whole tiles
            if not two(S):
                assert np.array_equal(got[:, :n // 32 * 32], ref[:, :n // 32 * 32]), (n, S)
            assert np.abs(got.astype(np.float32) - ref.astype(np.float32)).max() <= 4e-3, (n, S)


@pytest.mark.parametrize("B,S", [(43, 288), (64, 320), (107, 288), (110, 352), (107, 368),
                                 (172, 496), (256, 512), (60, 256), (300, 96), (128, 48), (129, 48),
                                 (129, 64)])
def test_attention_bits_do_not_depend_on_the_batch(torch_cuda, B, S):
    # From 1281 (sequence, head) pairs on, 9-11 query tiles run on 8 wavefronts
    # instead of 12, 9 and 10 also at 513-768 and 1025-1280, two tiles on 2 instead
    # of 4 from 1537 on; 8 and 16 tiles take one shape in every batch (two tiles a
    # wavefront).  The rows of a sentence are, bit for bit, those it has in a
    # batch of three, scores rising along the keys included, and close to fp32.
    # (256 x 512 also walks the sequences from the last one.)
    torch = torch_cuda
    from bbh import engine

    g = torch.Generator(device="cuda").manual_seed(S)
    qkv = 2.0 * torch.randn((B, S, 1152), device="cuda", generator=g)
    qkv[:, :, 384:768] += 0.02 * torch.arange(S, device="cuda")[None, :, None]
    qkv = qkv.half()
    n = torch.randint(1, S + 1, (B,), device="cuda", generator=g)
    n[0] = S
    mask = (torch.arange(S, device="cuda")[None] < n[:, None]).int()

    def attend(rows):
        out = torch.empty((len(rows) * S, 384), dtype=torch.float16, device="cuda")
        engine.launch_attention(qkv[rows].reshape(-1, 1152).contiguous(), mask[rows].contiguous(),
                                out, len(rows), S)
        return out.view(len(rows), S, 384)

    whole = attend(list(range(B)))
    few = [0, B // 2, B - 1]
    part = attend(few)
    for i, b in enumerate(few):
        assert torch.equal(part[i], whole[b]), b
        q, k, v = (qkv[b].float()[:, 384 * j:384 * j + 384].reshape(S, 12, 32).transpose(0, 1)
                   .contiguous() for j in range(3))
        p = torch.softmax((q @ k.transpose(1, 2).contiguous()) / 32 ** 0.5
                          + torch.where(mask[b] != 0, 0.0, float("-inf")), -1)
        want = (p @ v).transpose(0, 1).reshape(S, 384)
        assert (whole[b].float() - want).abs().max().item() <= TOL, b


def test_unfused_attention_pieces_match_fused(torch_cuda):
    # launch_attention_scores -> launch_softmax(mask) -> launch_attention_context
    # (src/model/encoder.cu:39-45) against the oracle and the fused kernel.
    torch = torch_cuda
    from bbh import engine

    rng = np.random.default_rng(21)
    B, S, H = 2, 48, 12
    qkv = _h(rng, (B, S, 1152), 1.5)
    mask = _masks(rng, B, S, "prefix")
    tq, tm = to_dev(torch, qkv.reshape(B * S, 1152)), to_dev(torch, mask)
    scale = 1.0 / np.sqrt(32)
    scores = torch.empty((B * H, S, S), dtype=torch.float16, device="cuda")
    engine.launch_attention_scores(tq, scores, B, H, S, 32, 1152, 0, 384, scale)
    q = qkv[..., :384].astype(np.float32).reshape(B, S, H, 32).transpose(0, 2, 1, 3)
    k = qkv[..., 384:768].astype(np.float32).reshape(B, S, H, 32).transpose(0, 2, 1, 3)
    want_s = (q @ k.transpose(0, 1, 3, 2) * scale).reshape(B * H, S, S)
    assert np.abs(_np(scores) - want_s).max() <= TOL
    engine.launch_softmax(scores, B * H * S, S, tm, H * S)
    want_p = O.masked_softmax(want_s.reshape(B, H, S, S), mask[:, None, None, :]).reshape(B * H, S, S)
    assert np.abs(_np(scores) - want_p).max() <= 2e-3
    merged = torch.empty((B * S, 384), dtype=torch.float16, device="cuda")
    engine.launch_attention_context(scores, tq, merged, B, H, S, 32, 1152, 768)
    want = O.attention(qkv.astype(np.float32), mask).reshape(B * S, 384)
    assert np.abs(_np(merged) - want).max() <= TOL
    fused = torch.empty_like(merged)
    engine.launch_attention(tq, tm, fused, B, S)
    assert np.abs(_np(fused) - _np(merged)).max() <= TOL


@pytest.mark.parametrize("K", [384, 1536])
def test_residual_layernorm_rows_above_8192(torch_cuda, K):
    # From 8193 rows on the row sums are normalised in fp32, by whichever
    # kernel: the rows of any such call are, bit for bit, those of a call with
    # 65535 rows (a pass over fp16 sums would differ); K = 1536 those of one
    # with 70000 rows too.  (K = 384 runs on the weight-resident kernel from
    # 65536 rows on, which groups the columns of a row's statistics otherwise.)
    torch = torch_cuda
    from bbh import engine

    g = torch.Generator(device="cuda").manual_seed(K)
    r = lambda *s: torch.randn(s, device="cuda", generator=g).half()  # noqa: E731
    A, R = r(70000, K), r(70000, 384)
    W, b, gm, be = (r(384, K) / K ** 0.5).half(), r(384), r(384), r(384)
    ref, rows = torch.empty_like(R), 65535 if K == 384 else 70000
    engine.launch_linear_residual_layernorm(A, W, b, R, gm, be, ref, rows, K)
    for M in (8193, 8705, 10881, 16384, 16385, 50000):
        y = torch.full((M + 1, 384), 7.0, dtype=torch.float16, device="cuda")
        engine.launch_linear_residual_layernorm(A, W, b, R, gm, be, y, M, K)
        assert torch.equal(y[:M], ref[:M]), M
        assert torch.all(y[M] == 7.0)


@pytest.mark.parametrize("N,K,Ms", [
    # The one-workgroup-per-CU tiles: at most 256 workgroups of 32x64, 64x64,
    # 96x64, 128x64, 96x128 and 128x128 (K >= 1024), each at its last row count
    # and one past it; 17 slices leave a part-filled group of two.
    (384, 1536, (1, 33, 1344, 1345, 2688, 2689, 4032, 4033, 5376, 5377, 8160, 8161)),
    (384, 1088, (16, 2500)), (64, 1024, (8000,)),
    # K < 1024: 32x64, 64x64, 96x64, 64x128; three slices, one slice.
    (384, 384, (16, 1345, 2689, 4033, 5440)), (1536, 384, (320, 321, 641, 961, 1344, 1345)),
    (1152, 192, (31, 449)), (128, 64, (1, 4097)),
    # N = 1152 past one round of 128x128 tiles
    (1152, 384, (7168, 7169))])
def test_linear_rows_do_not_depend_on_the_tile(torch_cuda, N, K, Ms):
    # Every tile adds k in the same order and rounds the same way: the rows of
    # any row count are, bit for bit, those of a call with 50000 rows.
    torch = torch_cuda
    from bbh import engine

    g = torch.Generator(device="cuda").manual_seed(N + K)
    A = torch.randn((50000, K), device="cuda", generator=g).half()
    W = (torch.randn((N, K), device="cuda", generator=g) / K ** 0.5).half()
    b = (torch.randn((N,), device="cuda", generator=g) * 0.1).half()
    ref = torch.empty((50000, N), dtype=torch.float16, device="cuda")
    engine.launch_matmul(A, W, ref, 50000, N, K, bias=b)
    for M in Ms:
        C = torch.full((M + 1, N), 7.0, dtype=torch.float16, device="cuda")
        engine.launch_matmul(A, W, C, M, N, K, bias=b)
        assert torch.equal(C[:M], ref[:M]), M
        assert torch.all(C[M] == 7.0)  # nothing past the last row


@pytest.mark.parametrize("B,S,off", [(1, 16, 0), (3, 48, 1), (2, 80, 0), (2, 128, 3), (1, 144, 0),
                                     (1, 528, 1), (2, 33, 0), (1, 520, 1), (1, 1040, 0)])
def test_unfused_attention_pieces_edges(torch_cuda, B, S, off):
    # Tile edges of the three operators (32 queries, 64 keys, 16-key steps,
    # 512 staged keys, rows of 2 to 64 lanes and longer), lengths that only the
    # general kernels take (S % 16), and buffers at odd element addresses.
    # Each is compared with float64 on its own fp16 input; bounds: fp16
    # rounding 2^-11 plus the fp32 sums' S * 2^-24 of the absolute sum, both
    # doubled.
    torch = torch_cuda
    from bbh import engine

    rng = np.random.default_rng(S)
    H, ld, scale = 3, 3 * 96 + 8, 1.0 / np.sqrt(32)
    qkv = _h(rng, (B * S, ld), 1.5)
    tq = to_dev(torch, qkv)
    q, k, v = (qkv[:, o:o + 96].astype(np.float64).reshape(B, S, H, 32).transpose(0, 2, 1, 3)
               for o in (8, 104, 200))
    mask = _masks(rng, B, S, "random")
    mask[-1] = 0  # every key masked: zero probabilities
    scores = torch.zeros(B * H * S * S + off, dtype=torch.float16, device="cuda")[off:]
    if S % 16 == 0:
        engine.launch_attention_scores(tq, scores, B, H, S, 32, ld, 8, 104, scale)
        want = np.matmul(q, k.transpose(0, 1, 3, 2)) * scale
        mag = np.matmul(np.abs(q), np.abs(k).transpose(0, 1, 3, 2)) * scale
        got = _np(scores).reshape(want.shape)
        assert np.all(np.abs(got - want) <= 2 ** -10 * np.abs(want) + 32 * 2 ** -23 * mag)
    else:
        scores += to_dev(torch, _h(rng, (B * H * S * S,), 2.0))
    x = _np(scores).reshape(B, H, S, S).astype(np.float64)
    engine.launch_softmax(scores, B * H * S, S, to_dev(torch, mask), H * S)
    m = mask[:, None, None, :] != 0
    e = np.where(m, np.exp(x - np.max(np.where(m, x, -1e9), -1, keepdims=True)), 0.0)
    want = e / np.maximum(e.sum(-1, keepdims=True), 1e-300)
    probs = _np(scores).reshape(want.shape)
    assert np.all(np.abs(probs - want) <= (2 ** -10 + S * 2 ** -23) * want + 2 ** -23)
    out = torch.empty(B * S * H * 32 + off, dtype=torch.float16, device="cuda")[off:]
    engine.launch_attention_context(scores, tq, out, B, H, S, 32, ld, 200)
    p = probs.astype(np.float64)
    want = np.matmul(p, v).transpose(0, 2, 1, 3).reshape(B * S, H * 32)
    mag = np.matmul(p, np.abs(v)).transpose(0, 2, 1, 3).reshape(B * S, H * 32)
    got = _np(out).reshape(want.shape)
    assert np.all(np.abs(got - want) <= 2 ** -10 * np.abs(want) + S * 2 ** -23 * mag + 2 ** -24)


@pytest.mark.parametrize("B,S,D,off", [(1, 1, 8, 0), (3, 7, 384, 1), (2, 512, 384, 0), (2, 40, 1032, 0),
                                       (5, 33, 100, 0), (1, 90, 8200, 0), (2, 3, 512, 1),
                                       # the pool's workgroup a sentence, at its edges
                                       (2, 8, 8, 0), (3, 9, 384, 1), (2, 40, 1024, 0), (600, 12, 512, 1),
                                       (600, 8, 384, 0), (256, 8, 8192, 0)])
def test_row_operators_edges(torch_cuda, B, S, D, off):
    # embedding, mean pool and L2 normalise at any width (the vector kernels
    # take D % 8 == 0, the pool's up to 8192 columns where it pays, the
    # normalise's up to 512), at odd element addresses,
    # with an all-masked sentence; NaN in masked rows is not read.  Bounds as
    # above; the embedding is exact up to its fp16 rounding.
    torch = torch_cuda
    from bbh import engine

    rng = np.random.default_rng(D + S)
    at = lambda a: to_dev(torch, np.concatenate([np.zeros(off, a.dtype), a.ravel()]))[off:]  # noqa: E731
    word, pos, typ = np.zeros((30522, D), np.float16), _h(rng, (S, D)), _h(rng, (2, D))
    rows = rng.integers(0, 30522, 64)
    word[rows] = _h(rng, (64, D))
    ids = rng.choice(rows, (B, S)).astype(np.int32)
    types = rng.integers(0, 2, (B, S)).astype(np.int32)
    out = torch.empty(B * S * D + off, dtype=torch.float16, device="cuda")[off:]
    engine.launch_embedding(to_dev(torch, ids), to_dev(torch, types), at(word), at(pos), at(typ), out,
                            S, D, B)
    f = lambda a: a.astype(np.float32)  # noqa: E731
    want = ((f(word)[ids] + f(pos)[None]) + f(typ)[types]).astype(np.float16)
    assert np.array_equal(out.cpu().numpy().reshape(B, S, D), want)
    h = _h(rng, (B, S, D))
    mask = _masks(rng, B, S, "random")
    mask[B - 1] = B == 1
    h[mask == 0] = np.nan
    pooled = torch.empty(B * D + off, dtype=torch.float16, device="cuda")[off:]
    engine.launch_mean_pool(at(h), to_dev(torch, mask), pooled, S, D, B)
    hz, n = np.where(mask[..., None] != 0, h, 0).astype(np.float64), np.maximum(mask.sum(1), 1)[:, None]
    want, mag = hz.sum(1) / n, np.abs(hz).sum(1) / n
    got = _np(pooled).reshape(B, D)
    assert np.all(np.abs(got - want) <= 2 ** -10 * np.abs(want) + S * 2 ** -23 * mag + 2 ** -24)
    engine.launch_l2_normalize(pooled, D, B)
    want = got / np.maximum(np.linalg.norm(got.astype(np.float64), axis=1, keepdims=True), 1e-12)
    got = _np(pooled).reshape(B, D)
    assert np.all(np.abs(got - want) <= (2 ** -10 + D * 2 ** -23) * np.abs(want) + 2 ** -24)


def test_mean_pool_of_many_short_rows(torch_cuda):
    # More sentences than a launch of one 1024-thread workgroup each can hold
    # (2^32 threads): every row is written, the last ones too.
    torch = torch_cuda
    from bbh import engine

    B, D = (1 << 22) + 8, 8
    h = (torch.arange(B, device="cuda") % 2048).half()[:, None] + torch.arange(D, device="cuda").half()
    mask = torch.ones((B, 1), dtype=torch.int32, device="cuda")
    out = torch.full((B, D), -1.0, dtype=torch.float16, device="cuda")
    engine.launch_mean_pool(h, mask, out, 1, D, B)
    assert torch.equal(out, h)  # the mean of one row


def test_softmax_reference_kat(torch_cuda, kats):
    torch = torch_cuda
    from bbh import engine

    x = to_dev(torch, kats["softmax_x"])
    engine.launch_softmax(x, 128, 128)
    got = _np(x)
    assert cosine_rows(got.ravel(), kats["softmax_y"].ravel()) >= 0.9999
    assert np.abs(got - kats["softmax_y"]).max() <= 2e-3


# ---- GELU ----------------------------------------------------------------------

def test_gelu_reference_kat(torch_cuda, kats):
    # tests/test_gelu.cu: exact GELU in place over 128 x 1536 fp16 values
    torch = torch_cuda
    from bbh import engine

    x = to_dev(torch, kats["gelu_x"])
    engine.launch_gelu(x, x.numel())
    got, want = _np(x), kats["gelu_y"]
    assert cosine_rows(got.ravel(), want.ravel()) >= 0.9999
    assert np.abs(got - want).max() <= 4e-3  # half an fp16 ulp at |y| ~ 8


def test_gelu_unaligned_and_ragged(torch_cuda, kats):
    # a start 6 bytes past a 16-byte boundary and a length that is not a
    # multiple of 8 take the one-value-per-thread kernel; nothing outside is touched
    torch = torch_cuda
    from bbh import engine

    src = kats["gelu_x"][:1000]
    x = to_dev(torch, src)
    engine.launch_gelu(x[3:], 990)
    got = _np(x)
    want = O.gelu(src[3:993].astype(np.float32))
    assert np.abs(got[3:993] - want).max() <= 4e-3
    assert np.array_equal(got[:3], src[:3].astype(np.float32))
    assert np.array_equal(got[993:], src[993:].astype(np.float32))


# ---- pooling / normalize --------------------------------------------------------

@pytest.mark.parametrize("B,S", [(1, 16), (5, 48), (64, 128), (3, 512)])
def test_pool_normalize(torch_cuda, B, S):
    torch = torch_cuda
    from bbh import engine

    rng = np.random.default_rng(B * S)
    h = _h(rng, (B, S, 384))
    mask = _masks(rng, B, S, "prefix")
    if B > 2:
        mask[2] = 0  # no real token -> zero embedding (pooling.cu:30, normalize.cu:30)
    th, tm = to_dev(torch, h.reshape(B * S, 384)), to_dev(torch, mask)
    f32 = h.astype(np.float32)
    out = torch.empty((B, 384), dtype=torch.float16, device="cuda")
    engine.launch_pool_normalize(th, tm, out, S, B)
    want = O.l2_normalize(O.mean_pool(f32, mask))
    got = _np(out)
    assert np.abs(got - want).max() <= 2e-3
    pooled = torch.empty((B, 384), dtype=torch.float16, device="cuda")
    engine.launch_mean_pool(th, tm, pooled, S, 384, B)
    assert np.abs(_np(pooled) - O.mean_pool(f32, mask)).max() <= 2e-3
    engine.launch_l2_normalize(pooled, 384, B)
    assert np.abs(_np(pooled) - want).max() <= 2e-3
    if B > 2:
        assert np.all(got[2] == 0.0)


@pytest.mark.parametrize("B,S", [(256, 32), (171, 48), (95, 96), (113, 144), (256, 64), (205, 80)])
def test_ffn_block_from_sliced_weights(torch_cuda, ws, model, weights32, B, S):
    # 8192 to 16400 rows: above 8192 and up to 16384 ffn_block reads FFN2's weights
    # from the model's sliced copy, the standalone launchers read them
    # row-major.  Same bits, and no row past the last one written.
    from bbh import engine

    torch = torch_cuda
    M = B * S
    g = torch.Generator(device="cuda").manual_seed(M)
    hid = torch.randn((M, 384), device="cuda", generator=g).half()
    for i in (0, 5):
        p = "encoder.layer.%d." % i
        w = {k[len(p):]: to_dev(torch, v.astype(np.float16)) for k, v in weights32.items()
             if k.startswith(p)}
        inter = torch.empty((M, 1536), dtype=torch.float16, device="cuda")
        engine.launch_matmul(hid, w["intermediate.dense.weight"], inter, M, 1536, 384,
                             bias=w["intermediate.dense.bias"], gelu=True)
        want = torch.empty_like(hid)
        engine.launch_linear_residual_layernorm(
            inter, w["output.dense.weight"], w["output.dense.bias"], hid,
            w["output.LayerNorm.weight"], w["output.LayerNorm.bias"], want, M, 1536)
        out = torch.full((M + 1, 384), 7.0, dtype=torch.float16, device="cuda")
        engine.ffn_block(ws, model, i, hid, out, B, S)
        assert torch.equal(out[:M], want)
        assert torch.all(out[M] == 7.0)


@pytest.mark.parametrize("B,S", [(4097, 16), (192, 512), (256, 512)])
def test_ffn_one_kernel_equals_two_kernels(torch_cuda, ws, model, weights32, weights16, B, S):
    # From 65536 rows bbh_ffn_block runs the FFN as one kernel (intermediate
    # kept on chip).  Against the intermediate Linear + GELU and the output
    # Linear + residual + LayerNorm launched one by one through the standalone
    # launchers, call after call: a ragged last 128-row block (4097 x 16 =
    # 65552 rows), three and four row blocks per workgroup (98304, 131072
    # rows).  Same arithmetic, so the outputs agree except where an fp16
    # rounding falls on a midpoint: at most one fp16 step, on at most 2e-5 of
    # the elements.  Then against the fp32 oracle on every 7th row (all row
    # positions of the 128-row blocks, every block) and the last 40.  (The
    # forward runs the kernel in place on its last layer: covered end to end
    # by the cfg5 tests.)
    from bbh import engine

    torch = torch_cuda
    rng = np.random.default_rng(B * 7 + S)
    M = B * S
    p = "encoder.layer.4."
    w = {k[len(p):]: to_dev(torch, v.astype(np.float16)) for k, v in weights32.items()
         if k.startswith(p)}
    hid = to_dev(torch, _h(rng, (M, 384)))
    inter = torch.empty((M, 1536), dtype=torch.float16, device="cuda")
    engine.launch_matmul(hid, w["intermediate.dense.weight"], inter, M, 1536, 384,
                         bias=w["intermediate.dense.bias"], gelu=True)
    want = torch.empty_like(hid)
    engine.launch_linear_residual_layernorm(inter, w["output.dense.weight"], w["output.dense.bias"],
                                            hid, w["output.LayerNorm.weight"],
                                            w["output.LayerNorm.bias"], want, M, 1536)
    del inter
    wn = _np(want)
    step = np.spacing(np.abs(wn).astype(np.float16)).astype(np.float32)  # one fp16 step
    first = None
    for rep in range(2):
        got = torch.empty_like(hid)
        engine.ffn_block(ws, model, 4, hid, got, B, S)
        torch.cuda.synchronize()
        g = _np(got)
        diff = g != wn
        assert diff.mean() <= 2e-5, (rep, int(diff.sum()))
        assert np.all(np.abs(g - wn)[diff] <= step[diff]), rep
        if first is None:
            first = g
        else:
            assert np.array_equal(g, first)  # deterministic call after call
    rows = np.unique(np.r_[0:M:7, M - 40:M])
    x = _np(hid)[rows]
    ref = O.ffn_block(x.reshape(1, -1, 384), O._layer(weights16, 4)).reshape(-1, 384)
    assert np.abs(_np(got)[rows] - ref).max() <= TOL


@pytest.mark.parametrize("B,S", [(1, 16), (64, 16), (5, 32), (31, 48), (64, 48), (64, 64), (96, 64),
                                 (128, 64), (64, 128)])
def test_workspace_residual_layernorm_equals_two_pass(torch_cuda, ws, model, weights32, B, S):
    # The workspace blocks (bbh_ffn_block, bbh_attention_block) against their
    # kernels launched one by one through the standalone launchers (Linear,
    # attention, Linear + residual + LayerNorm): equal bit for bit, call after
    # call, at every M regime of a batch-64 forward (and 8192 rows, the last
    # with a separate LayerNorm pass); masks with holes, a fully masked
    # sentence and a one-key sentence included.
    from bbh import engine

    torch = torch_cuda
    rng = np.random.default_rng(B * 1000 + S)
    M = B * S
    p = "encoder.layer.2."
    w = {k[len(p):]: to_dev(torch, v.astype(np.float16)) for k, v in weights32.items()
         if k.startswith(p)}
    hid = to_dev(torch, _h(rng, (M, 384)))
    m = (rng.random((B, S)) < 0.8).astype(np.int32)
    m[0, :] = 1
    if B > 2:
        m[1, :] = 0  # every key masked: zero context
        m[2, 1:] = 0  # one key
    mask = to_dev(torch, m)
    # FFN block: FFN1 + GELU, then FFN2 + residual + LayerNorm
    inter = torch.empty((M, 1536), dtype=torch.float16, device="cuda")
    engine.launch_matmul(hid, w["intermediate.dense.weight"], inter, M, 1536, 384,
                         bias=w["intermediate.dense.bias"], gelu=True)
    want = torch.empty_like(hid)
    engine.launch_linear_residual_layernorm(inter, w["output.dense.weight"], w["output.dense.bias"],
                                            hid, w["output.LayerNorm.weight"],
                                            w["output.LayerNorm.bias"], want, M, 1536)
    for rep in range(3):
        got = torch.empty_like(hid)
        engine.ffn_block(ws, model, 2, hid, got, B, S)
        torch.cuda.synchronize()
        assert torch.equal(got, want), (rep, (got.float() - want.float()).abs().max().item())
    # attention block: QKV, attention, O-proj + residual + LayerNorm
    qkv_w = torch.cat([w[f"attention.self.{n}.weight"] for n in ("query", "key", "value")])
    qkv_b = torch.cat([w[f"attention.self.{n}.bias"] for n in ("query", "key", "value")])
    qkv = torch.empty((M, 1152), dtype=torch.float16, device="cuda")
    engine.launch_matmul(hid, qkv_w, qkv, M, 1152, 384, bias=qkv_b)
    ctx = torch.empty_like(hid)
    engine.launch_attention(qkv, mask, ctx, B, S)
    want_a = torch.empty_like(hid)
    engine.launch_linear_residual_layernorm(ctx, w["attention.output.dense.weight"],
                                            w["attention.output.dense.bias"], hid,
                                            w["attention.output.LayerNorm.weight"],
                                            w["attention.output.LayerNorm.bias"], want_a, M, 384)
    for rep in range(2):
        got_a = torch.empty_like(hid)
        engine.attention_block(ws, model, 2, hid, mask, got_a, B, S)
        torch.cuda.synchronize()
        assert torch.equal(got_a, want_a), rep
