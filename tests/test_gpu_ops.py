"""Op-tier parity on the GPU: each C-ABI op against the oracle on seeded inputs.

Shapes: the five GEMV shapes of the isolated-kernel microbench (lm_head
151936x1536, gate/up 8960x1536, down 1536x8960, q/o 1536x1536, k/v 256x1536)
plus tails that take the generic kernel (k % 8 != 0), and the reference's
own hand cases.
"""
import importlib

import numpy as np
import pytest

import oracle
from model_fixtures import THETA, bits, rne_bf16
from parity import dot_bound, max_rel

torch = pytest.importorskip("torch")
myos = importlib.import_module("an-operating-system-for-ai-models-and-tensor-inference_amd")

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def dev(a, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a))
    if dtype is not None:
        t = t.view(dtype)
    return t.to(DEV)


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def rand_w(rng, m, k):
    return rne_bf16(rng.standard_normal((m, k), dtype=np.float32) * np.float32(0.02))


MICRO = [(151936, 1536), (8960, 1536), (1536, 8960), (1536, 1536), (256, 1536)]


@pytest.mark.parametrize("m,k", MICRO + [(17920, 1536), (2048, 1536), (3584, 18944),
                                         (7, 3), (9, 17), (33, 24), (5, 1000), (40, 4104)])
def test_gemv_vs_oracle(m, k):
    rng = np.random.default_rng(m * 31 + k)
    w = rand_w(rng, m, k)
    x = rng.standard_normal(k, dtype=np.float32)
    ref = oracle.gemv_bf16(w, x, m, k, threads=8)
    y = torch.full((m,), 7.0, dtype=torch.float32, device=DEV)
    myos.gemv_bf16(y, dev(w, torch.int16), dev(x), m, k)
    got = host(y)
    bound = dot_bound(oracle.bf16_to_f32(w), x)
    assert np.all(np.abs(got.astype(np.float64) - ref) <= bound)
    assert max_rel(got, ref) < 1e-5


def test_gemv_hand_values_and_errors():
    w = dev(bits([1.0, 2.0, 0.5, -1.0, 4.0, 1.5]), torch.int16)
    x = dev(np.array([1.0, -2.0, 0.5], np.float32))
    y = torch.zeros(2, dtype=torch.float32, device=DEV)
    myos.gemv_bf16(y, w, x, 2, 3)
    assert list(host(y)) == [-2.75, -8.25]
    # k == 0 fills zero; errors leave y untouched
    y = torch.tensor([1.0, 2.0], device=DEV)
    myos.gemv_bf16(y, torch.zeros(0, dtype=torch.int16, device=DEV),
                   torch.zeros(0, device=DEV), 2, 0)
    assert list(host(y)) == [0.0, 0.0]
    kept = torch.tensor([7.0, 8.0], device=DEV)
    with pytest.raises(myos.MyosError) as e:
        myos.gemv_bf16(kept, dev(bits([1.0, 2.0]), torch.int16), dev(np.ones(2, np.float32)), 2, 2)
    assert e.value.kind == "RowOutOfBounds" and list(host(kept)) == [7.0, 8.0]


def test_gemv_order_cancellation():
    # gemv_bf16_kernel.rs:929-951: exact in any summation order only if the
    # 2^24 terms cancel before the ones are absorbed; record what the GPU gives
    row = [16777216.0, 1.0, 1.0, 1.0, -16777216.0, 1.0, 1.0, 1.0]
    w = dev(bits(np.tile(row, 64)), torch.int16)
    y = torch.zeros(64, device=DEV)
    myos.gemv_bf16(y, w, dev(np.ones(8, np.float32)), 64, 8)
    got = host(y)
    # any order: the result is one of the values a reordering can produce
    assert np.all(np.isin(got, [0.0, 1.0, 2.0, 3.0, 4.0]))


# projections of the 1.5B and 7B shapes and generic ones: split K, row tails,
# several row tiles, nine of them (the XCD-aware tile order) with K splits, and
# K % 64 != 0 (the single-stage kernel); test_gemm_tiles goes over every tile
@pytest.mark.parametrize("batch,m,k", [(128, 1536, 1536), (128, 256, 1536), (37, 8960, 1536),
                                       (128, 1536, 8960), (128, 4608, 3584), (100, 17920, 1536),
                                       (1100, 1536, 640), (200, 1536, 8960), (1100, 4096, 256),
                                       (600, 4096, 512), (300, 8960, 512), (300, 1536, 4096),
                                       (300, 1280, 4096), (1030, 1536, 8960),
                                       (5, 7, 3), (33, 70, 45), (200, 130, 200)])
def test_gemm_vs_oracle(batch, m, k):
    rng = np.random.default_rng(batch + m + k)
    w = rand_w(rng, m, k)
    x = rng.standard_normal((batch, k), dtype=np.float32)
    ref = oracle.gemm_bf16(w, x, batch, m, k, threads=8)
    y = torch.zeros((batch, m), dtype=torch.float32, device=DEV)
    myos.gemm_bf16(y, dev(w, torch.int16), dev(x), batch, m, k)
    got = host(y)
    # hi + lo split keeps x to within 2^-17 |x| (two RNE roundings of 2^-9)
    # MFMA accumulation may not round to nearest: allow 4 gamma_k
    bound = dot_bound(oracle.bf16_to_f32(w), x, extra_rel=2.0 ** -17, gamma_mult=4).T
    assert np.all(np.abs(got.astype(np.float64) - ref) <= bound)


def test_bias_embed_rmsnorm_swiglu():
    rng = np.random.default_rng(3)
    y0 = rng.standard_normal(1536).astype(np.float32)
    b = rand_w(rng, 1, 1536)[0]
    y = dev(y0)
    myos.add_bf16_bias(y, dev(b, torch.int16))
    assert np.array_equal(host(y), oracle.add_bf16_bias(y0, b))  # one f32 add: exact

    table = rand_w(rng, 1000, 1536)
    out = torch.zeros(1536, device=DEV)
    myos.embed_gather_bf16(out, dev(table, torch.int16), (1000, 1536), 417)
    assert np.array_equal(host(out), oracle.embed_gather_bf16(table, 1000, 1536, 417)[1])
    with pytest.raises(myos.MyosError) as e:
        myos.embed_gather_bf16(out, dev(table, torch.int16), (1000, 1536), 1000)
    assert e.value.kind == "TokenOutOfBounds"

    x = rng.standard_normal(1536).astype(np.float32)
    g = rand_w(rng, 1, 1536)[0]
    y = torch.zeros(1536, device=DEV)
    myos.rmsnorm_bf16_weight(y, dev(g, torch.int16), dev(x), np.float32(1e-6))
    assert max_rel(host(y), oracle.rmsnorm_bf16_weight(g, x, np.float32(1e-6))) < 1e-6
    # hand values (bf16.rs:469-486) are exact in any order
    y = torch.zeros(4, device=DEV)
    myos.rmsnorm_bf16_weight(y, dev(bits([1.5, 4.0, -2.0, 0.5]), torch.int16),
                             dev(np.array([8.0, 0, 0, 0], np.float32)), 0.0)
    assert list(host(y)) == [3.0, 0.0, 0.0, 0.0]

    gate = rng.standard_normal(8960).astype(np.float32) * 3
    up = rng.standard_normal(8960).astype(np.float32)
    h = torch.zeros(8960, device=DEV)
    myos.swiglu_mul_f32(h, dev(gate), dev(up))
    assert max_rel(host(h), oracle.swiglu_mul_f32(gate, up)) < 1e-6


@pytest.mark.parametrize("hidden,inter", [(1536, 8960), (48, 100), (37, 19)])
def test_swiglu_bf16_vs_oracle(hidden, inter):
    # swiglu.rs:184-213 composed on the oracle: gate, up, h, y
    rng = np.random.default_rng(hidden + inter)
    x = rng.standard_normal(hidden).astype(np.float32)
    wg, wu, wd = rand_w(rng, inter, hidden), rand_w(rng, inter, hidden), rand_w(rng, hidden, inter)
    g_ref = oracle.gemv_bf16(wg, x, inter, hidden, threads=8)
    u_ref = oracle.gemv_bf16(wu, x, inter, hidden, threads=8)
    h_ref = oracle.swiglu_mul_f32(g_ref, u_ref)
    y_ref = oracle.gemv_bf16(wd, h_ref, hidden, inter, threads=8)
    y = torch.zeros(hidden, device=DEV)
    g, u, h = (torch.zeros(inter, device=DEV) for _ in range(3))
    myos.swiglu_bf16(y, dev(x), dev(wg, torch.int16), dev(wu, torch.int16), dev(wd, torch.int16),
                     g, u, h, hidden, inter)
    assert max_rel(host(g), g_ref) < 1e-5 and max_rel(host(u), u_ref) < 1e-5
    assert max_rel(host(h), h_ref) < 1e-5
    assert max_rel(host(y), y_ref) < 1e-4
    # a shape error leaves every output as it was
    y.fill_(7.0)
    with pytest.raises(myos.MyosError) as e:
        myos.swiglu_bf16(y, dev(x), dev(wg, torch.int16), dev(wu, torch.int16),
                         dev(wd[:-1], torch.int16), g, u, h, hidden, inter)
    assert e.value.kind == "Shape" and bool((y == 7.0).all())


def test_silu_rmsnorm_f32_inv_freqs_scale():
    # silu_f32 (swiglu.rs:113-115) elementwise, against the oracle's libm silu
    # and the reference's bits (swiglu.rs:362-377: silu(1) = 0x3F3B26A8)
    z0 = np.concatenate([np.float32([1.0, 0.0, -1.0, 20.0, -20.0, 1e-3]),
                         np.random.default_rng(4).standard_normal(4000).astype(np.float32) * 6])
    y = torch.zeros(z0.size, device=DEV)
    myos.silu_f32(y, dev(z0))
    got = host(y)
    ref = np.array([oracle.silu_f32(float(v)) for v in z0], np.float32)
    assert got[0].view(np.uint32) == 0x3F3B26A8
    assert np.all(np.abs(got - ref) <= 4 * 2.0 ** -24 * np.maximum(np.abs(ref), 2.0 ** -126))
    # rmsnorm_f32 (bf16.rs:200-216) against the reference's f32 expression
    rng = np.random.default_rng(6)
    x = rng.standard_normal(1536).astype(np.float32)
    w = rng.uniform(0.5, 1.5, 1536).astype(np.float32)
    yr = torch.zeros(1536, device=DEV)
    myos.rmsnorm_f32(yr, dev(w), dev(x), np.float32(1e-6))
    inv = np.float32(1) / np.float32(np.sqrt(np.float32(np.sum(x.astype(np.float64) ** 2) / 1536)
                                             + np.float32(1e-6)))
    assert max_rel(host(yr), w * (x * inv)) < 1e-6
    yr = torch.zeros(4, device=DEV)
    myos.rmsnorm_f32(yr, dev(np.float32([1.5, 4.0, -2.0, 0.5])), dev(np.float32([8, 0, 0, 0])), 0.0)
    assert list(host(yr)) == [3.0, 0.0, 0.0, 0.0]
    # rope_inv_freqs (rope.rs:89-98) bit for bit with the oracle (both libm powf)
    for d in (2, 64, 128):
        t = torch.zeros(d // 2, device=DEV)
        myos.rope_inv_freqs(t, d, THETA)
        assert list(host(t).view(np.uint32)) == list(oracle.rope_inv_freqs(d, THETA).view(np.uint32))
    # attn_scale_f32 (gqa.rs:158-163)
    for d in (1, 32, 128):
        assert np.float32(myos.attn_scale_f32(d)) == oracle.attn_scale_f32(d)


@pytest.mark.parametrize("pos,d,heads", [(1, 2, 1), (3, 4, 2), (8, 128, 12), (2303, 128, 2),
                                         (0, 128, 12)])
def test_rope(pos, d, heads):
    rng = np.random.default_rng(pos + d)
    x0 = rng.standard_normal(heads * d).astype(np.float32)
    _, ref = oracle.rope_f32_inplace(x0, pos, d, THETA)
    x = dev(x0)
    myos.rope_f32_inplace(x, pos, d, THETA)
    got = host(x)
    # angles are the reference's (host libm); only the 2-term combine may
    # round differently (a fused multiply-add), so within 2 ulp of |x0|+|x1|
    assert np.all(np.abs(got - ref) <= 8 * 2.0 ** -24 * np.abs(x0).max())
    if pos == 0:
        assert np.array_equal(got, x0)


def test_rope_hand_bits():
    x = dev(np.array([1.0, 0.0], np.float32))
    myos.rope_f32_inplace(x, 1, 2, THETA)
    assert [int(v) for v in host(x).view(np.uint32)] == [0x3F0A5140, 0x3F576AA4]


@pytest.mark.parametrize("nq,nkv,d,seq,causal", [(12, 2, 128, 1, None), (12, 2, 128, 256, None),
                                                 (12, 2, 128, 300, 150), (4, 2, 1, 2, None),
                                                 (28, 4, 128, 700, None), (1, 1, 4, 2, 0)])
def test_gqa(nq, nkv, d, seq, causal):
    rng = np.random.default_rng(nq * seq + d)
    q = rng.standard_normal(nq * d).astype(np.float32)
    k = rng.standard_normal(nkv * seq * d).astype(np.float32)
    v = rng.standard_normal(nkv * seq * d).astype(np.float32)
    ref, probs_ref = oracle.gqa_attn_f32(q, k, v, nq, nkv, d, seq, causal)
    y = torch.zeros(nq * d, device=DEV)
    probs = torch.zeros(seq, device=DEV)
    myos.gqa_attn_f32(y, dev(q), dev(k), dev(v), probs, nq, nkv, d, seq, causal)
    assert max_rel(host(y), ref) < 1e-5
    assert max_rel(host(probs), probs_ref) < 1e-5


def test_gqa_hand_bits_close():
    # gqa.rs:366-401
    y = torch.zeros(4, device=DEV)
    probs = torch.zeros(2, device=DEV)
    myos.gqa_attn_f32(y, dev(np.array([1, 1, 4, 4], np.float32)),
                      dev(np.array([1, 0, 0, 2], np.float32)),
                      dev(np.array([10, 0, 0, 7], np.float32)), probs, 4, 2, 1, 2)
    ref = np.array([0x40E9F052, 0x40E9F052, 0x40DFECC5, 0x40DFECC5], np.uint32).view(np.float32)
    assert max_rel(host(y), ref) < 1e-6


@pytest.mark.parametrize("case", ["ties", "nan", "allnan", "neginf", "big"])
def test_greedy_token(case):
    rng = np.random.default_rng(11)
    if case == "big":
        lg = rng.standard_normal(151936).astype(np.float32)
        lg[[5000, 140000]] = 9.0  # tie across blocks: lowest index wins
    elif case == "ties":
        lg = np.array([1.0, 3.0, 3.0, 2.0], np.float32)
    elif case == "nan":
        lg = np.array([np.nan, 1.0, np.nan], np.float32)
    elif case == "allnan":
        lg = np.full(9000, np.nan, np.float32)
    else:
        lg = np.full(5, -np.inf, np.float32)
        lg[3] = np.nan
    assert myos.greedy_token(dev(lg)) == oracle.greedy_token(lg)


def _gqa64(q, k, v, n):
    """Row-wide softmax attention in float64 over the first n positions."""
    g = q.shape[0] // k.shape[0]
    K, V = (np.repeat(t.astype(np.float64), g, 0)[:, :n] for t in (k, v))
    with np.errstate(all="ignore"):
        s = np.einsum("hd,htd->ht", q.astype(np.float64), K) / np.sqrt(q.shape[1])
        e = np.exp(s - s.max(1, keepdims=True))
        p = e / e.sum(1, keepdims=True)
        return (p[:, :, None] * V).sum(1), p[-1]


# the chunked kernel: one chunk (up to 1024 positions and 131072 values of K per
# head) and the first split beyond, a last chunk of one position, 16 / 32 / 64 column groups with idle lanes
# (d = 4, 36, 100, 256), more heads than CUs, a masked tail; d = 30 and an
# offset view stay on the general kernel
@pytest.mark.parametrize("nq,nkv,d,seq,causal,shift", [
    (12, 2, 128, 128, None, 0), (12, 2, 128, 1024, None, 0), (12, 2, 128, 1025, None, 0),
    (2, 1, 256, 512, None, 0), (2, 1, 256, 513, None, 0), (28, 4, 128, 2049, None, 0),
    (12, 2, 128, 512, 300, 0), (4, 4, 64, 1000, 999, 0), (3, 1, 4, 129, None, 0), (2, 1, 36, 161, 5, 0),
    (2, 2, 100, 333, 200, 0), (7, 7, 256, 700, None, 0), (300, 1, 64, 257, None, 0),
    (2, 1, 30, 300, None, 0), (2, 1, 64, 300, None, 1)])
def test_gqa_chunks(nq, nkv, d, seq, causal, shift):
    rng = np.random.default_rng(nq + d + seq)
    q, k, v = (rng.standard_normal(s, dtype=np.float32)
               for s in ((nq, d), (nkv, seq, d), (nkv, seq, d)))
    kd = torch.zeros(k.size + shift, device=DEV)[shift:]
    kd.copy_(dev(k).flatten())
    y, probs = torch.zeros(nq * d, device=DEV), torch.full((seq,), 7.0, device=DEV)
    myos.gqa_attn_f32(y, dev(q), kd, dev(v), probs, nq, nkv, d, seq, causal)
    n = seq if causal is None else causal + 1
    yr, pr = _gqa64(q, k, v, n)
    # a score is a dot of d products within gamma_d |q||k| (< 2 gamma_d d for
    # unit normals at these sizes) and moves its probability by that factor
    tol = 8 * d * np.sqrt(d) * 2.0 ** -24 + seq * 2.0 ** -24
    assert np.linalg.norm(host(y) - yr.ravel()) <= tol * np.linalg.norm(yr)
    assert np.linalg.norm(host(probs)[:n] - pr) <= tol * np.linalg.norm(pr)
    assert not host(probs)[n:].any()


def test_gqa_chunks_non_finite():
    # the row-wide definition, over 1100 positions (several chunks): a NaN score
    # takes its head; a chunk of -inf scores weighs nothing; all -inf is NaN; an
    # infinite value under a zero probability is NaN in its column alone
    nq, d, seq = 2, 64, 1100
    rng = np.random.default_rng(0)
    q, k, v = (rng.standard_normal(s, dtype=np.float32) for s in ((nq, d), (nq, seq, d), (nq, seq, d)))
    q[:, 0], k[:, :, 0] = 1.0, 0.0
    cases = []
    for name in ("nan", "chunk", "all", "value"):
        k2, v2 = k.copy(), v.copy()
        if name == "nan":
            k2[0, 40, 3] = np.nan
        elif name == "chunk":
            k2[0, 0:64, 0] = -np.inf
        elif name == "all":
            k2[0, :, 0] = -np.inf
        else:
            k2[0, 64:128, 0] = -2000.0  # e^-250 next to the row's maximum: zero
            v2[0, 70, 5] = np.inf
        y, probs = torch.zeros(nq * d, device=DEV), torch.zeros(seq, device=DEV)
        myos.gqa_attn_f32(y, dev(q), dev(k2), dev(v2), probs, nq, nq, d, seq)
        got = host(y).reshape(nq, d)
        with np.errstate(all="ignore"):
            s = (np.einsum("hd,htd->ht", q, k2) / np.float32(np.sqrt(d))).astype(np.float32)
            e = np.exp(s - np.nanmax(s, 1, keepdims=True), dtype=np.float32)
            p = e / e.sum(1, keepdims=True)
            ref = (p[:, :, None].astype(np.float64) * v2).sum(1)
        assert np.array_equal(np.isnan(got), np.isnan(ref)), name
        ok = ~np.isnan(ref)
        assert np.allclose(got[ok], ref[ok], rtol=1e-4, atol=1e-5), name


# the table rides in the launch's arguments up to 128 pairs and is copied to the
# device beyond; both must give the oracle's bits' values
@pytest.mark.parametrize("d,heads", [(2, 3), (128, 12), (254, 2), (256, 2), (258, 2), (512, 1)])
def test_rope_table_sizes(d, heads):
    x0 = np.random.default_rng(d).standard_normal(heads * d, dtype=np.float32)
    _, ref = oracle.rope_f32_inplace(x0, 77, d, THETA)
    x = dev(x0)
    myos.rope_f32_inplace(x, 77, d, THETA)
    # the products may contract into fmas: one rounding of each term apart
    assert np.max(np.abs(host(x) - ref)) <= 4 * 2.0 ** -24 * np.max(np.abs(x0))


def test_scratch_streams_and_threads():
    # calls that need scratch, from threads on their own streams and on one
    # shared stream, growing and shrinking: each result is the one a lone call
    # gives, bit for bit
    import threading
    rng = np.random.default_rng(5)
    shapes = [(37, 640, 1536), (200, 1536, 640), (5, 70, 45)]
    ins = [(dev(rand_w(rng, m, k), torch.int16),
            dev(rng.standard_normal((b, k), dtype=np.float32))) for b, m, k in shapes]

    def call(i):
        b, m, k = shapes[i]
        y = torch.zeros((b, m), device=DEV)
        myos.gemm_bf16(y, *ins[i], b, m, k)
        return y
    want = [host(call(i)) for i in range(3)]
    shared = torch.cuda.Stream()
    torch.cuda.synchronize()
    bad = []

    def work(t):
        s = shared if t % 2 else torch.cuda.Stream()
        with torch.cuda.stream(s):
            ys = [(i, call(i)) for _ in range(10) for i in range(3)]
            s.synchronize()
        bad.extend(i for i, y in ys if not np.array_equal(host(y), want[i]))
    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


# gemm_bf16 over the direct-to-LDS tiles: each tile whole and, but for 128 x 160, which
# the plan never splits, in K splits (test_abi.py checks that against the plan), with
# row and column remainders, N % 4 != 0 (scalar stores), one row, one K step, 8 or more
# M tiles (XCD runs)
TILE_SHAPES = [
    (2, 3515, 320), (34, 386, 1600), (66, 4269, 2112), (442, 458, 1664), (3, 671, 1536),
    (244, 637, 2304), (39, 6293, 2368), (985, 350, 128), (90, 1510, 1856), (205, 1465, 768),
    (140, 3545, 1536), (1012, 979, 384), (1, 3203, 2176), (757, 6394, 192), (21, 1535, 2176),
    (305, 67, 2176), (527, 3087, 256), (513, 1240, 1600), (596, 3666, 512), (78, 2018, 2240),
    (566, 5227, 64), (1207, 7514, 128), (2047, 8203, 448), (381, 37888, 192), (128, 20479, 320),
    (2048, 1536, 8960), (1, 1, 64),
    (130, 81, 1920), (195, 82, 2432), (266, 82, 3264), (131, 1383, 1984), (33, 453, 2688),
    (130, 10333, 64), (1035, 11363, 64), (390, 8565, 4224), (2047, 3584, 4096), (1, 9615, 4160),
    (1, 4909, 4672)]


@pytest.mark.parametrize("batch,m,k", TILE_SHAPES)
def test_gemm_tiles(batch, m, k):
    g = torch.Generator(device=DEV).manual_seed(batch + m + k)
    w = (torch.randn(m, k, generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    x = torch.randn(batch, k, generator=g, device=DEV)
    y = torch.full((batch, m), float("nan"), device=DEV)
    myos.gemm_bf16(y, w, x, batch, m, k)
    ref = torch.mm(x.double(), w.double().t().contiguous())
    mag = torch.mm(x.double().abs(), w.double().abs().t().contiguous())
    # hi + lo keeps x to 2^-17 |x|; any summation order is within gamma_k, and
    # MFMA accumulation may not round to nearest: 4 gamma_k
    bound = (2.0 ** -17 + 4 * k * 2.0 ** -24) * mag
    assert bool(((y.double() - ref).abs() <= bound).all())


# X off the 16-byte grid, and Y over X: the bits of the same call on aligned operands
# of their own, through both entry points, on a tile that splits X itself whole and
# in K splits, on one that reads planes of it, and on the single-stage kernel
@pytest.mark.parametrize("call", [myos.gemm_bf16, myos.gemm_bf16_noalloc])
@pytest.mark.parametrize("batch,m,k", [(37, 1536, 1536), (16, 256, 1536), (600, 4096, 512), (9, 70, 70)])
def test_gemm_x_in_any_place(batch, m, k, call):
    g = torch.Generator(device=DEV).manual_seed(batch + m)
    w = (torch.randn(m, k, generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    x = torch.randn(batch, k, generator=g, device=DEV)
    want = torch.full((batch, m), float("nan"), device=DEV)
    call(want, w, x, batch, m, k)
    for shift in (1, 2, 3):
        xs = torch.empty(batch * k + shift, device=DEV)[shift:]
        xs.copy_(x.flatten())
        y = torch.full((batch, m), float("nan"), device=DEV)
        call(y, w, xs, batch, m, k)
        assert torch.equal(y, want), shift
    # Y starts one row into X, and at X
    for first in (0, k):
        room = torch.zeros(batch * max(m, k) + k, device=DEV)
        room[:batch * k] = x.flatten()
        call(room[first:first + batch * m], w, room[:batch * k], batch, m, k)
        assert torch.equal(room[first:first + batch * m].view(batch, m), want), first


# The outputs that meet an infinity, a NaN or an activation beyond bf16's range, in the
# first and last rows and columns, against the reference's chain: by the tile kernel's
# two epilogues (16 x 64, 128 x 128; 128 x 384, 256 x 256), by both reductions of K
# splits (N % 4 == 0 and not; 32 x 64 and 256 x 256), and by the pass after the
# single-stage kernel
@pytest.mark.parametrize("batch,m,k", [(442, 458, 1664), (566, 5227, 64), (1207, 7514, 128), (1035, 11363, 64),
                                       (33, 164, 3712), (33, 169, 3712), (2047, 3584, 4096), (390, 8565, 4224),
                                       (130, 71, 100)])
def test_gemm_non_finite(batch, m, k):
    rng = np.random.default_rng(batch + m + k)
    w = rand_w(rng, m, k)
    x = rng.standard_normal((batch, k), dtype=np.float32)
    clean_w, clean_x = dev(w, torch.int16).view(torch.bfloat16), dev(x)
    w[m - 1, 0], w[m // 2, k - 1], w[0, 5] = 0x7F80, 0x7FC0, 0xFF80  # inf, NaN, -inf
    x[::2, 0] = 2.0  # no lo part: the infinite weight meets a zero there
    x[1, 5] = 0.0    # inf times zero: the chain's NaN
    x[batch - 1, 3], x[0, k - 1] = np.inf, 3.4e38
    y = torch.full((batch, m), 7.0, device=DEV)
    myos.gemm_bf16(y, dev(w, torch.int16), dev(x), batch, m, k)
    got = host(y)
    rows, cols = [0, batch - 1], [0, m // 2, m - 1]
    with np.errstate(all="ignore"):
        want_r = oracle.gemm_bf16(w, x[rows], 2, m, k, threads=8)
        want_c = oracle.gemm_bf16(w[cols], x, batch, 3, k, threads=8)
    assert np.array_equal(got[rows], want_r, equal_nan=True)
    assert np.array_equal(got[:, cols], want_c, equal_nan=True)
    assert np.isinf(want_c[:, 2]).sum() > batch // 3 and np.isfinite(want_r[0]).sum() > m - 4
    # the others: the finite product, with x[:, 0] as the call had it
    clean_x[::2, 0], clean_x[1, 5] = 2.0, 0.0
    ref = torch.mm(clean_x.double(), clean_w.double().t().contiguous())
    mag = torch.mm(clean_x.double().abs(), clean_w.double().abs().t().contiguous())
    bound = (2.0 ** -17 + 4 * k * 2.0 ** -24) * mag
    ok = ((y.double() - ref).abs() <= bound).cpu().numpy()
    ok[rows], ok[:, cols] = True, True
    assert ok.all()
