"""GPU parity of the separated-layout (reference tensor layout) quantized
matmul through the C ABI against the oracle's restatement of the harness loops
(tests/harness/OpRegistry.h:2043-2051, 2107-2112 of the reference), including
the reference's own known-answer cases and the affine Q4 path fed by the
oracle's requantizeQ4KToAffine.  Tolerance 1e-3 normwise (fp32 throughout;
observed ~1e-6), known answers to the reference's own tolerances."""
import numpy as np
import pytest

import oracle
from helpers import normwise_rel_err

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from cut_amd import lib, ops as _ops
    lib.check(lib.load().cuthip_init(0))
    return _ops


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def run(ops, A, B, S, N, **kw):
    out = ops.matmul_sep(dev(A), dev(B), dev(S.astype(np.float16)), N, **kw)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def test_reference_known_answers(ops):
    # q8_simple (OpRegistry.h:1995-2010): A = 1, B[k,0] = 1, B[k,1] = 2, scales 1 -> [32, 64]
    A = np.ones((1, 32), np.float32)
    B = np.stack([np.ones(32, np.int8), np.full(32, 2, np.int8)], axis=1)
    np.testing.assert_allclose(run(ops, A, B, np.ones((1, 2), np.float32), 2), [[32, 64]], atol=1e-3)
    # q8_withscales (:2012-2026): K = 64, B = 4, scales [[0.5, 2], [1, 0.25]] -> [192, 288]
    A = np.ones((1, 64), np.float32)
    B = np.full((64, 2), 4, np.int8)
    np.testing.assert_allclose(run(ops, A, B, np.array([[0.5, 2], [1, 0.25]], np.float32), 2), [[192, 288]], atol=1.0)
    # q4: nibbles 9 / 10 (values 1 / 2) -> [32, 64]; nibble 12 with the same scales -> [192, 288]
    A = np.ones((1, 32), np.float32)
    Bp = np.full((32, 1), 9 | (10 << 4), np.uint8)
    np.testing.assert_allclose(run(ops, A, Bp, np.ones((1, 2), np.float32), 2, q4=True), [[32, 64]], atol=1e-3)
    A = np.ones((1, 64), np.float32)
    Bp = np.full((64, 1), 12 | (12 << 4), np.uint8)
    np.testing.assert_allclose(run(ops, A, Bp, np.array([[0.5, 2], [1, 0.25]], np.float32), 2, q4=True), [[192, 288]], atol=1.0)


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 9])
@pytest.mark.parametrize("K,N", [(256, 1024), (4096, 1088), (96, 50)])
def test_q8_against_oracle(ops, M, K, N):
    rng = np.random.default_rng(M * K + N)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.integers(-127, 128, (K, N)).astype(np.int8)
    S = rng.uniform(0.001, 0.02, (K // 32, N)).astype(np.float16).astype(np.float32)
    want = oracle.matmul_sep_q8(A, B, S, f64=True)
    assert normwise_rel_err(run(ops, A, B, S, N), want) < 2e-6


@pytest.mark.parametrize("affine", [False, True])
@pytest.mark.parametrize("M", [1, 4, 6])
@pytest.mark.parametrize("K,N", [(256, 2048), (4096, 1056), (64, 34)])
def test_q4_against_oracle(ops, affine, M, K, N):
    rng = np.random.default_rng(M * K + N + affine)
    A = rng.standard_normal((M, K)).astype(np.float32)
    Bp = rng.integers(0, 256, (K, N // 2)).astype(np.uint8)
    S = rng.uniform(0.001, 0.02, ((2 if affine else 1) * (K // 32), N)).astype(np.float16).astype(np.float32)
    if affine:
        S[K // 32:] = rng.uniform(-0.1, 0.1, (K // 32, N)).astype(np.float16).astype(np.float32)
    want = oracle.matmul_sep_q4(A, Bp, S, affine=affine).astype(np.float64)   # the harness loop sums in fp32
    assert normwise_rel_err(run(ops, A, Bp, S, N, q4=True, affine=affine), want) < 2e-5


@pytest.mark.parametrize("M", [1, 7, 31])
@pytest.mark.parametrize("K,N", [(128, 1040), (160, 16), (4096, 260), (4128, 2064), (14336, 272), (4128, 1030), (16416, 64)])
def test_row_passes_and_reduce_edges(ops, M, K, N):
    """Rows of A in one, two and eight passes (the last one short), column tiles and K ranges whose product is no multiple
    of eight, 1, 2, 32, 33, 112 and 129 ranges in the reduce, rows that allow no vector accesses there, and the residual
    add; fp32 sums in any order, as above."""
    rng = np.random.default_rng(M * K + N)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.integers(-127, 128, (K, N)).astype(np.int8)
    S = rng.uniform(0.001, 0.02, (K // 32, N)).astype(np.float16).astype(np.float32)
    want = oracle.matmul_sep_q8(A, B, S, f64=True)
    assert normwise_rel_err(run(ops, A, B, S, N), want) < 2e-6
    D = dev(rng.standard_normal((M, N)).astype(np.float32))
    got = ops.matmul_sep(dev(A), dev(B), dev(S.astype(np.float16)), N, out=torch.full((M, N), 7.0, device="cuda"), binary="add", d=D)
    assert normwise_rel_err((got - D).cpu().numpy(), want) < 4e-6


@pytest.mark.parametrize("kind", ["q8", "q4", "affine"])
@pytest.mark.parametrize("M,K,N", [(3, 32, 8), (16, 160, 264), (17, 4128, 520), (31, 4096, 256), (33, 96, 136), (70, 2080, 248), (4, 2048, 20)])
def test_rows_on_the_matrix_cores(ops, kind, M, K, N):
    """Streaming variants from three rows on: lanes and sides of a column tile without columns, waves and ranges without
    blocks, short last row tiles and passes, one launch through the operators and several ranges; columns that are no
    multiple of eight stay on the vector kernel.  Exact products and fp32 sums: the bounds of the vector kernel."""
    rng = np.random.default_rng(M * K + N)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.integers(-127, 128, (K, N)).astype(np.int8) if kind == "q8" else rng.integers(0, 256, (K, N // 2)).astype(np.uint8)
    S = rng.uniform(0.001, 0.02, ((2 if kind == "affine" else 1) * (K // 32), N)).astype(np.float16).astype(np.float32)
    if kind == "affine":
        S[K // 32:] = rng.uniform(-0.1, 0.1, (K // 32, N)).astype(np.float16).astype(np.float32)
    how = dict(q4=kind != "q8", affine=kind == "affine", variant=1)
    if kind == "q8":
        w = B * S.astype(np.float64).repeat(32, 0)
    else:
        q = np.stack((B & 15, B >> 4), -1).reshape(K, N).astype(np.float64) - 8
        w = q * S[:K // 32].astype(np.float64).repeat(32, 0)
        if kind == "affine":
            w += S[K // 32:].astype(np.float64).repeat(32, 0)
    want = A.astype(np.float64) @ w
    assert normwise_rel_err(run(ops, A, B, S, N, **how), want) < 2e-6
    D = rng.standard_normal((M, N)).astype(np.float32)
    got = ops.matmul_sep(dev(A), dev(B), dev(S.astype(np.float16)), N, binary="add", d=dev(D), **how).cpu().numpy()
    assert normwise_rel_err(got - D, want) < 4e-6


@pytest.mark.parametrize("ks", ["", "1", "3"])
@pytest.mark.parametrize("kind", ["q8", "q4", "affine"])
@pytest.mark.parametrize("M,K,N", [(32, 128, 8), (33, 384, 264), (64, 640, 136), (65, 1152, 520), (130, 256, 1032), (32, 512, 8), (33, 512, 264), (130, 640, 1032), (200, 512, 776),
                                   (300, 512, 2312)])   # (three and nine column tiles of four and five passes: shared out over the XCDs)
def test_rows_on_rounded_operands(ops, kind, ks, M, K, N):
    """The default from 32 rows: two, three and four row tiles in one pass and several, sides and lanes without columns, waves
    without blocks, one range and several.  Against the float64 product of the operands rounded to fp16 once each: fp32 sums."""
    from cut_amd import lib
    rng = np.random.default_rng(M * K + N)
    A = rng.standard_normal((M, K)).astype(np.float32)
    S = rng.uniform(0.001, 0.02, ((2 if kind == "affine" else 1) * (K // 32), N)).astype(np.float16).astype(np.float64)
    if kind == "affine":
        S[K // 32:] = rng.uniform(-0.1, 0.1, (K // 32, N)).astype(np.float16)
    scale = S[:K // 32].repeat(32, 0)
    if kind == "q8":
        B = rng.integers(-128, 128, (K, N)).astype(np.int8)
        w = B * scale
    else:
        B = rng.integers(0, 256, (K, N // 2)).astype(np.uint8)
        w = (np.stack((B & 15, B >> 4), -1).reshape(K, N).astype(np.float64) - 8) * scale
        if kind == "affine":
            w += S[K // 32:].repeat(32, 0)
    want = A.astype(np.float16).astype(np.float64) @ w.astype(np.float16).astype(np.float64)
    D = rng.standard_normal((M, N)).astype(np.float32)
    how = dict(q4=kind != "q8", affine=kind == "affine")
    dll = lib.load()
    lib.check(dll.cuthip_set_tuning(b"gemm_ksplit", ks.encode()))
    try:
        got = run(ops, A, B, S, N, **how)
        added = ops.matmul_sep(dev(A), dev(B), dev(S.astype(np.float16)), N, binary="add", d=dev(D), **how).cpu().numpy()
    finally:
        lib.check(dll.cuthip_set_tuning(b"gemm_ksplit", b""))
    assert normwise_rel_err(got, want) < 2e-6
    assert normwise_rel_err(added - D, want) < 4e-6


@pytest.mark.parametrize("kind", ["q8", "q4", "affine"])
@pytest.mark.parametrize("N", [1040, 1036])
@pytest.mark.parametrize("view", ["offset", "pitch"])
def test_many_rows_that_are_not_aligned(ops, kind, N, view):
    """Rows of A off the 16 bytes that the fp16 route from 32 rows on reads: exact products in the workspace of that route, which is
    smaller than the vector kernel's partial sums of all rows (K / 128 x M x N x 4 bytes).  Columns in multiples of eight
    take the matrix cores, others the vector kernel, some rows at a time.  Bounds as below 32 rows."""
    M, K = 512, 4096
    g = torch.Generator("cuda").manual_seed(N)
    buf = torch.randn((M, K + 8), generator=g, device="cuda")
    A = buf[:, 1:K + 1] if view == "offset" else torch.randn((M, K + 1), generator=g, device="cuda")[:, :K]
    q4, affine = kind != "q8", kind == "affine"
    B = torch.randint(0, 256, (K, N // 2 if q4 else N), generator=g, device="cuda", dtype=torch.uint8)
    S = (torch.rand(((2 if affine else 1) * (K // 32), N), generator=g, device="cuda") * 0.02 + 0.001).half()
    q = torch.stack((B & 15, B >> 4), -1).reshape(K, N).double() - 8 if q4 else B.view(torch.int8).double()
    w = q * S[:K // 32].double().repeat_interleave(32, 0)
    if affine:
        w += S[K // 32:].double().repeat_interleave(32, 0)
    want = (A.double() @ w).cpu().numpy()
    B = B if q4 else B.view(torch.int8)
    assert normwise_rel_err(ops.matmul_sep(A, B, S, N, q4=q4, affine=affine).cpu().numpy(), want) < 2e-6
    D = torch.randn((M, N), generator=g, device="cuda")
    got = ops.matmul_sep(A, B, S, N, q4=q4, affine=affine, binary="add", d=D)
    assert normwise_rel_err((got - D).cpu().numpy(), want) < 4e-6


def test_rows_on_the_matrix_cores_extreme_activations(ops):
    """Magnitudes from 1e-30 to 1e30 in one row tile, and an infinity: it reaches its own row alone, as infinity where the
    weight is not zero."""
    M, K, N = 5, 64, 32
    rng = np.random.default_rng(5)
    A = (rng.standard_normal((M, K)) * np.array([1e-30, 1e-8, 1.0, 1e8, 1e30])[:, None]).astype(np.float32)
    B = rng.integers(1, 128, (K, N)).astype(np.int8)
    B[9, 4:7] = (0, -3, 5)
    S = np.full((K // 32, N), 0.0078125, np.float32)
    want = A.astype(np.float64) @ (B * S.astype(np.float64).repeat(32, 0))
    got = run(ops, A, B, S, N)
    for m in range(M):
        assert normwise_rel_err(got[m], want[m]) < 2e-6
    A[2, 9] = np.inf
    inf = run(ops, A, B, S, N)
    np.testing.assert_array_equal(np.delete(inf, 2, 0), np.delete(got, 2, 0))
    with np.errstate(invalid="ignore"):
        np.testing.assert_array_equal(inf[2], np.where(B[9] == 0, np.nan, np.inf * B[9].astype(np.float32)))


@pytest.mark.parametrize("kind", ["q8", "q4", "affine"])
@pytest.mark.parametrize("M", [6, 20])
def test_rows_on_the_matrix_cores_small_activations(ops, kind, M):
    """Down to the smallest subnormal numbers, beside ordinary rows: 24 bits of every activation, as the fp32 multiply-adds have
    them.  (Parts of such numbers lie below the smallest bf16; scales of 64 keep the results normal.)  One block for a wave and
    several.  Then rows whose magnitude changes inside the range of a wave, from one to which the waves scale up to one that has no
    room for that and back: what they hold is scaled with it."""
    rng = np.random.default_rng(M)
    N, q4, affine = 264, kind != "q8", kind == "affine"
    size = np.array([1.0, 1e-34, 1e-36, 2e-38, 1e-40, 1e-43])[np.arange(M) % 6]
    for K in (96, 4160):
        S = np.full(((2 if affine else 1) * (K // 32), N), 64.0, np.float32)
        if q4:
            B = rng.integers(0, 256, (K, N // 2)).astype(np.uint8)
            q = np.stack((B & 15, B >> 4), -1).reshape(K, N).astype(np.float64) - 8
        else:
            B = rng.integers(-127, 128, (K, N)).astype(np.int8)
            q = B.astype(np.float64)
        w = q * 64 + (64 if affine else 0)
        A = (rng.standard_normal((M, K)) * size[:, None]).astype(np.float32)
        for rows in (slice(None), slice(1, None, 6), slice(3, None, 6)):   # and rows of one size by themselves
            a = np.ascontiguousarray(np.repeat(A[rows], 3, 0)[:M])
            want, got = a.astype(np.float64) @ w, run(ops, a, B, S, N, q4=q4, affine=affine, variant=1)
            for m in range(len(a)):
                assert normwise_rel_err(got[m], want[m]) < 2e-6, (K, m, np.abs(a[m]).max())
        for sizes in ((1e-36, 1.0, 1e25), (1e25, 1e-36, 1.0), (1e25, 1.0, 1e-36), (1e-36, 1e25, 1e-36)):
            a = (A / size[:, None] * np.repeat(np.resize(sizes, K // 32), 32)[None]).astype(np.float32)
            want, got = a.astype(np.float64) @ w, run(ops, a, B, S, N, q4=q4, affine=affine, variant=1)
            assert normwise_rel_err(got, want) < 2e-6, (K, sizes)


@pytest.mark.parametrize("kind", ["q8", "q4", "affine"])
@pytest.mark.parametrize("M", [6, 20])
@pytest.mark.parametrize("beside", [1e25, np.inf, np.nan])
def test_rows_on_the_matrix_cores_small_rows_beside_large_ones(ops, kind, M, beside):
    """A row of a tile that has no room above it (large numbers, an infinity, a NaN; in the first block of a wave or in a later one)
    takes nothing from the rows beside it: 24 bits of their activations however small they are, as in the test before this one."""
    rng = np.random.default_rng(M)
    K, N, q4, affine = 4160, 264, kind != "q8", kind == "affine"
    S = np.full(((2 if affine else 1) * (K // 32), N), 64.0, np.float32)
    if q4:
        B = rng.integers(0, 256, (K, N // 2)).astype(np.uint8)
        q = np.stack((B & 15, B >> 4), -1).reshape(K, N).astype(np.float64) - 8
    else:
        B = rng.integers(-127, 128, (K, N)).astype(np.int8)
        q = B.astype(np.float64)
    w = q * 64 + (64 if affine else 0)
    size = np.array([1e-34, 1.0, 1e-36, 2e-38, 1e-40])[np.arange(M) % 5]
    for row in (0, M - 1):
        for k in (5, 2600):
            a = (rng.standard_normal((M, K)) * size[:, None]).astype(np.float32)
            a[row, k] = beside
            want, got = a.astype(np.float64) @ w, run(ops, a, B, S, N, q4=q4, affine=affine, variant=1)
            for m in range(M):
                if m != row or np.isfinite(beside):
                    assert normwise_rel_err(got[m], want[m]) < 2e-6, (row, k, m)
                else:
                    assert not np.isfinite(got[m]).any()


def test_affine_layout_from_q4k_requantizer(ops):
    """Q4_K blocks -> requantizeQ4KToAffine (oracle restatement of llama.cpp:573-619) -> separated affine matmul
    agrees with the matmul over the decoded affine weights."""
    N, K = 64, 512
    rng = np.random.default_rng(3)
    raw = oracle.quantize(oracle.Q4_K, (rng.standard_normal(N * K) * 0.02).astype(np.float32))
    packedT, scalesT = oracle.requantize_q4k_to_affine(raw, N, K)
    Wf = oracle.decode_affine_q4(packedT, scalesT, N, K)          # [N, K]
    A = rng.standard_normal((2, K)).astype(np.float32)
    want = A.astype(np.float64) @ Wf.astype(np.float64).T
    S = oracle.f16_to_f32_array(np.asarray(scalesT).reshape(-1)).reshape(2 * K // 32, N)
    got = run(ops, A, np.asarray(packedT).reshape(K, N // 2), S, N, q4=True, affine=True)
    assert normwise_rel_err(got, want) < 5e-6


def test_fused_epilogues_and_errors(ops):
    from cut_amd import lib
    rng = np.random.default_rng(9)
    M, K, N = 3, 128, 96
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.integers(-127, 128, (K, N)).astype(np.int8)
    S = rng.uniform(0.001, 0.02, (K // 32, N)).astype(np.float16).astype(np.float32)
    base = run(ops, A, B, S, N)
    D = rng.standard_normal((M, N)).astype(np.float32)
    got = ops.matmul_sep(dev(A), dev(B), dev(S.astype(np.float16)), N, binary="add", d=dev(D))
    torch.cuda.synchronize()
    np.testing.assert_allclose(got.cpu().numpy(), base + D, rtol=1e-6, atol=1e-6)
    got = ops.matmul_sep(dev(A), dev(B), dev(S.astype(np.float16)), N, unary="relu")
    torch.cuda.synchronize()
    np.testing.assert_array_equal(got.cpu().numpy(), np.maximum(base, 0))
    with pytest.raises(lib.CutHipError):
        ops.matmul_sep(dev(A[:, :100].copy()), dev(B[:100]), dev(S.astype(np.float16)[:3]), N)   # K not a multiple of 32


# ---- prefill route: from 32 rows on (K a multiple of 128) the tensors are dequantized to fp16 [N][K] and multiplied by
# the dense GEMM; fp16 weights and activations, fp32 accumulation: the tolerance of the native prefill path -------------

@pytest.mark.parametrize("M,K,N", [(32, 128, 64), (70, 256, 200), (300, 1024, 520), (1030, 512, 264)])
def test_prefill_route_q8(ops, M, K, N):
    rng = np.random.default_rng(M + K + N)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.integers(-127, 128, (K, N)).astype(np.int8)
    S = rng.uniform(0.001, 0.02, (K // 32, N)).astype(np.float16).astype(np.float32)
    want = oracle.matmul_sep_q8(A, B, S, f64=True)
    assert normwise_rel_err(run(ops, A, B, S, N), want) < 1e-3
    D = rng.standard_normal((M, N)).astype(np.float32)
    got = ops.matmul_sep(dev(A), dev(B), dev(S.astype(np.float16)), N, binary="add", d=dev(D))   # fused epilogue: own GEMM
    torch.cuda.synchronize()
    assert normwise_rel_err(got.cpu().numpy() - D, want) < 1e-3


def test_prefill_route_rounds_activations_to_fp16(ops):
    """The contract of the prefill route in cut_hip.h: fp32 activations are rounded to fp16 once.  Large magnitudes
    inside the fp16 range keep the 1e-3 normwise bound; beyond 65504 the result is not finite there, while the GEMV
    variant (reference index 1) computes in fp32 and stays within 1e-5."""
    M, K, N = 64, 512, 136
    rng = np.random.default_rng(77)
    A = (rng.standard_normal((M, K)) * 1.0e3).astype(np.float32)
    B = rng.integers(-127, 128, (K, N)).astype(np.int8)
    S = rng.uniform(0.001, 0.02, (K // 32, N)).astype(np.float16).astype(np.float32)
    want = oracle.matmul_sep_q8(A, B, S, f64=True)
    assert normwise_rel_err(run(ops, A, B, S, N), want) < 1e-3
    A[3, 17] = 1.0e5
    want = oracle.matmul_sep_q8(A, B, S, f64=True)
    assert not np.isfinite(run(ops, A, B, S, N)[3]).all()
    assert normwise_rel_err(run(ops, A, B, S, N, variant=1), want) < 1e-5


@pytest.mark.parametrize("affine", [False, True])
@pytest.mark.parametrize("M,K,N", [(32, 128, 66), (300, 1024, 520)])
def test_prefill_route_q4(ops, affine, M, K, N):
    rng = np.random.default_rng(M + K + N + affine)
    A = rng.standard_normal((M, K)).astype(np.float32)
    Bp = rng.integers(0, 256, (K, N // 2)).astype(np.uint8)
    S = rng.uniform(0.001, 0.02, ((2 if affine else 1) * (K // 32), N)).astype(np.float16).astype(np.float32)
    if affine:
        S[K // 32:] = rng.uniform(-0.1, 0.1, (K // 32, N)).astype(np.float16).astype(np.float32)
    want = oracle.matmul_sep_q4(A[:8], Bp, S, affine=affine).astype(np.float64)   # the CPU loop on the first rows
    got = run(ops, A, Bp, S, N, q4=True, affine=affine)
    assert normwise_rel_err(got[:8], want) < 1e-3
    # rows are independent: the GEMV route on a few rows gives what the prefill route gave for them
    few = run(ops, A[8:12], Bp, S, N, q4=True, affine=affine)
    assert normwise_rel_err(got[8:12], few) < 1e-3


def test_prefill_route_after_device_preparation(ops):
    """GGUF Q8_0 blocks -> cuthip_prepare_sep -> separated matmul at prefill size, against the native-block path."""
    from helpers import quantized_weights
    M, K, N = 256, 512, 384
    blocks = quantized_weights(oracle.Q8_0, N, K, seed=9)
    B, S = ops.prepare_sep(dev(blocks), "Q8_0", N, K)
    A = np.random.default_rng(10).standard_normal((M, K)).astype(np.float32)
    got = ops.matmul_sep(dev(A), B, S, N)
    torch.cuda.synchronize()
    want = oracle.matmul_gguf(oracle.Q8_0, blocks, A, N, f64=True)
    assert normwise_rel_err(got.cpu().numpy(), want) < 1e-3


@pytest.mark.parametrize("M", [1, 2, 4, 5])
def test_more_k_ranges_than_a_grid_dimension(ops, M):
    """65,537 ranges of K: one pass of rows in a grid of one dimension as several are.  Whole numbers, so that every sum is exact."""
    K, N = 65537 * 128, 16
    g = torch.Generator("cuda").manual_seed(M)
    b = torch.randint(-2, 3, (K, N), device="cuda", dtype=torch.int8, generator=g)
    a = torch.randint(-1, 2, (M, K), device="cuda", generator=g).float()
    scales = torch.ones((K // 32, N), device="cuda", dtype=torch.float16)
    want = torch.zeros((M, N), device="cuda", dtype=torch.float64)
    for k in range(0, K, 1 << 20):
        want += a[:, k:k + (1 << 20)].double() @ b[k:k + (1 << 20)].double()
    assert torch.equal(ops.matmul_sep(a, b, scales, N).double(), want)
