"""The cost models behind the automatic choice between the matmul paths (host logic, no device): what each rule says against
what was measured on either side of its line (us, HIP-graph replay, MI355X)."""
import ctypes as C

import pytest

from cut_amd import lib

FORMATS = {"Q8_0": lib.Q8_0, "Q4_0": lib.Q4_0, "Q4_K": lib.Q4_K, "Q6_K": lib.Q6_K}
SCRATCH = 1 << 28


class RowsLayout(C.Structure):
    _fields_ = [("t", C.c_uint32), ("nw", C.c_uint32), ("per", C.c_uint32), ("ksplit", C.c_uint32), ("cost", C.c_double)]


def cost(name, *args):
    so = lib.load()
    symbol, res, more = {"rows": ("_ZN6cuthip16rows_gemm_layoutEijjjim", RowsLayout, [C.c_size_t]),
                         "lds": ("_ZN6cuthip16lds_gemm_cost_usEijjji", C.c_double, []),
                         "dense": ("_ZN6cuthip13dense_cost_usEijjji", C.c_double, [])}[name]
    f = getattr(so, symbol)
    f.restype, f.argtypes = res, [C.c_int, C.c_uint32, C.c_uint32, C.c_uint32, C.c_int] + more
    r = f(*args)
    return r.cost if name == "rows" else r


@pytest.fixture
def rows_tile():
    so = lib.load()
    yield lambda v: lib.check(so.cuthip_set_tuning(b"rows_tile", v.encode()))
    lib.check(so.cuthip_set_tuning(b"rows_tile", None))


@pytest.mark.parametrize("fmt", list(FORMATS))
@pytest.mark.parametrize("a_f16", [0, 1])
def test_row_tile_layout_is_the_cheapest_of_its_model(rows_tile, fmt, a_f16):
    """No number of row tiles and panel width that can be forced costs less than the layout that is chosen, with scratch memory
    for a K split and without."""
    for M in (9, 48, 64, 96, 100, 128, 160, 300, 512, 1000, 2048):
        for N, K in ((512, 512), (1024, 4096), (2048, 2048), (2560, 2560), (5632, 2048), (4096, 14336), (14336, 4096)):
            for scratch in (0, SCRATCH):
                rows_tile("")
                chosen = cost("rows", FORMATS[fmt], M, K, N, a_f16, scratch)
                for tile in ("1,2", "2,2", "1,4", "2,4", "3,4", "4,4"):
                    rows_tile(tile)
                    assert chosen <= cost("rows", FORMATS[fmt], M, K, N, a_f16, scratch) + 1e-9, (M, N, K, scratch, tile)


# measured: (format, M, N, K, fp16 activations, row tiles, decoding through LDS); no scratch memory
LDS_LINE = [("Q4_K", 2048, 32000, 256, 1, 120, 60), ("Q6_K", 2048, 8192, 256, 0, 61, 29), ("Q8_0", 2048, 16384, 512, 1, 77, 54),
            ("Q4_0", 2048, 128256, 512, 0, 860, 552), ("Q8_0", 2048, 32000, 2048, 1, 414, 372), ("Q4_K", 4096, 3072, 768, 1, 44, 33),
            ("Q4_K", 96, 16384, 512, 0, 10, 15), ("Q4_K", 300, 2048, 2048, 1, 10, 32), ("Q8_0", 1024, 4096, 4096, 1, 49, 79),
            ("Q6_K", 128, 14336, 4096, 1, 38, 93), ("Q4_0", 4096, 5632, 2048, 0, 148, 164)]


@pytest.mark.parametrize("fmt,M,N,K,a_f16,rows,lds", LDS_LINE)
def test_line_between_row_tiles_and_decoding_through_lds(fmt, M, N, K, a_f16, rows, lds):
    f = FORMATS[fmt]
    row_tiles = cost("rows", f, M, K, N, a_f16, 0) + 0.12e-6 * M * N * (2 if a_f16 else 4)   # and the store of C
    assert (cost("lds", f, M, K, N, a_f16) < row_tiles) == (lds < rows)


# measured: (format, M, N, K, fp16 activations, row tiles, two passes); workspace at hand
DENSE_LINE = [("Q4_K", 640, 14336, 4096, 1, 112, 105), ("Q4_K", 768, 14336, 4096, 1, 116, 107), ("Q4_0", 832, 14336, 4096, 1, 131, 113),
              ("Q8_0", 576, 14336, 4096, 1, 123, 103), ("Q8_0", 512, 14336, 4096, 1, 95, 85), ("Q4_K", 1536, 4096, 4096, 1, 71, 62),
              ("Q4_K", 2048, 4096, 14336, 1, 274, 227), ("Q8_0", 2048, 28672, 4096, 1, 678, 430), ("Q8_0", 384, 14336, 4096, 1, 83, 103),
              ("Q4_K", 512, 14336, 4096, 1, 78, 85), ("Q4_K", 1024, 4096, 4096, 1, 45, 56), ("Q6_K", 350, 11008, 4096, 1, 77, 83),
              ("Q6_K", 512, 11008, 4096, 1, 92, 84), ("Q6_K", 512, 14336, 4096, 1, 98, 90), ("Q6_K", 2048, 2048, 2048, 0, 50, 44),
              ("Q6_K", 300, 11008, 4096, 0, 75, 88),   # (640 rows of it with fp16 activations: 135 in two passes before tiles of 256 x 192, now 93 either way)
              ("Q8_0", 2048, 1024, 4096, 0, 45, 47), ("Q6_K", 224, 32000, 2048, 0, 81, 119), ("Q4_K", 100, 14336, 4096, 1, 26, 66)]


@pytest.mark.parametrize("fmt,M,N,K,a_f16,rows,dense", DENSE_LINE)
def test_line_between_row_tiles_and_two_passes(fmt, M, N, K, a_f16, rows, dense):
    f = FORMATS[fmt]
    row_tiles = cost("rows", f, M, K, N, a_f16, SCRATCH) + 0.12e-6 * M * N * (2 if a_f16 else 4)
    assert (cost("dense", f, M, K, N, a_f16) < row_tiles) == (dense < rows)


@pytest.mark.parametrize("M,N,K", [(2048, 5120, 4096), (1024, 5120, 4096), (2048, 11008, 4096), (700, 5632, 2048)])
def test_tiles_without_the_32x32x16_kernel_are_not_chosen_for_it(M, N, K):
    """These shapes take tiles of 256 by 128, 160 or 192; a comparison of the two kernels compares them on a tile that both have."""
    both = ("256,224", "128,448", "256,256", "128,256")
    try:
        best = cost("dense", lib.Q4_K, M, K, N, 1)
        lib.set_tuning("dense_mfma16", "0")
        without = cost("dense", lib.Q4_K, M, K, N, 1)
        forced = []
        for tile in both:
            lib.set_tuning("dense_tile", tile)
            forced.append(cost("dense", lib.Q4_K, M, K, N, 1))
    finally:
        lib.set_tuning("dense_mfma16", None)
        lib.set_tuning("dense_tile", None)
    assert best < without == min(forced)


# measured: (rows, N, K, fp16 activations, scratch memory, 8-row GEMV, streaming matmul)
STREAM_LINE = [(8, 14336, 4096, 1, 1, 19.7, 16.9), (8, 14336, 4096, 0, 1, 19.4, 16.9), (8, 4096, 14336, 1, 1, 20.7, 18.7), (8, 5120, 5120, 1, 1, 18.7, 13.0),
               (5, 10240, 2048, 1, 0, 11.1, 10.0), (8, 3072, 11008, 1, 1, 19.9, 16.6), (8, 2560, 8192, 1, 1, 17.3, 11.8), (8, 20480, 1536, 1, 1, 16.6, 16.3),
               (8, 8192, 2560, 1, 1, 9.8, 10.7), (8, 8192, 2560, 0, 1, 11.7, 11.3), (5, 8192, 3072, 1, 0, 10.1, 11.5), (8, 8192, 4096, 1, 0, 13.4, 14.9),
               (6, 14336, 1536, 0, 1, 9.6, 10.2), (8, 16384, 1536, 1, 1, 9.6, 10.2), (8, 4096, 5120, 1, 1, 10.8, 11.3), (8, 4096, 5120, 0, 1, 12.8, 11.7),
               (8, 2048, 11008, 1, 1, 11.7, 12.3), (8, 2048, 11008, 0, 1, 12.1, 12.7), (8, 2048, 14336, 1, 1, 14.3, 13.2)]


@pytest.mark.parametrize("M,N,K,a_f16,scratch,gemv,stream", STREAM_LINE)
def test_line_between_the_8_row_gemv_and_the_streaming_matmul_on_q8_0(M, N, K, a_f16, scratch, gemv, stream):
    f = lib.load()._ZN6cuthip19stream_q8_preferredEjjjibm
    f.restype, f.argtypes = C.c_bool, [C.c_uint32, C.c_uint32, C.c_uint32, C.c_int, C.c_bool, C.c_size_t]
    assert f(M, K, N, a_f16, False, SCRATCH if scratch else 0) == (stream < gemv)


class SepRowsParams(C.Structure):
    _fields_ = ([(n, C.c_void_p) for n in ("A", "B", "S", "C", "partial")] + [("kind", C.c_int), ("op", C.c_int), ("D", C.c_void_p)] +
                [(n, C.c_uint32) for n in ("M", "K", "N", "strideA", "strideB", "strideC", "scaleStride")] + [("A16", C.c_void_p)] +
                [(n, C.c_uint32) for n in ("t", "nsplit", "per", "tiles", "passes")] + [("cost_us", C.c_double)])


# measured: (layout, rows, N, K, two passes, weights decoded as they are needed)
SEP_LINE = [("q8", 64, 256, 256, 12.9, 16.6), ("q8", 512, 512, 256, 14.5, 17.5), ("q4", 128, 96, 256, 13.5, 14.7), ("affine", 64, 512, 256, 13.3, 15.3),
            ("q8", 64, 512, 512, 14.5, 15.5), ("q8", 48, 512, 512, 14.0, 13.7), ("q8", 200, 1024, 512, 16.6, 16.2), ("affine", 500, 5120, 4096, 58.2, 55.1),
            ("q8", 64, 14336, 4096, 86, 34), ("q8", 256, 4096, 4096, 47, 32), ("q4", 512, 1024, 512, 18.4, 16.3)]


@pytest.mark.parametrize("layout,M,N,K,two,direct", SEP_LINE)
def test_line_between_two_passes_and_direct_decoding_on_the_separated_layout(layout, M, N, K, two, direct):
    so, q4 = lib.load(), layout != "q8"
    f = so._ZN6cuthip20sep_rows16_preferredERNS_13SepRowsParamsEbbm
    f.restype, f.argtypes = C.c_bool, [C.POINTER(SepRowsParams), C.c_bool, C.c_bool, C.c_size_t]
    p = SepRowsParams(M=M, K=K, N=N, strideA=K, strideB=N // 2 if q4 else N, strideC=N, scaleStride=N)
    room = so.cuthip_matmul_sep_workspace_bytes_for(lib.OP_MATMUL_Q4 if q4 else lib.OP_MATMUL_Q8, -1, M, K, N) - ((M * K * 2 + 255) & ~255)
    assert f(C.byref(p), q4, layout == "affine", room) == (direct < two)


# measured on resident fp16 weights: (rows, N, K, K split, us, one range, us)
SPLIT_LINE = [(1, 512, 512, "128,256,4", 8.8, "256,128", 10.1), (64, 512, 512, "128,256,4", 10.0, "256,128", 11.0), (64, 1024, 1024, "128,256,4", 12.2, "128,256", 16.4)]


@pytest.mark.parametrize("M,N,K,split,us,whole,more", SPLIT_LINE)
def test_small_problems_split_k(M, N, K, split, us, whole, more):
    try:
        chosen = cost("dense", lib.Q4_K, M, K, N, 1)
        forced = {}
        for tile in (split, whole):
            lib.set_tuning("dense_tile", tile)
            forced[tile] = cost("dense", lib.Q4_K, M, K, N, 1)
    finally:
        lib.set_tuning("dense_tile", None)
    assert chosen <= forced[split] < forced[whole]


# measured on resident fp16 weights: (rows, N, K, fp16 activations, tile whose panels lie in one XCD each, us, tile whose panels are cut, us)
CUT_LINE = [(719, 1632, 7552, 0, "128,256", 82, "256,128", 100), (790, 17768, 5888, 0, "256,160", 182, "128,256", 215),
            (677, 1624, 2176, 1, "128,256", 30, "256,128", 35)]


@pytest.mark.parametrize("M,N,K,a_f16,whole,us,cut,more", CUT_LINE)
def test_tiles_whose_panels_lie_in_one_xcd(M, N, K, a_f16, whole, us, cut, more):
    try:
        chosen = cost("dense", lib.Q4_K, M, K, N, a_f16)
        forced = {}
        for tile in (whole, cut):
            lib.set_tuning("dense_tile", tile)
            forced[tile] = cost("dense", lib.Q4_K, M, K, N, a_f16)
    finally:
        lib.set_tuning("dense_tile", None)
    assert chosen == forced[whole] < forced[cut]


# measured with fp16 rows of A off 16 bytes: (format, rows, N, K, scratch memory, row tiles and panel width, us, with the cut of the kernel that
# loads A straight to LDS, us)
OFF16 = [("Q4_K", 49, 14292, 8704, 1, (2, 4), 44.1, 57.4), ("Q4_K", 799, 1523, 6656, 1, (2, 4), 42.6, 49.0),
         ("Q4_K", 40, 13878, 3584, 1, (1, 4), 24.9, 28.2), ("Q6_K", 51, 6045, 7680, 0, (1, 2), 43.4, 54.5),
         ("Q6_K", 229, 1673, 10752, 0, (1, 2), 51.8, 64.6), ("Q6_K", 136, 2612, 6400, 0, (1, 2), 37.2, 45.4)]


@pytest.mark.parametrize("fmt,M,N,K,scratch,tile,us,other", OFF16)
def test_rows_off_16_bytes_have_a_layout_of_their_own(fmt, M, N, K, scratch, tile, us, other):
    """They run through registers: the estimate for A straight to LDS is not theirs."""
    f = getattr(lib.load(), "_ZN6cuthip22rows_gemm_layout_off16Eijjjim")
    f.restype, f.argtypes = RowsLayout, [C.c_int, C.c_uint32, C.c_uint32, C.c_uint32, C.c_int, C.c_size_t]
    room = SCRATCH if scratch else 0
    own = f(FORMATS[fmt], M, K, N, 1, room)
    assert (own.t, own.nw) == tile and us < other
    assert own.cost >= cost("rows", FORMATS[fmt], M, K, N, 1, room)
    for same in (lib.Q8_0, lib.Q4_0):   # formats without that kernel: one layout
        assert f(same, M, K, N, 1, room).cost == cost("rows", same, M, K, N, 1, room)


# measured with fp16 rows of A on 16 bytes: (rows, N, K, scratch memory, tile chosen, us, other tile, us)
Q6_K_TILE = [(53, 5788, 12544, 0, "1,2", 56.0, "2,2", 63.7), (229, 1673, 10752, 0, "1,2", 46.4, "2,2", 51.9), (64, 5512, 5376, 0, "1,2", 28.7, "2,2", 32.3),
             (340, 1046, 1792, 1, "1,2", 14.1, "2,2", 16.0), (169, 1387, 2048, 1, "1,2", 13.6, "2,2", 15.1), (317, 929, 4096, 1, "2,2", 18.9, "2,4", 21.4),
             (481, 1787, 3840, 1, "2,2", 23.4, "4,4", 32.0)]


@pytest.mark.parametrize("M,N,K,scratch,tile,us,other,more", Q6_K_TILE)
def test_tiles_of_q6_k_that_go_straight_to_lds_beside_the_others(rows_tile, M, N, K, scratch, tile, us, other, more):
    room = SCRATCH if scratch else 0
    chosen = cost("rows", lib.Q6_K, M, K, N, 1, room)
    rows_tile(tile)
    own = cost("rows", lib.Q6_K, M, K, N, 1, room)
    rows_tile(other)
    assert chosen == own < cost("rows", lib.Q6_K, M, K, N, 1, room) and us < more


class AttnRoute(C.Structure):
    _fields_ = [("heads", C.c_uint32), ("nsplit", C.c_uint32)]


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("n_kv", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 16, 20, 32, 40])
def test_attention_of_four_heads_a_workgroup_has_one_on_every_cu(head_dim, n_kv):
    """The workgroups of a (KV head, split) share an XCD of 32 CUs: counted over the whole chip, three groups of four heads put 33 on some
    of them (48 / 4 heads at 32,000 positions 43.0 us, with 30 on each 32.2)."""
    f = lib.load()._ZN6cuthip10attn_routeEjjjj
    f.restype, f.argtypes = AttnRoute, [C.c_uint32] * 4
    taken = 0
    for n_rep in range(1, 41):
        for positions in (1, 64, 700, 2500, 6000, 12000, 20000, 32000, 65536):
            r, chunks = f(head_dim, n_kv * n_rep, n_kv, positions), (positions + 63) // 64
            assert 1 <= r.nsplit <= min(chunks, 1024)
            if r.heads == 4 and r.nsplit > 1:
                taken += 1
                assert (r.nsplit * n_kv + 7) // 8 * ((n_rep + 3) // 4) <= 32, (n_rep, positions, r.nsplit)
    assert taken
