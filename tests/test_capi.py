"""The C-ABI library: loads without a GPU, exports every symbol include/mxq.h
declares, and rejects bad arguments before any HIP call."""
import ctypes as C
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    from machx_inference_engine_amd import _lib
    return _lib.load(), _lib.parse_header()


def test_every_declared_symbol_is_exported(lib):
    l, protos = lib
    assert len(protos) >= 40
    raw = C.CDLL(os.path.join(ROOT, "machx_inference_engine_amd", "libmxq.so"))
    for name in protos:
        assert hasattr(raw, name), name


def test_status_strings_and_version(lib):
    l, _ = lib
    assert l.mx_version() >= 100
    assert l.mx_status_string(0) == b"ok"
    assert len({l.mx_status_string(i) for i in range(6)}) == 6


def test_argument_validation_without_gpu(lib):
    l, protos = lib
    OK, NULL, SHAPE, ALIGN = 0, 1, 2, 3
    p16, p8, p2 = 0x1000, 0x1008, 0x1002
    # NULL pointers
    assert l.mx_gemv_q4_K_q8(None, None, p16, p16, 4096, 4096) == NULL
    assert l.mx_gemv_q4_K_q8(None, p16, None, p16, 4096, 4096) == NULL
    assert l.mx_quantize_q8_1(None, None, p16, 64) == NULL
    assert l.mx_dequant_q6_K(None, p16, None, 256) == NULL
    # shape preconditions: K % 256 for K-quants, K % 32 for Q8_0 / MXFP4, T in 1..16, n % 32
    assert l.mx_gemv_q4_K_q8(None, p16, p16, p16, 4096 + 32, 16) == SHAPE
    assert l.mx_gemv_q6_K_q8(None, p16, p16, p16, 100, 16) == SHAPE
    assert l.mx_gemv_q8_0_q8(None, p16, p16, p16, 48, 16) == SHAPE
    assert l.mx_gemv_mxfp4_soa_q8(None, p16, p16, p16, p16, 2880 + 16, 16) == SHAPE
    assert l.mx_gemv_q4_K_q8(None, p16, p16, p16, 4096, 0) == SHAPE
    assert l.mx_gemv_q4_K_q8_batched(None, p16, p16, p16, 4096, 16, 0) == SHAPE
    assert l.mx_gemv_q4_K_q8_batched(None, p16, p16, p16, 4096, 16, 17) == SHAPE
    assert l.mx_quantize_q8_1(None, p16, p16, 33) == SHAPE
    assert l.mx_dequant_q4_K(None, p16, p16, 255) == SHAPE
    assert l.mx_dequant_q8_0_to_Bt(None, p16, p16, 48, 4) == SHAPE
    # alignment: Q4_K weights 16 B, q8 stream 8 B, SoA quant plane 16 B
    assert l.mx_gemv_q4_K_q8(None, p16, p8, p16, 4096, 16) == ALIGN
    assert l.mx_gemv_q4_K_q8(None, 0x1004, p16, p16, 4096, 16) == ALIGN
    assert l.mx_gemv_q8_0_soa_q8(None, p16, p8, p16, p16, 4096, 16) == ALIGN
    assert l.mx_gemv_q6_K_q8(None, p16, 0x1001, p16, 4096, 16) == ALIGN
    # host repackers work without a GPU
    import numpy as np
    blk = np.arange(17 * 3, dtype=np.uint8)
    qs, e = np.zeros(48, np.uint8), np.zeros(3, np.uint8)
    assert l.mx_repack_mxfp4_to_soa(blk.ctypes.data, 3, qs.ctypes.data, e.ctypes.data) == OK
    assert e.tolist() == [0, 17, 34] and qs[:16].tolist() == list(range(1, 17))
    assert l.mx_repack_mxfp4_to_soa(None, 3, qs.ctypes.data, e.ctypes.data) == NULL


def test_workspace_forms_validate_before_any_hip_call(lib):
    """The *_ws entry points: size query, NULL / misaligned / too-small workspace."""
    l, _ = lib
    OK, NULL, SHAPE, ALIGN, WORKSPACE = 0, 1, 2, 3, 9
    p16 = 0x1000
    n = C.c_uint64(7)
    # without a GPU the library assumes 256 CUs: 128 blocks of 32 rows want 4 K ranges of T x N partial sums
    assert l.mx_gemv_batched_ws_bytes(14336, 4096, 8, C.addressof(n)) == OK and n.value == 4 * 8 * 4096 * 4
    assert l.mx_gemv_batched_ws_bytes(4096, 151936, 8, C.addressof(n)) == OK and n.value == 0                   # enough row blocks: K is never split
    assert l.mx_gemv_batched_ws_bytes(14336, 4096, 1, C.addressof(n)) == OK and n.value == 0
    assert l.mx_gemv_batched_ws_bytes(14336, 4096, 8, None) == NULL
    assert l.mx_gemv_batched_ws_bytes(14336, 4096, 17, C.addressof(n)) == SHAPE
    need = 4 * 8 * 4096 * 4
    assert l.mx_gemv_q8_0_soa_q8_batched_ws(None, p16, p16, p16, p16, 14336, 4096, 8, None, need) == NULL
    assert l.mx_gemv_q8_0_soa_q8_batched_ws(None, p16, p16, p16, p16, 14336, 4096, 8, 0x1004, need) == ALIGN
    assert l.mx_gemv_q8_0_soa_q8_batched_ws(None, p16, p16, p16, p16, 14336, 4096, 8, p16, need - 4) == WORKSPACE
    assert l.mx_gemv_q6_K_q8_batched_ws(None, p16, p16, p16, 14336, 4096, 8, p16, 16) == WORKSPACE
    assert l.mx_status_string(WORKSPACE).startswith(b"workspace")
    assert l.mx_gemm_ws_bytes(128, 14336, 4096, None) == NULL
    assert l.mx_gemm_q4_K_ws(None, p16, p16, p16, 128, 14336, 4096, None, 64) == NULL
    assert l.mx_gemm_q4_K_ws(None, p16, p16, p16, 128, 14336, 4096, 0x1004, 64) == ALIGN


def test_query_sized_workspace_is_never_refused(lib):
    """mx_gemv_batched_ws_bytes carries no weight format, while the launch picks its kernel (and with it the number of K
    slices) by format: whatever the format, batch and shape, a workspace of the size the query names must not come back
    as MX_ERR_WORKSPACE.  Without a GPU the call gets past the workspace check and fails at the launch instead."""
    l, _ = lib
    WORKSPACE = 9
    p16 = 0x1000
    n = C.c_uint64(0)
    shapes = [(14336, 4096), (14336, 1000), (8192, 14336), (8192, 512), (4096, 14336), (4096, 4096), (12288, 256), (16384, 151936)]
    for K, N in shapes:
        for T in range(2, 17):
            assert l.mx_gemv_batched_ws_bytes(K, N, T, C.addressof(n)) == 0
            ws = p16 if n.value else None
            for rc in (l.mx_gemv_q8_0_soa_q8_batched_ws(None, p16, p16, p16, p16, K, N, T, ws, n.value),
                       l.mx_gemv_q4_K_q8_batched_ws(None, p16, p16, p16, K, N, T, ws, n.value),
                       l.mx_gemv_q6_K_q8_batched_ws(None, p16, p16, p16, K, N, T, ws, n.value),
                       l.mx_gemv_q8_0_q8_batched_ws(None, p16, p16, p16, K, N, T, ws, n.value)):
                assert rc != WORKSPACE, (K, N, T, n.value)


@pytest.mark.parametrize("K,N,T,ranges", [(4096, 2048, 8, 4), (4096, 1024, 5, 8), (6144, 2048, 7, 4), (6144, 3584, 7, 3), (6400, 2048, 8, 3), (4096, 8192, 8, 2)])
def test_workspace_covers_the_k_ranges_of_eight_wave_workgroups(lib, K, N, T, ranges):
    """Without a GPU: 256 CUs.  The form of eight waves takes more K ranges than the one of four; a workspace for fewer would be answered with
    other fp32 sums than the form without a workspace gives, so less than that is refused."""
    l, _ = lib
    n = C.c_uint64(7)
    assert l.mx_gemv_batched_ws_bytes(K, N, T, C.addressof(n)) == 0 and n.value == 4 * ranges * T * N
    for fmt in ("q4_K", "q6_K"):
        run = lambda size: getattr(l, "mx_gemv_%s_q8_batched_ws" % fmt)(None, 0x1000, 0x1000, 0x1000, K, N, T, 0x1000, size)  # noqa: E731,B023
        assert run(n.value) != 9 and run(n.value - 4) == 9


FOUR, EIGHT = (4, 2), (8, 2)   # waves and blocks of 32 rows of a workgroup


@pytest.mark.parametrize("K,N,forms", [(2816, 9888, dict.fromkeys(("q4_K", "q6_K", "q8_0", "q8_0_soa", "mxfp4_soa"), EIGHT)),
                                       (3072, 10880, {"q4_K": EIGHT, "q6_K": FOUR, "q8_0": FOUR, "q8_0_soa": EIGHT, "mxfp4_soa": EIGHT}),
                                       (4096, 9888, {"q4_K": EIGHT, "q6_K": FOUR, "q8_0": FOUR, "q8_0_soa": EIGHT, "mxfp4_soa": FOUR}),
                                       (8192, 10240, dict.fromkeys(("q4_K", "q6_K", "q8_0", "q8_0_soa", "mxfp4_soa"), FOUR)),
                                       (8192, 10944, dict.fromkeys(("q4_K", "q6_K", "q8_0", "q8_0_soa", "mxfp4_soa"), EIGHT))])
@pytest.mark.parametrize("T", [9, 16])
def test_int_dot_blocks_of_64_rows_where_eight_waves_are_faster(lib, T, K, N, forms):
    """Without a GPU: 256 CUs.  Up to two thirds of them in row blocks, four waves have a fourth K range and are faster over long rows."""
    from machx_inference_engine_amd import ops
    assert {f: ops.gemv_batched_plan(f, K, N, T)[:2] for f in forms} == forms
    assert all(ops.gemv_batched_plan(f, K, N, T)[2] == 1 or forms[f] == FOUR for f in forms)


@pytest.mark.parametrize("K,N,formats", [(256, 8192, ()), (512, 6144, ()), (544, 6144, ("q8_0", "mxfp4_soa")), (768, 4928, ("q4_K", "q6_K", "q8_0", "mxfp4_soa")),
                                         (1024, 8192, ("q4_K", "q6_K", "q8_0", "q8_0_soa", "mxfp4_soa"))])
def test_int_dot_blocks_of_32_rows_have_work_for_eight_waves(lib, K, N, formats):
    """Without a GPU: 256 CUs.  Rows of one or two groups leave six of eight waves without one."""
    from machx_inference_engine_amd import ops
    all_formats = ("q4_K", "q6_K", "q8_0", "q8_0_soa", "mxfp4_soa") if K % 256 == 0 else ("q8_0", "q8_0_soa", "mxfp4_soa")
    for f in all_formats:
        assert ops.gemv_batched_plan(f, K, N, 12)[:2] == ((8, 1) if f in formats else (4, 2)), f


@pytest.mark.parametrize("K,N,formats", [(4096, 3072, ("q4_K", "q6_K", "q8_0_soa")), (4608, 3072, ("q4_K", "q6_K", "q8_0_soa", "mxfp4_soa")), (5120, 3072, ()),
                                         (5888, 2816, ()), (5120, 2560, ("q4_K", "q6_K", "q8_0_soa", "mxfp4_soa")), (6144, 2560, ("q4_K", "q6_K", "q8_0_soa")),
                                         (6144, 3072, ("q4_K", "q6_K", "q8_0_soa", "mxfp4_soa")), (6144, 5440, ("q4_K", "q8_0_soa")),
                                         (6144, 5472, ("q4_K", "q6_K", "q8_0_soa", "mxfp4_soa"))])
def test_int_dot_k_ranges_of_eight_waves_where_they_are_faster(lib, K, N, formats):
    """Without a GPU: 256 CUs.  Up to 8 tokens: two K ranges of 10 to 12 groups and, by format, the shapes where four waves have a third range run in those."""
    from machx_inference_engine_amd import ops
    for f in ("q4_K", "q6_K", "q8_0_soa", "mxfp4_soa"):
        assert ops.gemv_batched_plan(f, K, N, 6)[0] == (8 if f in formats else 4), f


def test_int_dot_plan_query(lib):
    l, _ = lib
    from machx_inference_engine_amd import ops
    plan = (C.c_uint32 * 3)()
    p = C.addressof(plan)
    assert l.mx_gemv_batched_plan(None, 4096, 4096, 8, p) == 1 and l.mx_gemv_batched_plan(b"q4_K", 4096, 4096, 8, None) == 1
    assert l.mx_gemv_batched_plan(b"q4_K", 4096, 4096, 17, p) == 2 and l.mx_gemv_batched_plan(b"q5_K", 4096, 4096, 8, p) == 5
    assert ops.gemv_batched_plan("q4_K", 4096, 4096, 4) == (0, 0, 0) and ops.gemv_batched_plan("q8_0", 4096, 14336, 8) == (0, 0, 0)
    assert ops.gemv_batched_plan("q6_K", 8192, 4096, 4)[0] == 4 and ops.gemv_batched_plan("q4_K", 4096, 14336, 5) == (4, 1, 1)


def test_dense_gemm_uses_the_shared_scratch_only_where_the_header_says(lib):
    """Without a workspace a dense quant-GEMM is K-sliced, and so uses the scratch that overlapping calls race on, only for K >= 2048
    and 128 x 256 tiles on at most half of the CUs (256 without a GPU), within its 8 Mi floats.  A workspace lifts the first two
    conditions; the Python entry points bring one of their own where the tiles are too many."""
    l, _ = lib
    from machx_inference_engine_amd import ops
    sliced = own = 0
    for M in (1, 17, 64, 77, 137, 200, 256, 337, 512, 700, 1024, 2048):
        for K in (128, 1024, 1280, 1792, 1984, 2048, 2880, 5888, 8448, 14336):
            for N in (33, 512, 896, 1024, 4096, 11712, 14336, 16640):
                k = ops.gemm_plan(M, K, N)[2]
                documented = K >= 2048 and 2 * (-(-M // 128) * -(-N // 256)) <= 256
                assert 1 <= k <= 8 and (k == 1 or (documented and k * M * N <= 8 << 20)), (M, K, N, k)
                with_ws = ops.gemm_plan(M, K, N, 32 << 20)[2]
                assert k in (1, with_ws), (M, K, N, k, with_ws)
                assert ops._gemm_own_bytes(M, K, N) == (4 * with_ws * M * N if K >= 2048 and with_ws > k else 0), (M, K, N)
                assert ops.gemm_plan(M, K, N, 4 * with_ws * M * N) == ops.gemm_plan(M, K, N, 32 << 20)
                sliced += k > 1
                own += K >= 2048 and with_ws > k
    assert sliced > 50 and own > 2
    assert ops.gemm_plan(64, 1280, 896)[2] == ops.gemm_plan(256, 1792, 1024)[2] == ops.gemm_plan(137, 5888, 16640)[2] == 1
    plan = (C.c_uint32 * 3)()
    assert l.mx_gemm_plan(64, 1280, 896, 0, 0, None) == 1 and l.mx_gemm_plan(64, 0, 896, 0, 0, C.addressof(plan)) == 2
    p16 = 0x1000
    for name, w in (("q4_0", (p16,)), ("q5_K", (p16,)), ("mxfp4_soa", (p16, p16))):
        fn = getattr(l, "mx_gemm_%s_ws" % name)
        assert fn(None, p16, *w, p16, 64, 1280, 896, None, 64) == 1 and fn(None, p16, *w, p16, 64, 1280, 896, 0x1004, 64) == 3


DENSE = ("q4_K", "q6_K", "q8_0", "q8_0_soa", "q4_0", "q5_K", "mxfp4_soa")


def test_gemm_form_query(lib):
    """mx_gemm_plan is the plan the formats share; what a launch does depends on the format too, and mx_gemm_form says it."""
    l, _ = lib
    from machx_inference_engine_amd import ops
    for M, K, N in [(1, 64, 33), (77, 14336, 4096), (256, 14336, 4096), (512, 4096, 14336), (700, 1792, 9000)]:
        for f in DENSE:
            for ws in (None, 32 << 20):
                assert ops.gemm_form(f, M, K, N, ws)[:4] == ops.gemm_plan(M, K, N, ws) + (0,), (f, M, K, N)
    assert all(ops.gemm_form(f, 4096, 14336, 4096) == (8, 2, 1, 0, 0) for f in DENSE) and ops.gemm_plan(4096, 14336, 4096)[0] == 0
    form = (C.c_uint32 * 5)()
    p = C.addressof(form)
    assert l.mx_gemm_form(None, 64, 1280, 896, 0, 0, p) == 1 and l.mx_gemm_form(b"q4_K", 64, 1280, 896, 0, 0, None) == 1
    assert l.mx_gemm_form(b"q4_K", 64, 0, 896, 0, 0, p) == 2 and l.mx_gemm_form(b"q3_K", 64, 1280, 896, 0, 0, p) == 5


def test_gemm_column_halves_are_q6_K_s(lib):
    """Column halves of 256-token tiles: the formats whose tiles the model takes without a margin run them whole."""
    from machx_inference_engine_amd import ops
    for M, K, N in [(33000, 14336, 4096), (6400, 24576, 10496), (1644, 13056, 4608), (4096, 14336, 5000)]:
        assert ops.gemm_form("q6_K", M, K, N)[0] == 8 and all(ops.gemm_form(f, M, K, N)[3] == 0 for f in DENSE if f != "q6_K")
    assert ops.gemm_form("q6_K", 1644, 13056, 4500)[3] == 126 and ops.gemm_form("q6_K", 1600, 2048, 12900)[3] == 101


@pytest.mark.parametrize("M,K,N,tall", [(2048, 4096, 14336, True), (710, 8448, 20608, True), (1644, 13056, 4608, True), (2513, 2560, 3904, True), (676, 13824, 14528, True),
                                        (1166, 8960, 14848, True), (1292, 12032, 7936, False), (2145, 6912, 4416, False), (1589, 4352, 5056, False),
                                        (284, 5376, 26944, False), (266, 8704, 25344, False), (767, 5632, 11776, False)])
def test_gemm_q6_K_takes_256_token_tiles_where_they_are_faster(lib, M, K, N, tall):
    """Without a GPU: 256 CUs.  Timed against the plan's form: 0.74 to 0.95 of its time where taken, 1.01 to 1.15 where not."""
    from machx_inference_engine_amd import ops
    form = ops.gemm_form("q6_K", M, K, N)
    assert (form[0] == 8) == tall and (tall or form[:3] == ops.gemm_plan(M, K, N))


@pytest.mark.parametrize("M,K,N,light", [(520, 11008, 21208, False), (600, 14336, 21208, False), (640, 14336, 21208, False), (641, 14336, 21208, True), (780, 12032, 15232, False),
                                         (1100, 12288, 13000, False), (1300, 11008, 10456, False), (1540, 14336, 8920, True), (4621, 14336, 3288, True)])
def test_gemm_256_token_tiles_with_a_half_empty_one(lib, M, K, N, light):
    """Without a GPU: 256 CUs.  Formats that cost little to dequantize keep the plan where a last token tile of at most 128 rows is one of few."""
    from machx_inference_engine_amd import ops
    for f in DENSE[2:3] + DENSE[5:]:
        assert ops.gemm_form(f, M, K, N)[0] == 8, f
    for f in ("q4_K", "q4_0", "q8_0_soa"):
        assert (ops.gemm_form(f, M, K, N)[0] == 8) == light, f


@pytest.mark.parametrize("M,K,N,form,dwords", [(30, 2048, 6144, (1, 1), 1), (4, 6400, 17152, (1, 2), 1), (7, 11264, 14720, (1, 2), 0), (18, 12288, 10944, (1, 2), 0),
                                               (16, 5120, 20352, (1, 2), 0), (5, 4096, 19008, (1, 2), 0), (11, 4608, 11136, (1, 2), 1), (30, 3584, 12288, (1, 2), 1), (38, 6400, 8896, (2, 2), 1), (42, 7168, 18752, (2, 2), 0), (542, 6400, 1984, (4, 1), 1),
                                               (114, 11776, 6528, (4, 1), 0), (77, 14336, 4096, (3, 1), 0), (94, 7168, 13696, (3, 1), 0), (96, 7680, 17408, (3, 2), 0), (65, 3072, 9152, (3, 1), 1), (159, 5120, 3456, (3, 1), 1), (156, 2304, 10880, (2, 1), 1),
                                               (527, 3072, 10688, (3, 2), 1), (512, 4096, 14336, (4, 2), 0)])
def test_gemm_q6_K_loads_dwords_where_that_is_faster(lib, M, K, N, form, dwords):
    """Without a GPU: 256 CUs.  Rows of an odd number of blocks in every eight-wave form below 128 x 256; of an even number not in those that lose 1 to 7 %."""
    from machx_inference_engine_amd import ops
    f = ops.gemm_form("q6_K", M, K, N)
    assert f[:2] == form and f[4] == dwords
    assert all(ops.gemm_form(o, M, K, N)[4] == 0 for o in DENSE if o != "q6_K")


def test_gemm_workspace_query_names_what_the_plan_uses(lib):
    """A workspace of the queried size gives the plan of an unlimited one, and outside the shapes that the library's own scratch
    serves it is no larger than that plan's partial sums."""
    l, _ = lib
    from machx_inference_engine_amd import ops
    for M, K, N in [(572, 12800, 27584), (64, 1280, 896), (256, 1792, 1024), (137, 5888, 16640), (77, 14336, 4096), (256, 14336, 4096),
                    (512, 4096, 14336), (4096, 4096, 14336), (1, 128, 33), (337, 8448, 11712)]:
        need, k = ops.gemm_ws_bytes(M, K, N), ops.gemm_plan(M, K, N, 1 << 62)[2]
        assert ops.gemm_plan(M, K, N, need) == ops.gemm_plan(M, K, N, 1 << 62), (M, K, N)
        served = K >= 2048 and 2 * (-(-M // 128) * -(-N // 256)) <= 256
        assert need == (0 if k == 1 else (8 if served else k) * M * N * 4), (M, K, N, k, need)
