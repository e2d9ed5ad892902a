"""Parity of the HIP EXL3 path (through the C ABI) against the CPU oracle."""
import numpy as np
import pytest

from helpers import assert_close, make_linear, make_x

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hx():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from helios_glm53flash_amd import exl3
    return exl3


def _dev(a, dtype=None):
    import torch
    t = torch.from_numpy(np.ascontiguousarray(a))
    if dtype is not None:
        t = t.view(dtype)
    return t.cuda()


@pytest.mark.parametrize("bits", range(1, 9))
@pytest.mark.parametrize("cb", [0, 1, 2])
def test_reconstruct_bit_exact_golden(hx, bits, cb):
    import torch
    from pathlib import Path
    f = np.load(Path(__file__).parent / "golden" / "reconstruct_small.npz")
    tr = f[f"trellis_b{bits}_cb{cb}"]
    want = f[f"w_b{bits}_cb{cb}"]
    K, N = tr.shape[0] * 16, tr.shape[1] * 16
    out = torch.empty((K, N), dtype=torch.float16, device="cuda")
    hx.reconstruct(out, _dev(tr, torch.int16), K // 16, N // 16, N, bits, cb == 1, cb == 2)
    torch.cuda.synchronize()
    got = out.cpu().view(torch.int16).numpy().view(np.uint16)
    assert np.array_equal(got, want)


def test_reconstruct_slice_offset(hx):
    import torch
    from oracle import oracle as O
    K, N, bits = 64, 512, 3
    tr, _, _ = make_linear(3, K, N, bits)
    want = O.reconstruct(tr, K, N, bits, 2)[:, 256:384]
    out = torch.empty((K, 128), dtype=torch.float16, device="cuda")
    hx.reconstruct_slice(out, _dev(tr, torch.int16), K // 16, N // 16, 128, bits, False, True, 256)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().view(torch.int16).numpy().view(np.uint16), want)


def _run_linear(hx, M, K, N, bits, cb, y_fp32, seed=0):
    import torch
    from oracle import oracle as O
    tr, suh, svh = make_linear(seed + 1, K, N, bits)
    x = make_x(seed + 2, M, K)
    w = hx.GroupWords(_dev(tr, torch.int16), _dev(suh), _dev(svh), hx.MUL1 if cb == 2 else 0)
    y = torch.empty((M, N), dtype=torch.float32 if y_fp32 else torch.float16, device="cuda")
    path = hx.gemm(y, _dev(x), w, M, N, K, bits, y_fp32, mcg=(cb == 1))
    torch.cuda.synchronize()
    ref = O.linear(x, tr, suh, svh, K, N, bits, cb, out_f16=not y_fp32)
    return path, y.float().cpu().numpy(), ref


@pytest.mark.parametrize("M", [1, 3, 8, 13, 16])
@pytest.mark.parametrize("bits,cb", [(2, 2), (3, 2), (4, 2), (4, 0), (5, 1), (6, 2), (8, 2), (1, 0), (7, 1)])
def test_gemv_parity(hx, M, bits, cb):
    path, got, ref = _run_linear(hx, M, 1024, 512, bits, cb, True, seed=M * 10 + bits)
    assert path == hx.HX_GEMM_PATH_GEMV
    assert_close(got, ref, what=f"gemv M={M} bits={bits} cb={cb}")


@pytest.mark.parametrize("M,K", [(1, 128), (1, 2048), (1, 2176), (2, 1152), (3, 6400), (5, 384), (9, 1920), (16, 128)])
def test_gemv_input_transform_groups(hx, M, K):
    """The input transform's groups of 16 (row, block) pairs: one pair, exactly one group, remainders, more
    groups than waves; split ranges that are not a multiple of a group."""
    _, got, ref = _run_linear(hx, M, K, 256, 3, 2, True, seed=M + K)
    assert_close(got, ref, what=f"gemv M={M} K={K}")


def test_gemv_input_at_4_byte_alignment(hx):
    import torch
    from oracle import oracle as O
    K, N, bits = 1024, 256, 4
    tr, suh, svh = make_linear(8, K, N, bits)
    x = make_x(9, 3, K)
    at2 = [torch.cat([torch.zeros(2, dtype=torch.float16), torch.from_numpy(v).reshape(-1)]).cuda()[2:]
           for v in (x, suh)]  # contiguous, 4 bytes past a 16-byte boundary
    w = hx.GroupWords(_dev(tr, torch.int16), at2[1], _dev(svh), hx.MUL1)
    y = torch.empty((3, N), dtype=torch.float32, device="cuda")
    hx.gemm(y, at2[0], w, 3, N, K, bits, True)
    torch.cuda.synchronize()
    assert_close(y.cpu().numpy(), O.linear(x, tr, suh, svh, K, N, bits, 2, out_f16=False), what="4-byte alignment")


def test_gemv_fp16_out_and_repeat(hx):
    # second call reuses the workspace counters (must have been reset by the first)
    for _ in range(3):
        _, got, ref = _run_linear(hx, 2, 2048, 1024, 2, 2, False, seed=5)
        assert_close(got, ref, what="gemv fp16 out")


def test_gemv_attention_projection_shape(hx):
    """K=4096 -> N=12288, 4-bit, M in {1, 4, 8}."""
    for M in (1, 8):
        _, got, ref = _run_linear(hx, M, 4096, 12288, 4, 2, True, seed=40 + M)
        assert_close(got, ref, what=f"attn proj M={M}")


@pytest.mark.parametrize("M", [17, 32, 100, 256])
@pytest.mark.parametrize("bits,cb", [(2, 2), (3, 2), (4, 0), (5, 2)])
def test_mfma_parity(hx, M, bits, cb):
    path, got, ref = _run_linear(hx, M, 512, 384, bits, cb, True, seed=M + bits)
    assert path == hx.HX_GEMM_PATH_MFMA
    assert_close(got, ref, what=f"mfma M={M} bits={bits} cb={cb}")


@pytest.mark.parametrize("M,K,N,bits,cb", [(17, 4096, 256, 4, 2), (32, 640, 128, 2, 2), (33, 1152, 384, 3, 0),
                                           (64, 4096, 128, 5, 1), (65, 2176, 256, 8, 2), (97, 4096, 128, 2, 2),
                                           (129, 1024, 256, 6, 2), (224, 3968, 128, 1, 2), (300, 512, 128, 7, 0),
                                           (17, 128, 128, 4, 2), (40, 256, 128, 2, 1), (90, 128, 256, 3, 2)])
@pytest.mark.parametrize("y_fp32", [False, True])
def test_mfma_row_tiles_and_k_splits(hx, M, K, N, bits, cb, y_fp32):
    """Row tiles of every height with full and partial rows; K split into unequal chunk counts, too short to
    split, and shorter than the rings."""
    for _ in range(2):  # the second call finds the arrival counters as the first left them
        path, got, ref = _run_linear(hx, M, K, N, bits, cb, y_fp32, seed=M + K)
        assert path == hx.HX_GEMM_PATH_MFMA
        assert_close(got, ref, what=f"mfma M={M} K={K} N={N} bits={bits} cb={cb}")


@pytest.mark.parametrize("ws_bytes", [0, 64 * 1024, 64 * 1024 + 45 * 8 * 4, None])
def test_mfma_small_workspace(hx, ws_bytes):
    """a_had given with no workspace, a small one or one of the queried size: the call needs none and leaves it alone."""
    import ctypes as C
    import torch
    from oracle import oracle as O
    from helios_glm53flash_amd._lib import lib
    M, K, N, bits = 45, 1024, 256, 4
    tr, suh, svh = make_linear(21, K, N, bits)
    x = make_x(22, M, K)
    w = hx.GroupWords(_dev(tr, torch.int16), _dev(suh), _dev(svh), hx.MUL1)
    ref = O.linear(x, tr, suh, svh, K, N, bits, 2, out_f16=False)
    xd, a_had, y = _dev(x), torch.empty((M, K), dtype=torch.float16, device="cuda"), torch.empty((M, N), device="cuda")
    n = lib.hx_exl3_gemm_workspace_size(M, N, K) if ws_bytes is None else ws_bytes
    ws = torch.zeros(n + 256, dtype=torch.uint8, device="cuda")
    ws[n:] = 7
    gw = w.c()
    r = lib.hx_exl3_gemm(y.data_ptr(), xd.data_ptr(), C.byref(gw), M, N, K, bits, 1, None, a_had.data_ptr(), 0,
                         ws.data_ptr() if n else None, n)
    torch.cuda.synchronize()
    assert r == hx.HX_GEMM_PATH_MFMA
    assert_close(y.cpu().numpy(), ref, what=f"workspace {ws_bytes}")
    assert bool((ws[n:] == 7).all()) and not bool(ws[:min(n, 64 * 1024)].any())


@pytest.mark.parametrize("M,N", [(45, 512), (300, 256)])
def test_mfma_workspace_beyond_the_least(hx, M, N):
    """Without a_had: the least workspace, room for the row sums of K splits, one byte short of their partials, and enough
    for them.  Nothing past the end is written, the counters return to zero."""
    import ctypes as C
    import torch
    from oracle import oracle as O
    from helios_glm53flash_amd._lib import HX_ERR_WORKSPACE, lib
    K, bits = 2048, 4
    tr, suh, svh = make_linear(31, K, N, bits)
    x = make_x(32, M, K)
    w = hx.GroupWords(_dev(tr, torch.int16), _dev(suh), _dev(svh), hx.MUL1)
    ref = O.linear(x, tr, suh, svh, K, N, bits, 2, out_f16=False)
    xd, gw = _dev(x), w.c()
    least = lib.hx_exl3_gemm_workspace_size(M, N, K)
    rs = (M * K // 32 + 255) // 256 * 256  # an fp32 sum per 128 inputs
    # 2048 / 64 = 32 chunks of k: 5 splits of 6 and 7; a split stores 16-row fragments of 128 columns, a row tile at most 128 rows
    partial = (M + 127) // 128 * (N // 128) * 5 * ((min(M, 128) + 15) // 16 * 16) * 128 * 4
    outs = []
    for n in (least, least + rs, least + rs + partial - 1, least + rs + partial,
              least + lib.hx_exl3_gemm_extra_bytes()):
        ws = torch.zeros(n + 4096, dtype=torch.uint8, device="cuda")
        ws[n:] = 7
        y = torch.empty((M, N), device="cuda")
        r = lib.hx_exl3_gemm(y.data_ptr(), xd.data_ptr(), C.byref(gw), M, N, K, bits, 1, None, None, 0, ws.data_ptr(), n)
        torch.cuda.synchronize()
        assert r == hx.HX_GEMM_PATH_MFMA
        assert_close(y.cpu().numpy(), ref, what=f"workspace of {n}")
        assert bool((ws[n:] == 7).all()) and not bool(ws[:64 * 1024].any())
        outs.append(y)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[1], outs[2]) and torch.equal(outs[3], outs[4])
    assert not torch.equal(outs[2], outs[3])
    ws = torch.zeros(least, dtype=torch.uint8, device="cuda")
    assert lib.hx_exl3_gemm(outs[0].data_ptr(), xd.data_ptr(), C.byref(gw), M, N, K, bits, 1, None, None, 0,
                            ws.data_ptr(), 64 * 1024) == HX_ERR_WORKSPACE


@pytest.mark.parametrize("M,K,N,split", [(126, 1280, 17792, False), (512, 1024, 8192, False), (200, 2048, 17792, False),
                                         (17, 1280, 24576, False), (126, 2944, 17792, False), (126, 1280, 8192, True),
                                         (17, 3072, 17792, True), (45, 4096, 12288, True), (200, 6144, 12288, True)])
def test_mfma_splits_only_where_they_pay(hx, M, K, N, split):
    """Splits of a K that is too short for its number of tiles were up to 30 % slower than no split: with the least
    workspace the call is unsplit, with more room it is split, or, where K is too short, gives the same bits."""
    import ctypes as C
    import torch
    from helios_glm53flash_amd._lib import lib
    tr, suh, svh = make_linear(51, K, N, 2)
    w = hx.GroupWords(_dev(tr, torch.int16), _dev(suh), _dev(svh), hx.MUL1)
    xd, gw = _dev(make_x(52, M, K)), w.c()
    least = lib.hx_exl3_gemm_workspace_size(M, N, K)
    ys = []
    for n in (least, least + lib.hx_exl3_gemm_extra_bytes()):
        ws = torch.zeros(n, dtype=torch.uint8, device="cuda")
        y = torch.empty((M, N), device="cuda")
        lib.hx_exl3_gemm(y.data_ptr(), xd.data_ptr(), C.byref(gw), M, N, K, 2, 1, None, None, 0, ws.data_ptr(), n)
        torch.cuda.synchronize()
        ys.append(y)
    assert torch.equal(*ys) == (not split)
    assert float((ys[0] - ys[1]).norm() / ys[0].norm()) < 1e-5  # the order of fp32 sums: sqrt(K) * 2^-24 = 4e-6 of the size


@pytest.mark.parametrize("M,N,bits,ahead", [(130, 34816, 4, True), (170, 34816, 3, True), (200, 34816, 2, True),
                                            (256, 34816, 1, True), (256, 34816, 5, False), (130, 24576, 4, False)])
def test_mfma_many_tiles(hx, M, N, bits, ahead):
    """544 tiles, up to 4 bits: the row sums made ahead of the tiles if the workspace has room for them; in the tile
    otherwise, at more bits and at 384 tiles; last row tiles of every height."""
    import ctypes as C
    import torch
    from oracle import oracle as O
    from helios_glm53flash_amd._lib import lib
    K = 128
    tr, suh, svh = make_linear(61, K, N, bits)
    x = make_x(62, M, K)
    w = hx.GroupWords(_dev(tr, torch.int16), _dev(suh), _dev(svh), hx.MUL1)
    ref = O.linear(x, tr, suh, svh, K, N, bits, 2, out_f16=False)
    xd, gw = _dev(x), w.c()
    least = lib.hx_exl3_gemm_workspace_size(M, N, K)
    for room in (0, (M * K // 32 + 255) // 256 * 256):
        ws = torch.zeros(least + room + 4096, dtype=torch.uint8, device="cuda")
        y = torch.empty((M, N), device="cuda")
        lib.hx_exl3_gemm(y.data_ptr(), xd.data_ptr(), C.byref(gw), M, N, K, bits, 1, None, None, 0, ws.data_ptr(),
                         least + room)
        torch.cuda.synchronize()
        assert_close(y.cpu().numpy(), ref, what=f"room {room}")
        sums = ws[least:least + room].view(torch.float32)
        assert bool(sums.any()) == (room > 0 and ahead) and not bool(ws[least + room:].any())


def test_mfma_captured_on_a_decode_stream(hx):
    """An M > 16 linear captured on a stream that only ran M = 1: every replay gives the eager bits, also after eager
    calls of other shapes on the stream, which must not move or release the workspace that the graph holds."""
    import torch
    K, N, bits = 4096, 1024, 4
    tr, suh, svh = make_linear(41, K, N, bits)
    w = hx.GroupWords(_dev(tr, torch.int16), _dev(suh), _dev(svh), hx.MUL1)
    x = {M: _dev(make_x(42 + M, M, K)) for M in (1, 45, 100)}
    y = {M: torch.empty((M, N), device="cuda") for M in x}
    eager = torch.empty((45, N), device="cuda")
    hx.gemm(eager, x[45], w, 45, N, K, bits, True)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    hx.gemm(y[1], x[1], w, 1, N, K, bits, True, stream=s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        hx.gemm(y[45], x[45], w, 45, N, K, bits, True)
    for rep in range(4):
        y[45].fill_(float("nan"))
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y[45], eager), rep
        hx.gemm(y[100], x[100], w, 100, N, K, bits, True, stream=s)  # eager work between replays
        torch.full((1 << 20,), -1.0, device="cuda")
        torch.cuda.synchronize()


def test_mfma_with_a_had_leaves_the_workspace(hx):
    """The caller's a_had is all the scratch of an M > 16 call: a workspace that another call in flight may be using
    (nothing in it is zero here) is neither read nor written."""
    import ctypes as C
    import torch
    from oracle import oracle as O
    from helios_glm53flash_amd._lib import lib
    M, K, N, bits = 45, 2048, 256, 4
    tr, suh, svh = make_linear(23, K, N, bits)
    x = make_x(24, M, K)
    w = hx.GroupWords(_dev(tr, torch.int16), _dev(suh), _dev(svh), hx.MUL1)
    xd, a_had, y = _dev(x), torch.empty((M, K), dtype=torch.float16, device="cuda"), torch.empty((M, N), device="cuda")
    ws = torch.full((64 << 20,), 5, dtype=torch.uint8, device="cuda")
    gw = w.c()
    r = lib.hx_exl3_gemm(y.data_ptr(), xd.data_ptr(), C.byref(gw), M, N, K, bits, 1, None, a_had.data_ptr(), 0,
                         ws.data_ptr(), ws.numel())
    torch.cuda.synchronize()
    assert r == hx.HX_GEMM_PATH_MFMA and bool((ws == 5).all())
    assert_close(y.cpu().numpy(), O.linear(x, tr, suh, svh, K, N, bits, 2, out_f16=False), what="a_had")


def test_gemv_many_splits(hx):
    """More K splits than the last arriver reads together, with 1 and 2 16-byte pieces per thread."""
    for M in (3, 8, 11, 16):
        _, got, ref = _run_linear(hx, M, 9 * 512, 128, 4, 2, False, seed=60 + M)
        assert_close(got, ref, what=f"gemv splits M={M}")


def test_mfma_fp16_out(hx):
    _, got, ref = _run_linear(hx, 64, 1024, 256, 2, 2, False, seed=77)
    assert_close(got, ref, what="mfma fp16")


def test_config1_single_linear(hx):
    """K=4096, N=2048, 2-bit, M=1 vs fp64 decode+matmul."""
    _, got, ref = _run_linear(hx, 1, 4096, 2048, 2, 2, True, seed=1)
    assert_close(got, ref, what="config 1")


@pytest.mark.parametrize("M", [1, 64])
def test_dense_3bit_real_shape(hx, M):
    """3-bit dense linear at a projection's real shape (K=4096 -> N=12288), GEMV and MFMA paths."""
    path, got, ref = _run_linear(hx, M, 4096, 12288, 3, 2, True, seed=300 + M)
    assert path == (hx.HX_GEMM_PATH_GEMV if M <= 16 else hx.HX_GEMM_PATH_MFMA)
    assert_close(got, ref, what=f"3-bit 4096x12288 M={M}")


@pytest.mark.parametrize("cb", [2, 1, 0])
def test_gemv_stream_k_sampled_columns(hx, cb):
    """One row whose split-K grid would be one workgroup per column group, unevenly spread over the
    256 CUs (1100 groups), takes the stream-K grid: 1024 workgroups over equal runs of (column group,
    128-k block) units, so most column groups are shared by two workgroups whose partials the last
    arriver adds.  Sampled column groups against the oracle, fp16 output, three calls in a row (the
    arrival counters are reset by each call, and the result is the same every time); codebooks mul1
    (2), MCG (1) and the 3INST table (0)."""
    import torch
    from oracle import oracle as O
    K, N, bits = 4096, 1100 * 128, 2
    tr, suh, svh = make_linear(702 + cb, K, N, bits)
    x = make_x(703, 1, K)
    w = hx.GroupWords(_dev(tr, torch.int16), _dev(suh), _dev(svh), hx.MUL1 if cb == 2 else 0)
    # workgroup i takes units [i*T/1024, (i+1)*T/1024) of T = 1100 * 32 (34.4 blocks each): groups 1,
    # 30, 31 and 32 are split over two workgroups, 0, 549, 550 and the last lie in one
    groups = (0, 1, 30, 31, 32, 549, 550, N // 128 - 1)
    refs = {}
    for g in groups:
        sl = slice(128 * g, 128 * g + 128)
        sub = np.ascontiguousarray(tr[:, 8 * g:8 * g + 8, :])
        refs[g] = O.linear(x, sub, suh, np.ascontiguousarray(svh[sl]), K, 128, bits, cb, out_f16=True)
    first = None
    for call in range(3):
        y = torch.empty((1, N), dtype=torch.float16, device="cuda")
        assert hx.gemm(y, _dev(x), w, 1, N, K, bits, False, mcg=(cb == 1)) == hx.HX_GEMM_PATH_GEMV
        torch.cuda.synchronize()
        got = y.float().cpu().numpy()
        for g in groups:
            sl = slice(128 * g, 128 * g + 128)
            assert_close(got[:, sl], refs[g], what=f"stream-K {bits}-bit cb {cb} group {g} call {call}")
        if first is None:
            first = got
        else:
            assert np.array_equal(got, first), "stream-K result changed between calls"


@pytest.mark.parametrize("M", [1, 512])
def test_lm_head_6bit_sampled_columns(hx, M):
    """6-bit lm_head at its real shape (K=4096 -> N=151552), GEMV (M=1) and MFMA (M=512) paths; the
    oracle checks sampled 128-column groups (each group's output transform is independent of the
    others, so a tile-column slice of the weight is an exact sub-problem)."""
    import torch
    from oracle import oracle as O
    K, N, bits = 4096, 151552, 6
    tr, suh, svh = make_linear(600 + M, K, N, bits)
    x = make_x(601 + M, M, K)
    w = hx.GroupWords(_dev(tr, torch.int16), _dev(suh), _dev(svh), hx.MUL1)
    y = torch.empty((M, N), dtype=torch.float32, device="cuda")
    a_had = torch.empty((M, K), dtype=torch.float16, device="cuda") if M > hx.GEMV_MAX_M else None
    hx.gemm(y, _dev(x), w, M, N, K, bits, True, a_had=a_had)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    rows = np.arange(M) if M <= 16 else np.array([0, 1, 255, 256, 511])
    for g in (0, 517, N // 128 - 1):
        sl = slice(128 * g, 128 * g + 128)
        sub = np.ascontiguousarray(tr[:, 8 * g:8 * g + 8, :])
        ref = O.linear(x[rows], sub, suh, np.ascontiguousarray(svh[sl]), K, 128, bits, 2, out_f16=False)
        assert_close(got[rows, sl], ref, what=f"lm_head 6-bit M={M} group {g}")


@pytest.mark.parametrize("K", range(1, 9))
def test_pack_unpack_trellis_bit_exact(hx, K):
    """pack_trellis / unpack_trellis (pack.cu): GPU packing equals the oracle's packer for every block,
    and unpacking returns the symbols (low K bits of the oracle's windows)."""
    import torch
    from oracle import oracle as O
    rows, cols = 3, 5
    r = np.random.default_rng(K)
    sym = r.integers(0, 65536, size=(rows * cols, 256), dtype=np.uint16)  # bits above K are ignored
    packed = torch.empty((rows * cols, 16 * K), dtype=torch.int16, device="cuda")
    hx.pack_trellis(packed, _dev(sym, torch.int16), rows, cols, K)
    back = torch.empty((rows * cols, 256), dtype=torch.int16, device="cuda")
    hx.unpack_trellis(back, packed, rows, cols, K)
    torch.cuda.synchronize()
    got = packed.cpu().numpy().view(np.uint16)
    mask = (1 << K) - 1
    for b in range(rows * cols):
        want = O.pack_tile(sym[b] & mask, K)
        assert np.array_equal(got[b], want), b
        assert np.array_equal(O.unpack_tile(want, K) & mask, sym[b] & mask)
    assert np.array_equal(back.cpu().numpy().view(np.uint16), sym & mask)


@pytest.mark.parametrize("bits,cb", [(2, 2), (3, 0), (4, 1), (6, 2)])
def test_reconstruct_had_slice(hx, bits, cb):
    """Original-basis weights diag(suh) H W_hat H diag(svh) / 128 per 128 x 128 tile against fp64 on the
    bit-exact W_hat; a column slice with its pre-offset svh."""
    import torch
    from oracle import oracle as O
    K, N = 256, 512
    tr, suh, svh = make_linear(90 + bits, K, N, bits)
    w_hat = O.reconstruct(tr, K, N, bits, cb).view(np.float16).astype(np.float64)
    idx = np.arange(128)
    H = np.where(np.array([[bin(i & j).count("1") & 1 for j in idx] for i in idx]) == 0, 1.0, -1.0)
    ref = np.empty((K, N))
    for a in range(0, K, 128):
        for b in range(0, N, 128):
            ref[a:a + 128, b:b + 128] = H @ w_hat[a:a + 128, b:b + 128] @ H / 128.0
    ref *= suh.astype(np.float64)[:, None] * svh.astype(np.float64)[None, :]
    out = torch.empty((K, N), dtype=torch.float16, device="cuda")
    hx.reconstruct_had_slice(out, _dev(tr, torch.int16), _dev(suh), _dev(svh), K // 16, N // 16, K, N, bits,
                             cb == 1, cb == 2, 0)
    part = torch.empty((K, 256), dtype=torch.float16, device="cuda")
    hx.reconstruct_had_slice(part, _dev(tr, torch.int16), _dev(suh), _dev(np.ascontiguousarray(svh[128:384])),
                             K // 16, N // 16, K, 256, bits, cb == 1, cb == 2, 128)
    torch.cuda.synchronize()
    assert_close(out.float().cpu().numpy(), ref, what=f"reconstruct_had bits={bits} cb={cb}")
    assert np.array_equal(part.cpu().numpy(), out.cpu().numpy()[:, 128:384])
