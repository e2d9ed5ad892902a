"""Host side of the calls: the bit widths passed with the expert tables, the workspaces passed to the linear."""
import pytest
import torch

from helios_glm53flash_amd import exl3, moe


def _experts(bits):
    """A 128 x 128 ExpertSet on the CPU (the tables only hold addresses)."""
    tr = [[torch.zeros((8, 8, 16 * b), dtype=torch.int16) for b in bits] for _ in range(3)]
    v = [[torch.ones(128, dtype=torch.float16) for _ in bits] for _ in range(3)]
    return moe.ExpertSet(128, 128, tr, v, v, [list(bits) for _ in range(3)])


def test_call_bits_follow_the_tables():
    ex = _experts((2, 2, 2))
    assert ex.tables().bits_mask == 0 and ex.call_bits() == (2, 2, 2)
    ex.bits = [[3, 3, 3]] * 3
    ex._tables = None  # a rebuild of the tables takes the new widths with it
    assert ex.tables().bits_mask == 0 and ex.call_bits() == (3, 3, 3)
    mixed = _experts((2, 3, 2))
    assert mixed.tables().bits_mask == 0b1100 and mixed.call_bits() == (0, 0, 0)


def test_call_bits_with_tables_set_by_a_loader():
    ex = _experts((4, 4))
    ex._tables = object()  # the checkpoint loader builds the tables itself
    assert ex.call_bits() == (4, 4, 4)


@pytest.fixture
def gemm_args(monkeypatch):
    """exl3.gemm on CPU tensors, with the library call recorded instead of made and the workspace that a decode call
    leaves on a stream (7) already there: returns the call's (a_had, workspace, workspace_bytes)."""
    seen = []
    real = exl3.lib

    class Lib:
        def __getattr__(self, name):
            return getattr(real, name)

        def hx_exl3_gemm(self, *a):
            seen.append(a[9:10] + a[11:13])
            return exl3.HX_GEMM_PATH_MFMA

    monkeypatch.setattr(exl3, "lib", Lib())
    monkeypatch.setattr(exl3, "_need", lambda *a: None)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    monkeypatch.setattr(exl3, "_workspaces", {})
    ws = exl3.workspace(1000, torch.device("cpu"), 7)
    exl3._workspaces[None, 7] = ws  # None: the index of a CPU tensor's device

    def call(M, a_had, K=128, N=128):
        w = exl3.GroupWords(torch.zeros((K // 16, N // 16, 32), dtype=torch.int16), torch.ones(K).half(),
                            torch.ones(N).half(), exl3.MUL1)
        x, y = torch.zeros((M, K)).half(), torch.zeros((M, N))
        exl3.gemm(y, x, w, M, N, K, 2, True, stream=7, a_had=a_had)
        return seen.pop()

    return call


@pytest.mark.parametrize("capturing", [False, True])
def test_gemm_with_a_had_passes_no_shared_buffer(gemm_args, monkeypatch, capturing):
    """M > 16 with the caller's a_had: no buffer of the module goes into the call (a captured graph would keep its
    address past the buffer's replacement), none is allocated and the device is not synchronized."""
    def refused(*a, **k):
        raise AssertionError("allocation or synchronisation")
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
    monkeypatch.setattr(torch.cuda, "synchronize", refused)
    a_had = torch.zeros((45, 128)).half()
    assert gemm_args(45, a_had) == (a_had.data_ptr(), None, 0)
    ws = exl3._workspaces[0, 7]
    assert gemm_args(45, None) == (None, ws.data_ptr(), ws.numel())
    assert gemm_args(3, a_had[:3])[1] == ws.data_ptr()  # the GEMV takes its counters and partials from it
    exl3._workspaces.clear()
    assert gemm_args(45, a_had) == (a_had.data_ptr(), None, 0) and not exl3._workspaces


def test_gemm_workspace_size_grows_with_m_alone():
    """The size that a caller has to provide is that of the largest M: counters and the M x K transformed input.  One
    workspace of that size serves every smaller M and every N (the K splits' memory is not part of it)."""
    size = exl3.lib.hx_exl3_gemm_workspace_size
    for K in (128, 4096, 8192):
        for N in (128, 12288, 24576):
            need = [size(M, N, K) for M in (17, 45, 128, 512, 1024, 2000)]
            assert need == sorted(need) and need == [65536 + (M * K * 2 + 255) // 256 * 256
                                                     for M in (17, 45, 128, 512, 1024, 2000)]
    assert exl3.lib.hx_exl3_gemm_extra_bytes() == 64 << 20


def test_gemm_under_capture_on_a_decode_workspace(gemm_args, monkeypatch):
    """A captured M > 16 call takes the workspace that a decode call left on the stream, if its input fits there, with
    the room for K splits that an eager call has; an eager call of that shape does not replace it."""
    ws = exl3._workspaces[0, 7]
    assert ws.numel() == (1 << 20) + exl3._GEMM_EXTRA
    for capturing in (True, False):
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
        for M, K, N in ((45, 4096, 12288), (17, 4096, 2048), (120, 4096, 512), (512, 512, 4096)):
            assert gemm_args(M, None, K, N) == (None, ws.data_ptr(), ws.numel())
            assert ws.numel() >= exl3.lib.hx_exl3_gemm_workspace_size(M, N, K) + exl3._GEMM_EXTRA
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    with pytest.raises(RuntimeError, match="before graph capture"):
        gemm_args(128, None, 4096, 512)  # 1 MiB of input and the counters: refused, as without K splits
