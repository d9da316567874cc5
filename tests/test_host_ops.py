"""The native host side of the operators (cut_amd/csrc/host_ops.cpp): what it refuses, before anything reaches the GPU."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")
from cut_amd import lib as L  # noqa: E402
from cut_amd import ops  # noqa: E402


def vectors(K=32, N=8):
    """A contiguous vector of K, Q8_0 blocks of [N, K], an output of N."""
    return torch.zeros(K), torch.zeros(N * K // 32 * 34, dtype=torch.uint8), torch.zeros(N)


class Short(C.Structure):
    _fields_ = [("p", C.c_void_p)]


# what ctypes refuses where a pointer to one of the two structures is wanted: other structures, and what is none at all
@pytest.mark.parametrize("bad,error", [("other", C.ArgumentError), (Short(), C.ArgumentError), (b"x" * 128, TypeError),
                                       (bytearray(8), TypeError), (1, TypeError), (torch.zeros(64), TypeError)])
def test_carry_and_rope_take_their_own_structure_only(bad, error):
    a, w, o = vectors()
    norm, rope = L.NormCarry(), L.RopeAppend()
    for_norm, for_rope = (rope, norm) if isinstance(bad, str) else (bad, bad)
    with pytest.raises(error):
        ops.matmul_gguf_carry(a, w, "Q8_0", 8, 32, o, for_norm)
    with pytest.raises(error):
        ops.matmul_gguf_argmax(a, w, "Q8_0", 8, 32, o, torch.zeros(1, dtype=torch.int32), carry=for_norm)
    with pytest.raises(error):
        ops.matmul_gguf_pair(a, w, "Q8_0", 8, o, w, "Q8_0", 8, o, 32, carry=for_norm)
    with pytest.raises(error):
        ops.matmul_gguf_pair(a, w, "Q8_0", 8, o, w, "Q8_0", 8, o, 32, carry=norm, rope=for_rope)


STUB = """
#include <poll.h>
#include <unistd.h>
int stub_fd = -1;
volatile int stub_entered = 0;
/* stands for a launch that waits until the other thread of the test has written to the pipe */
int cuthip_silu_mul(const void *a, int b, void *c, int d, unsigned n, void *s) {
  struct pollfd p = {stub_fd, POLLIN, 0};
  stub_entered = 1;
  return poll(&p, 1, 5000) == 1 ? 0 : 7;
}
/* the current stream, where there is no device */
struct stream { long a, b; } _ZN3c103hip19getCurrentHIPStreamEa(signed char d) { struct stream s = {0, 0}; return s; }
void *_ZNK3c103hip9HIPStream6streamEv(const void *s) { return 0; }
"""
WAITING = """
import ctypes, os, sys, threading, time
import torch
stub = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)   # ahead of the library for the extension that is loaded next
from cut_amd import ops
r, w = os.pipe()
ctypes.c_int.in_dll(stub, "stub_fd").value = r
entered = ctypes.c_int.in_dll(stub, "stub_entered")
def other():
    while not entered.value:
        time.sleep(0.001)
    os.write(w, b"x")
threading.Thread(target=other, daemon=True).start()
ops.silu_mul(torch.zeros(8), torch.zeros(4))
print("launched")
"""


def test_other_threads_run_while_a_launch_waits(tmp_path):
    """A launch that can only go on when another Python thread has run (a full queue behind a host callback): the GIL is not held
    across the C ABI.  The entry point is a stub that waits at most 5 s; no device is needed."""
    src, so = tmp_path / "stub.c", tmp_path / "stub.so"
    src.write_text(STUB)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-O1", str(src), "-o", str(so)])
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", WAITING, str(so)], cwd=root, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "launched" in r.stdout, r.stderr[-2000:]


M, K, N = 4, 32, 8
# outputs the launch would write past: too few rows, too narrow ones, the columns of a wider one, the wrong strides, rows in one piece
ROOM = {"rows": lambda n, **k: torch.zeros(M - 1, n, **k), "narrow": lambda n, **k: torch.zeros(M, n - 1, **k),
        "part": lambda n, **k: torch.zeros(M, n, **k)[:, :n - 1], "columns": lambda n, **k: torch.zeros(n, M, **k).t(),
        "every other": lambda n, **k: torch.zeros(M, 2 * n, **k)[:, ::2], "one block": lambda n, **k: torch.zeros(1, M * n, **k),
        "batch": lambda n, **k: torch.zeros(1, M, n, **k)}


@pytest.mark.parametrize("room", list(ROOM))
def test_outputs_without_room_are_refused(room):
    """Every operator that takes its output from the caller, before any launch."""
    out, wide = ROOM[room](N), ROOM[room](32 * N)
    a, w = torch.zeros(M, K), torch.zeros(M * N * K, dtype=torch.uint8)
    ids = torch.zeros(M, dtype=torch.int32)
    for call in (lambda: ops.matmul_gguf(a, w, "Q8_0", N, K, out=out), lambda: ops.matmul_gguf(a, w, "Q8_0", 2 * N, K, out=out, swiglu_pairs=True),
                 lambda: ops.matmul_gguf(a, w, "Q8_0", N, K, out=out, binary="add", d=out),
                 lambda: ops.matmul_sep(a, torch.zeros(K, N, dtype=torch.int8), torch.zeros(1, N, dtype=torch.float16), N, out=out),
                 lambda: ops.rmsnorm(torch.zeros(M, 2 * N)[:, :N], torch.zeros(N), 1e-5, out=out),
                 lambda: ops.matmul_dense_f16(a, torch.zeros(N, K, dtype=torch.float16), out=out), lambda: ops.matmul_q8_i8(a, w, N, K, out=out),
                 lambda: ops.embedding_col(ids, torch.zeros(32 * N, 4, dtype=torch.float16), None, 32 * N, 4, out=wide)):
        with pytest.raises(L.CutHipError):
            call()


@pytest.mark.gpu
@pytest.mark.parametrize("room", [r for r in ROOM if r != "batch"])   # (which is one piece of the right size here)
def test_dequantize_without_room_is_refused(room):
    w = torch.zeros(M * 34, dtype=torch.uint8, device="cuda")
    for dt, more in ((torch.float32, {}), (torch.float16, {}), (torch.float32, dict(dtype=torch.float16))):
        out = ROOM[room](32, device="cuda", dtype=dt)
        with pytest.raises(L.CutHipError):
            ops.dequantize(w, "Q8_0", M, 32, **({"dtype": dt} | more), out=out)


@pytest.mark.gpu
def test_rmsnorm_of_rows_with_a_pitch_makes_its_own_output():
    """The launch keeps the pitch of x: an output that the operator makes has it too."""
    x = torch.randn(5, 24, device="cuda")
    got = ops.rmsnorm(x[:, :16], torch.ones(16, device="cuda"), 1e-5)
    want = x[:, :16] / torch.sqrt((x[:, :16].double() ** 2).mean(-1, keepdim=True) + 1e-5)
    assert got.shape == (5, 16)
    torch.testing.assert_close(got.double(), want, rtol=2e-6, atol=1e-7)


def test_outputs_of_other_types_are_refused():
    a, w = torch.zeros(M, K), torch.zeros(M * N * K, dtype=torch.uint8)
    for dt in (torch.bfloat16, torch.int16, torch.int8, torch.float64):
        with pytest.raises(L.CutHipError):
            ops.matmul_gguf(a, w, "Q8_0", N, K, out_dtype=dt)
        with pytest.raises(L.CutHipError):
            ops.matmul_gguf(a, w, "Q8_0", N, K, out=torch.zeros(M, N, dtype=dt))
        with pytest.raises(L.CutHipError):
            ops.matmul_sep(a, torch.zeros(K, N, dtype=torch.int8), torch.zeros(1, N, dtype=torch.float16), N, out=torch.zeros(M, N, dtype=dt))


def test_vectors_without_room_are_refused():
    a, w, o = vectors()
    x = torch.zeros(64)
    with pytest.raises(L.CutHipError):
        ops.silu_mul(x, torch.zeros(33))
    with pytest.raises(L.CutHipError):
        ops.attn_decode(x, x.half().view(1, 64), x.half().view(1, 64), torch.zeros(2, dtype=torch.int32), 1, 1, 64, 1.0,
                        torch.zeros(4096, dtype=torch.uint8), torch.zeros(63))
    with pytest.raises(L.CutHipError):
        ops.repetition_penalty(x, x, out=torch.zeros(63))
    with pytest.raises(L.CutHipError):
        ops.embedding_rows(w, "Q8_0", torch.zeros(2, dtype=torch.int32), 8, 32, torch.zeros(1, 64))


def test_formats_are_names_or_numbers():
    """As int() takes them; what follows is another check's error."""
    raw = torch.zeros(144, dtype=torch.uint8)
    for fmt in (2, 2.0, np.int64(2), np.float32(2.0), torch.tensor(2), True, "Q4_K"):
        with pytest.raises(L.CutHipError, match="device tensor"):
            ops.dequantize(raw, fmt, 1, 256)
        assert ops.n_bytes(fmt, 1, 256) == 144
    with pytest.raises(L.CutHipError, match="unknown quantization format"):
        ops.dequantize(raw, "Q5_K", 1, 256)
    for fmt, error in ((None, TypeError), (float("nan"), ValueError), (2.0j, TypeError)):
        with pytest.raises(error):
            ops.dequantize(raw, fmt, 1, 256)


@pytest.mark.parametrize("n", [2 ** 62, 2 ** 63 - 1, -1])
def test_row_counts_that_no_tensor_holds(n):
    """2^62 rows of 34 bytes are a negative number in 64 bits; the launch takes the lower 32 of what passes."""
    a, w, _ = vectors()
    with pytest.raises(L.CutHipError, match="too small"):
        ops.matmul_gguf_pair(a, w, "Q8_0", n, None, w, "Q8_0", n, None, 32, rope=L.RopeAppend())
