"""The native host side of the operators (cut_amd/csrc/host_ops.cpp): what it refuses, before anything reaches the GPU."""
import ctypes as C

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
