"""Which calls variant 0 of the batched GEMM gives to the kernels that need
vb_gemm_scratch's workspace: more than vb_gemm_workspace asks for is the sign
of it.  The calls here ran slower there than on the kernel they had left, or
gained most (MI355X; the figures stand at the rules)."""
import pytest

from vibeblade_amd import _lib, ggml

Q4K, Q5K, Q6K, Q80 = (ggml.GGML_TYPE_Q4_K, ggml.GGML_TYPE_Q5_K, ggml.GGML_TYPE_Q6_K, ggml.GGML_TYPE_Q8_0)
F32, F16 = 0, 1


def _more(qtype, xdt, m, n, k):
    lib = _lib.load()
    need, best = (f(m, n, k, qtype, xdt, 0) for f in (lib.vb_gemm_workspace, lib.vb_gemm_scratch))
    assert best >= need >= 0
    return best > need


@pytest.mark.parametrize("qtype,xdt,m,n,k", [(Q5K, F16, 256, 14336, 3072), (Q5K, F16, 17, 14336, 3072),
                                             (Q5K, F16, 193, 29702, 2304), (Q5K, F16, 224, 128256, 2304),
                                             (Q5K, F16, 33, 4096, 4096), (Q80, F16, 256, 8192, 3072),
                                             (Q80, F16, 33, 4096, 4096), (Q80, F16, 224, 32768, 2048),
                                             (Q4K, F16, 224, 4096, 5120), (Q4K, F16, 17, 6144, 8192),
                                             (Q4K, F16, 33, 14336, 8192), (Q6K, F16, 256, 4096, 5120),
                                             (Q6K, F16, 33, 4096, 6144), (Q5K, F32, 256, 14336, 3072)])
def test_wreg_leaves(qtype, xdt, m, n, k):
    assert not _more(qtype, xdt, m, n, k)


@pytest.mark.parametrize("qtype,xdt,m,n,k", [(Q4K, F16, 100, 4096, 14336), (Q4K, F16, 17, 4096, 14336),
                                             (Q5K, F16, 64, 14336, 4096), (Q6K, F16, 128, 4096, 4096),
                                             (Q80, F16, 256, 4096, 14336), (Q4K, F32, 33, 1024, 4096),
                                             (Q80, F32, 8, 4096, 14336), (Q6K, F32, 256, 14336, 8192)])
def test_wreg_takes(qtype, xdt, m, n, k):
    assert _more(qtype, xdt, m, n, k)
