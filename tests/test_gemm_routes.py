"""Which calls variant 0 of the batched GEMM gives to the kernels that need
vb_gemm_scratch's workspace: more than vb_gemm_workspace asks for is the sign
of it.  The calls here ran slower there than on the kernel they had left, or
gained most (MI355X; the figures stand at the rules)."""
import pytest

from vibeblade_amd import _lib, ggml

Q4K, Q5K, Q6K, Q80 = (ggml.GGML_TYPE_Q4_K, ggml.GGML_TYPE_Q5_K, ggml.GGML_TYPE_Q6_K, ggml.GGML_TYPE_Q8_0)
Q40, Q50 = ggml.GGML_TYPE_Q4_0, ggml.GGML_TYPE_Q5_0
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
                                             (Q6K, F16, 33, 4096, 6144), (Q5K, F32, 256, 14336, 3072),
                                             (Q4K, F16, 17, 1536, 8192), (Q4K, F32, 17, 1536, 4864)])
def test_wreg_leaves(qtype, xdt, m, n, k):
    assert not _more(qtype, xdt, m, n, k)


@pytest.mark.parametrize("qtype,xdt,m,n,k", [(Q4K, F16, 100, 4096, 14336), (Q4K, F16, 17, 4096, 14336),
                                             (Q5K, F16, 64, 14336, 4096), (Q6K, F16, 128, 4096, 4096),
                                             (Q80, F16, 256, 4096, 14336), (Q4K, F32, 33, 1024, 4096),
                                             (Q80, F32, 8, 4096, 14336), (Q6K, F32, 256, 14336, 8192)])
def test_wreg_takes(qtype, xdt, m, n, k):
    assert _more(qtype, xdt, m, n, k)


@pytest.mark.parametrize("qtype,xdt,m,n,k", [(Q80, F32, 257, 3000, 1536), (Q5K, F32, 300, 2048, 2048),
                                             (Q6K, F32, 300, 2048, 2048), (Q4K, F32, 257, 4096, 1024),
                                             (Q4K, F32, 513, 9871, 4096), (Q4K, F32, 1024, 8192, 1024),
                                             (Q5K, F16, 2048, 4096, 5120), (Q40, F16, 1024, 8191, 4096),
                                             (Q40, F32, 300, 3000, 1536)])
def test_packed_x_leaves(qtype, xdt, m, n, k):
    assert not _more(qtype, xdt, m, n, k)


@pytest.mark.parametrize("qtype,xdt,m,n,k", [(Q6K, F32, 777, 4096, 14336), (Q4K, F32, 512, 14336, 4096),
                                             (Q4K, F32, 600, 1000, 4096), (Q80, F32, 300, 14336, 512),
                                             (Q5K, F32, 400, 11008, 2048), (Q40, F32, 257, 32768, 2048)])
def test_packed_x_takes(qtype, xdt, m, n, k):
    assert _more(qtype, xdt, m, n, k)
