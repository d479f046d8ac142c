"""What the entry points of libbr_hip.so decide on the host, before a kernel runs.

Calls are made by a child process that is shown no GPU, so that nothing can be
launched wherever the tests run: an accepted call ends in the runtime's error
for a missing device, a refused one in the library's own code (negative)."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def answer(call):
    """Return code of `L.<call>`, made without a GPU."""
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", ROCR_VISIBLE_DEVICES="-1")
    text = "from blackriver_amd import hip; L = hip.load(); print('answer', L.%s)" % call
    out = subprocess.run([sys.executable, "-c", text], cwd=ROOT, env=env, timeout=60, capture_output=True, text=True)
    assert out.returncode == 0, out
    return int(out.stdout.split("answer")[1])


@pytest.mark.parametrize("call", [
    "br_hip_softmax_fwd(4097, 8192, 4, 8, None)",
    "br_hip_softmax_fwd(4096, 8194, 4, 7, None)",
    "br_hip_softmax_bwd(4096, 8192, 16387, 4, 8, None)",
    "br_hip_alibi_masked_softmax_fwd(4096, 8193, 16384, 32768, 1, 1, 4, 4, None)",
])
def test_softmax_takes_addresses_of_any_alignment(call):
    assert answer(call) > 0


@pytest.mark.parametrize("hidden", [65535 * 256 + 1, 65535 * 1024 + 4])
def test_embedding_backward_takes_rows_of_any_length(hidden):
    assert answer("br_hip_embedding_scatter_add(4096, 8192, 16384, 2, %d, 4, 1.0, None)" % hidden) > 0


def test_gemm_kernel_names_the_kernel_of_a_product():
    from blackriver_amd import hip
    assert hip.gemm_kernel(0, 1, 4096, 4096, 4096)[0] == "256"
    assert hip.gemm_kernel(0, 1, 32, 32, 64) == ("flex 32", 1)
    kernel, slices = hip.gemm_kernel(0, 1, 512, 4096, 16384, staged=True)
    assert kernel in hip.GEMM_KERNELS and slices > 1
    assert hip.gemm_kernel(0, 1, 512, 4096, 16384)[1] == 1   # nowhere to put partial sums
    with pytest.raises(hip.BrHipError):
        hip.gemm_kernel(0, 1, 0, 32, 64)


@pytest.mark.parametrize("m,n,k", [(4096, 4096, 1056), (8192, 2048, 1002), (16384, 4096, 96), (2048, 2048, 8160)])
def test_ragged_products_run_on_large_tiles_in_every_layout(m, n, k):
    from blackriver_amd import hip
    kernels = {hip.gemm_kernel(ta, tb, m, n, k, c_dtype=c) for ta in (0, 1) for tb in (0, 1) for c in (hip.F32, hip.F16)}
    assert len(kernels) == 1 and not {"flex", "ring"} & {name.split()[0] for name, _ in kernels}
