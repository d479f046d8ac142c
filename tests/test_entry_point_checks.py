"""What the entry points of libbr_hip.so decide on the host, before a kernel runs.

Calls are made by a child process that is shown no GPU, so that nothing can be
launched wherever the tests run: an accepted call ends in the runtime's error
for a missing device, a refused one in the library's own code (negative)."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# (kernel, slices, m, n, k, batch): products of the staged entry that reach every kernel in each of its forms -- whole
# and partial tiles, K of whole and of partial steps, slices of one length and not
PLANNED = [
    ("256", 1, 2048, 8192, 64, 1), ("256", 1, 4000, 4096, 64, 1), ("256", 1, 4000, 4096, 72, 1),
    ("256", 1, 1024, 1024, 256, 16), ("256", 4, 520, 4096, 8192, 1), ("256", 4, 4000, 520, 8200, 1),
    ("256x128", 1, 1000, 8192, 256, 1), ("256x128", 1, 1000, 8192, 136, 1), ("256x128", 8, 488, 2048, 8192, 1),
    ("256x128", 15, 488, 1000, 8200, 1), ("256x128", -2, 1024, 4096, 2048, 1), ("256x128", -2, 4000, 1000, 2048, 1),
    ("256x128 groups", 1, 1000, 2056, 4160, 2), ("256x128 groups", 4, 488, 4096, 8192, 1),
    ("128", 1, 2048, 520, 64, 1), ("128", 1, 488, 4096, 72, 1), ("128", 1, 488, 520, 192, 16),
    ("128", 16, 488, 520, 8192, 1), ("128", 8, 1000, 520, 4104, 1),
    ("128 half", 1, 488, 1000, 96, 1), ("128 half", 1, 2048, 2048, 2016, 1),
    ("flex 64", 1, 488, 4096, 256, 1), ("flex 64", 1, 488, 4096, 200, 1), ("flex 64", 4, 488, 512, 8192, 1),
    ("flex 64", 4, 488, 512, 8200, 1), ("flex 64 short", 1, 488, 4104, 2048, 1), ("flex 64 short", 1, 488, 4104, 520, 1),
    ("flex 32x64", 1, 488, 2048, 64, 1), ("flex 32x64", 1, 488, 2048, 72, 1), ("flex 32", 1, 488, 512, 72, 1),
    ("flex 32", 4, 64, 1024, 4096, 1), ("ring 64x128", 1, 488, 4096, 2048, 1), ("ring 64x128", 1, 488, 4096, 520, 1),
    ("ring 64x128", 4, 64, 4096, 8200, 1), ("flex 32", 4, 47, 896, 2688, 1), ("flex 32x64", 8, 41, 1152, 3456, 1),
]


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
    assert hip.gemm_kernel(0, 1, 512, 4096, 16384, staged=True)[1] > 1
    assert hip.gemm_kernel(0, 1, 512, 4096, 16384)[1] == 1   # nowhere to put partial sums
    with pytest.raises(hip.BrHipError):
        hip.gemm_kernel(0, 1, 0, 32, 64)


@pytest.mark.parametrize("m,n,k", [(4096, 4096, 1056), (8192, 2048, 1002), (16384, 4096, 96), (2048, 2048, 8160)])
def test_ragged_products_run_on_large_tiles_in_every_layout(m, n, k):
    from blackriver_amd import hip
    kernels = {hip.gemm_kernel(ta, tb, m, n, k, c_dtype=c) for ta in (0, 1) for tb in (0, 1) for c in (hip.F32, hip.F16)}
    assert len(kernels) == 1 and not {"flex", "ring"} & {name.split()[0] for name, _ in kernels}


@pytest.mark.parametrize("kernel,slices,m,n,k,batch", PLANNED)
def test_gemm_plan_reaches_every_kernel(kernel, slices, m, n, k, batch):
    from blackriver_amd import hip
    assert hip.gemm_kernel(0, 1, m, n, k, batch=batch, staged=True) == (kernel, slices)
    assert {kernel for kernel, *_ in PLANNED} == set(hip.GEMM_KERNELS)


@pytest.mark.parametrize("out", [(1 << 21) - 8, 1 << 21, (1 << 21) + 8, (1 << 26)])
def test_linear_gelu_takes_wide_outputs(out):
    assert answer("br_hip_linear_gelu(4096, 8192, None, 1 << 40, 1 << 41, 2, 300, %d, 32, None)" % out) > 0
