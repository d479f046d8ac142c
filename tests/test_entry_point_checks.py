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


# (kernel, waves along K, m, n, k, batch): fp32 products that reach every kernel in each of its forms -- K of one walk's parts added
# apart (up to 256 k-values a wave) and folded, whole and partial steps, sizes that are loaded in quads and value by value
FP32_PLANNED = [
    ("flex 32", 4, 33, 36, 40, 2), ("flex 32", 4, 31, 65, 7, 2), ("flex 32", 4, 520, 1028, 1024, 1), ("flex 32", 4, 1000, 1100, 2120, 1),
    ("flex 32", 8, 200, 768, 512, 1), ("flex 32", 8, 31, 1025, 1025, 1), ("flex 32", 8, 64, 256, 4100, 1),
    ("flex 32x64", 4, 1000, 1028, 36, 4), ("flex 32x64", 4, 501, 501, 65, 16), ("flex 32x64", 4, 1000, 2100, 2100, 1),
    ("flex 32x64", 8, 500, 520, 512, 1), ("flex 32x64", 8, 333, 1025, 1025, 1), ("flex 32x64", 8, 500, 520, 2052, 1),
    ("flex 64", 4, 500, 2049, 200, 4), ("flex 64", 4, 500, 4096, 516, 1), ("flex 64", 4, 500, 2048, 1025, 2), ("flex 64", 4, 500, 2048, 2052, 1),
    ("128", 4, 512, 512, 72, 48), ("128", 4, 256, 384, 65, 128),
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


@pytest.mark.parametrize("kernel,waves,m,n,k,batch", FP32_PLANNED)
def test_fp32_products_run_on(kernel, waves, m, n, k, batch):
    from blackriver_amd import hip
    assert hip.gemm_fp32_kernel(m, n, k, batch) == (kernel, waves)


@pytest.mark.parametrize("m,n", [(512, 1024), (32, 16384), (2048, 256), (513, 992)])
def test_eight_waves_walk_along_k_where_a_cu_has_one_small_tile(m, n):
    """Up to 256 of the small tiles, from a K of 512 on."""
    from blackriver_amd import hip
    for k in (511, 512, 1024, 3071, 3072, 8192):
        kernel, waves = hip.gemm_fp32_kernel(m, n, k)
        tiles = -(-m // 32) * -(-n // {"flex 32": 32, "flex 32x64": 64}[kernel])
        assert waves == (8 if k >= 512 and tiles <= 256 else 4)


@pytest.mark.parametrize("n,inn,out,name", [(64, 2048, 6144, "flex 32"), (200, 2048, 2048, "flex 32x64"), (250, 2048, 3072, None),
                                            (65, 2048, 6144, None)])   # on 64 x 64 tiles; many whole 128 x 128 tiles: two launches
def test_fp32_pairs_that_cost_about_two_launches_by_the_rule(n, inn, out, name):
    from blackriver_amd import hip
    kernel = hip.load().br_hip_gemm_pair_kernel(out, inn, n, 1, n, inn, out, 1, hip.GEMM_F32)
    assert kernel == (-1 if name is None else hip.GEMM_KERNELS.index(name))


def on_wide_tiles(*products):
    """Whether two products, the weight gradient's (trans_a, trans_b, m, n, k) first, share a launch with wide tiles: by their sizes, and
    as operands in either order."""
    import ctypes
    from blackriver_amd import hip
    lib, wide = hip.load(), 10   # BR_GEMM_PAIR_WIDE
    (_, _, m1, n1, k1), (_, _, m2, n2, k2) = products
    by_size = lib.br_hip_gemm_pair_kernel(m1, n1, k1, 1, m2, n2, k2, 1, hip.GEMM_F16)
    made = [hip.Product(ta, tb, m, n, k, 1.0, 64 * MB, hip.F16, m if ta else k, 0, at, hip.F16, k if tb else n, 0, 2 * at, hip.F32, n, 0, 1)
            for at, (ta, tb, m, n, k) in zip((256 * MB, 1024 * MB), products)]
    joined = [lib.br_hip_gemm_pair_joined(ctypes.byref(a), ctypes.byref(b), None, None, hip.GEMM_F16, None, 0)
              for a, b in (made, made[::-1])]
    assert joined[0] == joined[1] == by_size
    return by_size == wide


@pytest.mark.parametrize("n,inn,out,wide", [(78, 1024, 4096, True), (200, 512, 2048, True), (32, 8192, 400, True), (256, 512, 2048, True),
                                            # more tokens than outputs: K of the gradient is the longer one
                                            (400, 8192, 32, False), (256, 8192, 32, False), (2048, 512, 128, False),
                                            (4096, 512, 256, False), (1024, 4096, 64, False)])
def test_wide_pairs_are_priced_with_the_weight_gradient_on_the_wide_tiles(n, inn, out, wide):
    assert on_wide_tiles((1, 0, out, inn, n), (0, 0, n, inn, out)) == wide


@pytest.mark.parametrize("t,hd", [(776, 64), (1024, 64), (1024, 128), (400, 64)])
def test_a_heads_backward_products_keep_off_wide_tiles(t, hd):
    assert not on_wide_tiles((1, 0, t, hd, t), (0, 1, t, t, hd))   # of the values and the scores
    assert not on_wide_tiles((1, 0, t, hd, t), (0, 0, t, hd, t))   # of the keys and the queries


@pytest.mark.parametrize("out", [(1 << 21) - 8, 1 << 21, (1 << 21) + 8, (1 << 26)])
def test_linear_gelu_takes_wide_outputs(out):
    assert answer("br_hip_linear_gelu(4096, 8192, None, 1 << 40, 1 << 41, 2, 300, %d, 32, None)" % out) > 0


MB = 1 << 20
# addresses, a megabyte and more from each other: output gradient, input, weight, their gradients, sums
PLACES = {"dy": 16 * MB, "x": 32 * MB, "w": 48 * MB, "dw": 64 * MB, "dx": 80 * MB, "sums.x": 96 * MB, "sums.out": 112 * MB,
          "partials": 128 * MB, "out0": 144 * MB, "out1": 160 * MB, "ws": 176 * MB}


def pair_joined(compute, x_f32=False, **moved):
    """Kernel of a linear layer's backward products (64 tokens, 256 -> 256) with column sums and two arrays of partial sums
    beside them, or -1; `moved`: tensors at other addresses."""
    import ctypes
    from blackriver_amd import hip
    at = dict(PLACES, **{k.replace("_", "."): v for k, v in moved.items()})
    dt = {hip.GEMM_F16: hip.F16, hip.GEMM_BF16: hip.BF16, hip.GEMM_F32: hip.F32}[compute]
    xt = hip.F32 if x_f32 else dt
    dw = hip.Product(1, 0, 256, 256, 64, 1.0, at["dy"], dt, 256, 0, at["x"], xt, 256, 0, at["dw"], hip.F32, 256, 0, 1)
    dx = hip.Product(0, 0, 64, 256, 256, 1.0, at["dy"], dt, 256, 0, at["w"], dt, 256, 0, at["dx"], dt, 256, 0, 1)
    sums = hip.ColumnSums(at["sums.x"], dt, at["sums.out"], 40, 256, 1.0, None, 0)
    later = hip.PartialSums(at["partials"], 2, 7, 256, (ctypes.c_void_p * 3)(at["out0"], at["out1"]), 1.0)
    lib, pair = hip.load(), (ctypes.byref(dw), ctypes.byref(dx))
    return lib.br_hip_gemm_pair_joined(*pair, ctypes.byref(sums), ctypes.byref(later), compute, at["ws"],
                                       lib.br_hip_gemm_pair_workspace(*pair, compute))


@pytest.mark.parametrize("compute", [0, 1, 2])
def test_two_products_and_sums_that_do_not_meet_are_one_launch(compute):
    from blackriver_amd import hip
    assert {hip.GEMM_F16, hip.GEMM_BF16, hip.GEMM_F32} == {0, 1, 2}
    assert pair_joined(compute) == hip.load().br_hip_gemm_pair_kernel(256, 256, 64, 1, 64, 256, 256, 1, compute) >= 0
    assert pair_joined(compute, x_f32=True) >= 0
    assert pair_joined(compute, sums_x=PLACES["dy"]) >= 0            # a bias gradient: both are read
    assert pair_joined(compute, x_f32=True, dx=PLACES["x"]) == (-1 if compute == 2 else pair_joined(compute))   # x is copied first


@pytest.mark.parametrize("compute", [0, 1, 2])
@pytest.mark.parametrize("moved,onto", [
    ("dx", "dw"), ("dx", "dy"), ("dx", "x"), ("dw", "w"), ("dw", "dy"), ("sums_out", "dy"), ("sums_out", "x"), ("sums_out", "dw"),
    ("dx", "sums.x"), ("sums_out", "partials"), ("sums_out", "out0"), ("out0", "sums.x"), ("out1", "sums.x"), ("out0", "partials"),
    ("out1", "out0"), ("out0", "x"), ("out0", "dy"), ("out1", "w"), ("out0", "dw"), ("out1", "dx"), ("dw", "partials")])
def test_two_products_and_sums_that_meet_keep_their_order(moved, onto, compute):
    assert pair_joined(compute, **{moved: PLACES[onto] + 512}) == -1
    if onto == "x" and moved != "dx":   # also where x is read by way of a copy
        assert pair_joined(compute, x_f32=True, **{moved: PLACES[onto] + 512}) == -1
