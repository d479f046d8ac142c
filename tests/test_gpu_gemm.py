"""MFMA GEMM kernel against fp64 products through the C ABI: every operand
layout, storage type and compute type, odd sizes, batching, bias, alpha and
accumulation.  Tolerances: 2e-2 relative for fp16 / bf16 operands, 1e-5 for
the fp32-operand kernel."""
import ctypes
import math

import numpy as np
import pytest
import torch

from conftest import assert_close
from gpu_util import BF16, F16, F32, call, dev, empty, host, ptr, stream
from blackriver_amd import hip
from test_entry_point_checks import FP32_PLANNED, PLANNED

pytestmark = pytest.mark.gpu

TORCH_T = {F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}


def to_dev(a, dtype):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda().to(TORCH_T[dtype]).contiguous()


def to_host64(t):
    torch.cuda.synchronize()
    return t.detach().float().cpu().numpy().astype(np.float64)


def run_gemm(ta, tb, m, n, k, a, b, a_dt, b_dt, c_dt, compute, alpha=1.0, bias=None, c0=None, batch=1):
    da, db_ = to_dev(a, a_dt), to_dev(b, b_dt)
    if c0 is not None:
        c = to_dev(c0, c_dt)
    else:
        c = torch.full((batch, m, n), float("nan"), dtype=TORCH_T[c_dt], device="cuda")
    dbias = dev(bias) if bias is not None else None
    lda = m if ta else k
    ldb = k if tb else n
    call("br_hip_gemm", int(ta), int(tb), m, n, k, alpha, ptr(da), a_dt, lda, m * k, ptr(db_), b_dt, ldb, n * k,
         1 if c0 is not None else 0, ptr(c), c_dt, n, m * n, ptr(dbias), batch, compute, stream())
    # reference from the operands as the kernel saw them (after storage rounding)
    A = to_host64(da).reshape(batch, *((k, m) if ta else (m, k)))
    B = to_host64(db_).reshape(batch, *((n, k) if tb else (k, n)))
    if ta:
        A = A.transpose(0, 2, 1)
    if tb:
        B = B.transpose(0, 2, 1)
    ref = alpha * np.matmul(A, B)
    if bias is not None:
        ref = ref + bias.astype(np.float64)[None, None, :]
    if c0 is not None:
        ref = ref + to_host64(to_dev(c0, c_dt)).reshape(batch, m, n)
    return to_host64(c).reshape(batch, m, n), ref


def run_gemm_staged(ta, tb, m, n, k, a, b, a_dt, b_dt, c_dt, compute, batch=1, ws_bytes=None, bias=None):
    """br_hip_gemm_staged and br_hip_gemm on the same device operands."""
    da, db_ = to_dev(a, a_dt), to_dev(b, b_dt)
    dbias = dev(bias) if bias is not None else None
    lda = m if ta else k
    ldb = k if tb else n
    need = hip.load().br_hip_gemm_staged_workspace(int(ta), int(tb), m, n, k, a_dt, b_dt, batch)
    if ws_bytes is None:
        ws_bytes = need
    ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device="cuda")
    outs = []
    for staged in (True, False):
        c = torch.full((batch, m, n), float("nan"), dtype=TORCH_T[c_dt], device="cuda")
        common = (int(ta), int(tb), m, n, k, 1.0, ptr(da), a_dt, lda, m * k, ptr(db_), b_dt, ldb, n * k, 0, ptr(c),
                  c_dt, n, m * n, ptr(dbias), batch, compute)
        if staged:
            call("br_hip_gemm_staged", *common, ptr(ws), ws_bytes, stream())
        else:
            call("br_hip_gemm", *common, stream())
        outs.append(to_host64(c).reshape(batch, m, n))
    return outs[0], outs[1], need


def operands(rng, ta, tb, m, n, k, batch=1):
    a = rng.standard_normal((batch,) + ((k, m) if ta else (m, k))).astype(np.float32)
    b = rng.standard_normal((batch,) + ((n, k) if tb else (k, n))).astype(np.float32)
    return a, b


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("a_dt,b_dt,c_dt", [(F32, F32, F32), (F32, F16, F32), (F16, F16, F16), (F16, F32, F32)])
def test_gemm_f16_layouts_and_storage_types(ta, tb, a_dt, b_dt, c_dt):
    rng = np.random.default_rng(0)
    m, n, k = 256, 384, 160
    print("case ta=%d tb=%d dtypes=%s" % (ta, tb, (a_dt, b_dt, c_dt)), flush=True)
    a, b = operands(rng, ta, tb, m, n, k)
    got, ref = run_gemm(ta, tb, m, n, k, a, b, a_dt, b_dt, c_dt, hip.GEMM_F16)
    assert_close(got, ref, 2e-2, "gemm f16")
    # typical error is far below the bound: fp16 operand rounding only
    assert np.sqrt(np.mean((got - ref) ** 2)) < 3e-3 * np.sqrt(np.mean(ref ** 2)) + (1e-2 if c_dt == F16 else 0)


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (5, 7, 3), (33, 65, 17), (130, 129, 40), (12, 12, 16), (128, 128, 32),
                                   (200, 100, 1000)])
def test_gemm_odd_sizes(ta, tb, m, n, k):
    rng = np.random.default_rng(1)
    print("case ta=%d tb=%d m=%d n=%d k=%d" % (ta, tb, m, n, k), flush=True)
    a, b = operands(rng, ta, tb, m, n, k)
    got, ref = run_gemm(ta, tb, m, n, k, a, b, F32, F32, F32, hip.GEMM_F16)
    assert_close(got, ref, 2e-2, "gemm f16 odd sizes")
    got, ref = run_gemm(ta, tb, m, n, k, a, b, F32, F32, F32, hip.GEMM_F32)
    assert_close(got, ref, 1e-5, "gemm fp32 odd sizes")


def test_gemm_bias_alpha_accumulate_batched():
    rng = np.random.default_rng(2)
    m, n, k, batch = 96, 80, 64, 5
    a, b = operands(rng, 0, 1, m, n, k, batch)
    bias = rng.standard_normal(n).astype(np.float32)
    c0 = rng.standard_normal((batch, m, n)).astype(np.float32)
    for compute, tol in ((hip.GEMM_F16, 2e-2), (hip.GEMM_F32, 1e-5)):
        got, ref = run_gemm(0, 1, m, n, k, a, b, F32, F32, F32, compute, alpha=0.25, bias=bias, c0=c0, batch=batch)
        assert_close(got, ref, tol, "alpha/bias/accumulate/batch compute=%d" % compute)


def test_gemm_bf16():
    rng = np.random.default_rng(3)
    m, n, k = 192, 160, 96
    for ta, tb in ((0, 1), (1, 0)):
        a, b = operands(rng, ta, tb, m, n, k)
        got, ref = run_gemm(ta, tb, m, n, k, a, b, BF16, F32, BF16, hip.GEMM_BF16)
        assert_close(got, ref, 2e-2, "gemm bf16")


def test_gemm_fp32_kernel_is_fp32_faithful_at_block_sizes():
    rng = np.random.default_rng(4)
    m, n, k = 512, 1024, 4096
    a, b = operands(rng, 0, 1, m, n, k)
    got, ref = run_gemm(0, 1, m, n, k, a, b, F32, F32, F32, hip.GEMM_F32)
    assert_close(got, ref, 1e-5, "fp32 gemm, k=4096")


# Products of the plain entry that run on each direct-to-LDS tile (256x256, 256x128, 128x128 with K steps of 64 and of
# 32), with rows / columns that do not fill the last tile, several batch entries and a single K step.  The kernel is
# asserted: which sizes go where follows from a table of fitted costs.
DTL_SHAPES = [
    ("256", 1024, 1024, 128, 16),
    ("256", 1000, 1024, 192, 16),
    ("256x128", 1024, 1024, 256, 8),
    ("256x128", 1000, 8192, 256, 1),
    ("128", 128, 51200, 64, 1),
    ("128", 488, 520, 192, 16),
    ("128 half", 264, 392, 96, 24),
    ("256", 2048, 4096, 64, 2),
    ("128", 2048, 2056, 64, 1),
]


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("name,m,n,k,batch", DTL_SHAPES)
def test_gemm_direct_to_lds_kernel(ta, tb, name, m, n, k, batch):
    rng = np.random.default_rng(5)
    print("case %s ta=%d tb=%d m=%d n=%d k=%d batch=%d" % (name, ta, tb, m, n, k, batch), flush=True)
    assert hip.gemm_kernel(ta, tb, m, n, k, batch=batch) == (name, 1)
    a, b = operands(rng, ta, tb, m, n, k, batch)
    got, ref = run_gemm(ta, tb, m, n, k, a, b, F16, F16, F32, hip.GEMM_F16, batch=batch)
    assert_close(got, ref, 2e-2, "dtl gemm " + name)
    assert np.sqrt(np.mean((got - ref) ** 2)) < 1e-5 * np.sqrt(np.mean(ref ** 2)) * np.sqrt(k)


def test_gemm_direct_to_lds_epilogue_and_types():
    rng = np.random.default_rng(6)
    m, n, k, batch = 320, 256, 256, 2
    a, b = operands(rng, 0, 1, m, n, k, batch)
    bias = rng.standard_normal(n).astype(np.float32)
    c0 = rng.standard_normal((batch, m, n)).astype(np.float32)
    got, ref = run_gemm(0, 1, m, n, k, a, b, F16, F16, F32, hip.GEMM_F16, alpha=0.5, bias=bias, c0=c0, batch=batch)
    assert_close(got, ref, 2e-2, "dtl alpha/bias/accumulate")
    got, ref = run_gemm(0, 1, m, n, k, a, b, F16, F16, F16, hip.GEMM_F16, bias=bias, batch=batch)
    assert_close(got, ref, 2e-2, "dtl fp16 output")
    for ta, tb in ((0, 1), (0, 0), (1, 0), (1, 1)):
        a, b = operands(rng, ta, tb, m, n, k, batch)
        got, ref = run_gemm(ta, tb, m, n, k, a, b, BF16, BF16, BF16, hip.GEMM_BF16, batch=batch)
        assert_close(got, ref, 2e-2, "dtl bf16")


def test_gemm_direct_to_lds_at_linear_layer_shape():
    """BLOOM-7B1 h -> 4h at a quarter of the token count; checked on a sample
    of rows against fp64 and, for every element, through linearity:
    (A1 + A2) B == A1 B + A2 B up to fp32 accumulation error when the sums are
    exact in fp16."""
    rng = np.random.default_rng(7)
    m, n, k = 512, 16384, 4096
    a1 = rng.integers(-8, 9, (1, m, k)).astype(np.float32)
    a2 = rng.integers(-8, 9, (1, m, k)).astype(np.float32)
    b = rng.integers(-4, 5, (1, n, k)).astype(np.float32)
    c1, _ = run_gemm(0, 1, m, n, k, a1, b, F16, F16, F32, hip.GEMM_F16)
    c2, _ = run_gemm(0, 1, m, n, k, a2, b, F16, F16, F32, hip.GEMM_F16)
    c12, ref = run_gemm(0, 1, m, n, k, a1 + a2, b, F16, F16, F32, hip.GEMM_F16)
    # small integers: every product and partial sum is exact in fp32
    assert np.array_equal(c12, ref)
    assert np.array_equal(c1 + c2, c12)


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k,c_dt", [
    (2048, 8192, 192, F32),     # 256 tiles: one per workgroup, three K steps
    (2048, 16384, 128, F16),    # 512 tiles: two per workgroup, 16-bit C
    (3072, 16384, 64, F32),     # 768 tiles of a single K step
    (2816, 10240, 192, F32),    # 440 tiles: 55 per XCD for 32 workgroups, 23 of them walk twice
])
def test_gemm_workgroups_that_walk_the_tiles(ta, tb, m, n, k, c_dt):
    """Plain products (no bias, nothing accumulated) of 256 or more interior
    256 x 256 tiles run on 256 workgroups that each walk several tiles, loading
    the next tile's first K stages ahead of the current tile's stores.  Against
    fp64, and for an fp32 C bit for bit against the same product with a bias of
    zeros, which takes the one-workgroup-per-tile kernel."""
    rng = np.random.default_rng(31)
    print("case ta=%d tb=%d m=%d n=%d k=%d c_dt=%d" % (ta, tb, m, n, k, c_dt), flush=True)
    a, b = operands(rng, ta, tb, m, n, k)
    assert hip.gemm_kernel(ta, tb, m, n, k, c_dt) == ("256", 1)
    got, ref = run_gemm(ta, tb, m, n, k, a, b, F16, F16, c_dt, hip.GEMM_F16, alpha=0.5)
    assert_close(got, ref, 2e-2, "walking workgroups")
    per_tile, _ = run_gemm(ta, tb, m, n, k, a, b, F16, F16, c_dt, hip.GEMM_F16, alpha=0.5, bias=np.zeros(n, np.float32))
    assert np.array_equal(got, per_tile)


@pytest.mark.parametrize("dt", [F16, BF16])
@pytest.mark.parametrize("ta", [1, 0])
@pytest.mark.parametrize("m,n,k", [(4096, 4096, 64), (4000, 4096, 64), (8192, 8200, 128), (8184, 8192, 192), (6144, 2048, 768),
                                   (16384, 4096, 512), (4096, 16384, 512), (16384, 8192, 64),
                                   (4096, 4096, 128), (4000, 8184, 128), (4000, 8184, 64), (2048, 8160, 128), (8192, 2048, 768), (3000, 5000, 192)])
@pytest.mark.parametrize("gap", [32, 4])
def test_gemm_two_workgroups_to_a_cu_for_a_short_k(ta, dt, m, n, k, gap):
    """Plain products with an fp32 C of rows on 128-byte lines, a row-contiguous B and K up to 768 run on tiles of 128 x 256,
    two workgroups to a CU: whole and partial ones, four K steps and many, into a C whose rows lie apart.  Rows off such lines,
    or all of C in one round of 256 x 256 tiles and a pitch of 32 KB or K = 64: on 256 x 256 tiles.  Small integers, so exact."""
    gap += -n % 32
    assert hip.gemm_kernel(ta, 0, m, n, k, staged=True)[0] == "256"
    print("case ta=%d m=%d n=%d k=%d dt=%d" % (ta, m, n, k, dt), flush=True)
    torch.manual_seed(m + k)
    a = torch.randint(-3, 4, (k, m) if ta else (m, k), device="cuda").to(TORCH_T[dt])
    b = torch.randint(-2, 3, (k, n), device="cuda").to(TORCH_T[dt])
    c = torch.full((m, n + gap), float("nan"), device="cuda")
    call("br_hip_gemm", ta, 0, m, n, k, 0.5, ptr(a), dt, m if ta else k, 0, ptr(b), dt, n, 0, 0, ptr(c), F32, n + gap, 0, None, 1,
         hip.GEMM_F16 if dt == F16 else hip.GEMM_BF16, stream())
    torch.cuda.synchronize()
    assert torch.equal(c[:, :n], 0.5 * ((a.t() if ta else a).float() @ b.float())) and c[:, n:].isnan().all()


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("gap,off", [(32, 0), (4, 0), (0, 4)])
def test_gemm_workgroups_that_walk_into_a_c_of_any_rows(ta, tb, gap, off):
    """Rows of C that start on 128-byte lines, that do not, and a C that does not: four tiles a workgroup.  Exact."""
    m, n, k = 4096, 16384, 832   # 256 MB: stored past the caches in whole lines
    print("case ta=%d tb=%d gap=%d off=%d" % (ta, tb, gap, off), flush=True)
    torch.manual_seed(gap)
    a = torch.randint(-3, 4, (k, m) if ta else (m, k), device="cuda").half()
    b = torch.randint(-2, 3, (n, k) if tb else (k, n), device="cuda").half()
    buf = torch.full((m * (n + gap) + off,), float("nan"), device="cuda")
    c = buf[off:].view(m, n + gap)
    call("br_hip_gemm", ta, tb, m, n, k, 0.5, ptr(a), F16, m if ta else k, 0, ptr(b), F16, k if tb else n, 0, 0, ptr(c), F32, n + gap, 0,
         None, 1, hip.GEMM_F16, stream())
    torch.cuda.synchronize()
    assert torch.equal(c[:, :n], 0.5 * ((a.t() if ta else a).float() @ (b.t() if tb else b).float()))
    assert c[:, n:].isnan().all() and buf[:off].isnan().all()


@pytest.mark.parametrize("k", [512, 2048])
def test_gemm_walking_workgroups_at_the_weight_gradient_shape(k):
    """dW[16384, 4096] = dy[k, 16384]^T . x[k, 4096] (1024 tiles, four per
    workgroup) at both token counts of the benchmarks: bit for bit the
    one-workgroup-per-tile kernel (taken with a bias of zeros), three launches
    in a row on rotating operands, and a sample of rows against fp64."""
    torch.manual_seed(k)
    m, n = 16384, 4096
    sets = [(torch.randn((k, m), device="cuda").half(), torch.randn((k, n), device="cuda").half()) for _ in range(3)]
    zeros = torch.zeros(n, device="cuda")
    for a, b in sets:
        outs = []
        for bias in (None, zeros):
            c = torch.full((m, n), float("nan"), device="cuda")
            call("br_hip_gemm", 1, 0, m, n, k, 0.25, ptr(a), F16, m, 0, ptr(b), F16, n, 0, 0, ptr(c), F32, n, 0, ptr(bias),
                 1, hip.GEMM_F16, stream())
            outs.append(c)
        torch.cuda.synchronize()
        assert torch.equal(outs[0], outs[1])
        rows = torch.arange(0, m, 257, device="cuda")
        ref = 0.25 * (a[:, rows].double().t() @ b.double())
        err = (outs[0][rows].double() - ref).abs()
        assert bool((err <= 1e-5 * (ref.abs() + ref.pow(2).mean().sqrt()) * (k ** 0.5)).all())


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("n,c_dt", [(12288, F16), (12248, F32)])
def test_gemm_round_and_a_half_of_tiles(ta, tb, n, c_dt):
    """[2048 x 12288] from K = 1024: 384 tiles of 256 x 256 are a round and a
    half on 256 CUs, which the dispatcher runs as two launches (8192 columns on
    256 x 256 tiles, the rest on 256 x 128 tiles).  Bias, alpha and an
    accumulated C cross the seam; the ragged case ends inside the second
    launch's last tile."""
    rng = np.random.default_rng(21)
    m, k = 2048, 1024
    print("case ta=%d tb=%d n=%d c_dt=%d" % (ta, tb, n, c_dt), flush=True)
    a, b = operands(rng, ta, tb, m, n, k)
    bias = rng.standard_normal(n).astype(np.float32)
    c0 = rng.standard_normal((1, m, n)).astype(np.float32)
    got, ref = run_gemm(ta, tb, m, n, k, a, b, F16, F16, c_dt, hip.GEMM_F16, alpha=0.5, bias=bias, c0=c0)
    assert_close(got, ref, 2e-2, "two-launch product")
    if c_dt == F32:
        assert np.sqrt(np.mean((got - ref) ** 2)) < 1e-5 * np.sqrt(np.mean(ref ** 2)) * np.sqrt(k)


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("c_dt", [F32, F16])
def test_gemm_tile_on_two_groups_of_waves(ta, tb, c_dt):
    """[1024 x 8192] from K = 2048: 256 tiles of 256 x 128 and 32 K steps, which the dispatcher runs with the
    sub-steps of every K step dealt to two groups of four waves whose sums meet in LDS after the K loop.  Alpha,
    bias and an accumulated C; against fp64, and with small-integer operands (every partial sum exact) bit for
    bit."""
    rng = np.random.default_rng(33)
    m, n, k = 1024, 8192, 2048
    assert hip.gemm_kernel(ta, tb, m, n, k) == ("256x128 groups", 1)
    print("case ta=%d tb=%d c_dt=%d" % (ta, tb, c_dt), flush=True)
    a, b = operands(rng, ta, tb, m, n, k)
    bias = rng.standard_normal(n).astype(np.float32)
    c0 = rng.standard_normal((1, m, n)).astype(np.float32)
    got, ref = run_gemm(ta, tb, m, n, k, a, b, F16, F16, c_dt, hip.GEMM_F16, alpha=0.5, bias=bias, c0=c0)
    assert_close(got, ref, 2e-2, "two wave groups")
    if c_dt == F32:
        assert np.sqrt(np.mean((got - ref) ** 2)) < 1e-5 * np.sqrt(np.mean(ref ** 2)) * np.sqrt(k)
        ai = rng.integers(-8, 9, a.shape).astype(np.float32)
        bi = rng.integers(-4, 5, b.shape).astype(np.float32)
        got, ref = run_gemm(ta, tb, m, n, k, ai, bi, F16, F16, F32, hip.GEMM_F16)
        assert np.array_equal(got, ref)


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("a_dt,b_dt", [(F32, F16), (F16, F32), (F32, F32)])
def test_gemm_staged_matches_plain_entry(ta, tb, a_dt, b_dt):
    rng = np.random.default_rng(8)
    m, n, k, batch = 384, 256, 128, 3
    print("case staged ta=%d tb=%d dtypes=%s" % (ta, tb, (a_dt, b_dt)), flush=True)
    a, b = operands(rng, ta, tb, m, n, k, batch)
    bias = rng.standard_normal(n).astype(np.float32)
    staged, plain, need = run_gemm_staged(ta, tb, m, n, k, a, b, a_dt, b_dt, F32, hip.GEMM_F16, batch=batch, bias=bias)
    assert need == sum(2 * batch * r * c for r, c, dt in ((m, k, a_dt), (k, n, b_dt)) if dt == F32)
    # same operand rounding, same products; only the summation order inside a
    # K step may differ between the two kernels
    assert_close(staged, plain, 1e-5, "staged vs plain")


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("a_dt,b_dt,c_dt", [(F32, F16, F32), (F16, F16, F16), (F32, F32, F32)])
def test_gemm_staged_split_k(ta, tb, a_dt, b_dt, c_dt):
    """Few output tiles and a long K: the staged entry splits K (the workspace
    figure shows it) and must still give the plain product, with alpha, bias
    and accumulation applied once."""
    rng = np.random.default_rng(10)
    m, n, k = 256, 384, 4096
    print("case split-k ta=%d tb=%d dtypes=%s" % (ta, tb, (a_dt, b_dt, c_dt)), flush=True)
    a, b = operands(rng, ta, tb, m, n, k)
    bias = rng.standard_normal(n).astype(np.float32)
    c0 = rng.standard_normal((1, m, n)).astype(np.float32)
    da, db_, dbias = to_dev(a, a_dt), to_dev(b, b_dt), dev(bias)
    need = hip.load().br_hip_gemm_staged_workspace(int(ta), int(tb), m, n, k, a_dt, b_dt, 1)
    copies = sum(2 * r * c for r, c, dt in ((m, k, a_dt), (k, n, b_dt)) if dt == F32)
    splits = (need - copies) // (4 * m * n)
    assert splits >= 2 and need == copies + splits * 4 * m * n
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    c = to_dev(c0, c_dt)
    call("br_hip_gemm_staged", int(ta), int(tb), m, n, k, 0.5, ptr(da), a_dt, m if ta else k, 0, ptr(db_), b_dt,
         k if tb else n, 0, 1, ptr(c), c_dt, n, 0, ptr(dbias), 1, hip.GEMM_F16, ptr(ws), need, stream())
    A = to_host64(da).reshape((k, m) if ta else (m, k))
    B = to_host64(db_).reshape((n, k) if tb else (k, n))
    ref = 0.5 * ((A.T if ta else A) @ (B.T if tb else B)) + bias.astype(np.float64)[None, :] + \
        to_host64(to_dev(c0, c_dt)).reshape(m, n)
    assert_close(to_host64(c).reshape(m, n), ref, 2e-2, "split-k staged gemm")
    if c_dt == F32:
        assert np.sqrt(np.mean((to_host64(c).reshape(m, n) - ref) ** 2)) < 1e-3 * np.sqrt(np.mean(ref ** 2))


def test_gemm_split_in_two_on_two_streams_at_once():
    """The 4h -> h shape ([2048 x 4096] from K = 16384, split in two inside
    the kernel) on two streams at the same time, each with its own operands
    and workspace: the slices of a tile meet through a counter set per stream,
    so both streams give the bits they give alone."""
    torch.manual_seed(5)
    m, n, k = 2048, 4096, 16384
    lib = hip.load()
    need = lib.br_hip_gemm_staged_workspace(0, 1, m, n, k, F16, F16, 1)
    assert need >= m * n * 4          # room for the partial tiles: this shape takes the split
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    jobs = []
    for _ in streams:
        a = torch.randn((m, k), device="cuda").half()
        b = torch.randn((n, k), device="cuda").half()
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        jobs.append((a, b, ws))
    torch.cuda.synchronize()

    def launch(job, c, st):
        a, b, ws = job
        call("br_hip_gemm_staged", 0, 1, m, n, k, 1.0, ptr(a), F16, k, 0, ptr(b), F16, k, 0, 0, ptr(c), F32, n, 0, None, 1,
             hip.GEMM_F16, ptr(ws), need, ctypes.c_void_p(st.cuda_stream))
    alone = []
    for job, st in zip(jobs, streams):
        c = torch.full((m, n), float("nan"), device="cuda")
        launch(job, c, st)
        torch.cuda.synchronize()
        alone.append(c)
    together = [[torch.full((m, n), float("nan"), device="cuda") for _ in range(4)] for _ in streams]
    torch.cuda.synchronize()
    for r in range(4):
        for i, (job, st) in enumerate(zip(jobs, streams)):
            launch(job, together[i][r], st)
    torch.cuda.synchronize()
    for i in range(2):
        for r in range(4):
            assert torch.equal(together[i][r], alone[i]), (i, r)
    ref = jobs[0][0][:64].double() @ jobs[0][1].double().t()
    assert bool(((alone[0][:64].double() - ref).abs() <= 1e-5 * (ref.abs() + ref.pow(2).mean().sqrt()) * (k ** 0.5)).all())


def test_gemm_staged_falls_back():
    rng = np.random.default_rng(9)
    # K not a multiple of 32, fp32 compute, and a workspace that is too small
    for (m, n, k, compute, ws) in ((96, 80, 40, hip.GEMM_F16, None), (128, 128, 64, hip.GEMM_F32, None),
                                   (128, 128, 64, hip.GEMM_F16, 16)):
        a, b = operands(rng, 0, 1, m, n, k)
        staged, plain, _ = run_gemm_staged(0, 1, m, n, k, a, b, F32, F32, F32, compute, ws_bytes=ws)
        assert np.array_equal(staged, plain)


def test_gemm_rejects_bad_arguments():
    lib = hip.load()
    t = empty(64)
    args = lambda **kw: None
    assert lib.br_hip_gemm(0, 1, 8, 8, 8, 1.0, ptr(t), F32, 4, 0, ptr(t), F32, 8, 0, 0, ptr(t), F32, 8, 0, None, 1,
                           hip.GEMM_F16, stream()) == -4          # lda < k
    assert lib.br_hip_gemm(0, 1, 8, 8, 8, 1.0, ptr(t), F16, 8, 0, ptr(t), F32, 8, 0, 0, ptr(t), F32, 8, 0, None, 1,
                           hip.GEMM_BF16, stream()) == -1         # fp16 storage with bf16 compute
    assert lib.br_hip_gemm(0, 1, 8, 8, 8, 1.0, ptr(t), F32, 8, 0, ptr(t), F32, 8, 0, 0, None, F32, 8, 0, None, 1,
                           hip.GEMM_F16, stream()) == -3
    torch.cuda.synchronize()


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("rows,out,inn", [(512, 1024, 256), (200, 520, 96), (2048, 4096, 1024), (2048, 12288, 1024),
                                          (512, 16384, 2048)])   # the last: 256 x 128 tiles on two groups of waves
def test_linear_gelu_epilogue_writes_both_tensors(dtype, rows, out, inn):
    """br_hip_linear_gelu: u = x.W^T + bias and y = gelu(u) from one product.
    u against the fp64 product of the stored operands, y against the oracle's
    GELU of that fp64 u (the kernel takes the activation of the fp32 sum, so y
    does not inherit u's storage rounding); 2e-2 for 16-bit operands, plus the
    output's own rounding."""
    import oracle as orc
    print("case dtype=%d rows=%d out=%d in=%d" % (dtype, rows, out, inn), flush=True)
    rng = np.random.default_rng(rows + out)
    x = to_dev(rng.standard_normal((rows, inn)), dtype)
    w = to_dev(rng.standard_normal((out, inn)) / np.sqrt(inn) * 1.5, dtype)
    bias = (0.1 * rng.standard_normal(out)).astype(np.float32)
    u = torch.full((rows, out), float("nan"), dtype=TORCH_T[dtype], device="cuda")
    y = torch.full((rows, out), float("nan"), dtype=TORCH_T[dtype], device="cuda")
    call("br_hip_linear_gelu", ptr(x), ptr(w), ptr(dev(bias)), ptr(u), ptr(y), dtype, rows, out, inn, stream())
    ref_u = to_host64(x) @ to_host64(w).T + bias.astype(np.float64)
    ref_y = orc.gelu_fwd(ref_u.astype(np.float32)).astype(np.float64)
    tol = 2e-2 if dtype == F16 else 3e-2
    assert_close(to_host64(u), ref_u, tol, "pre-activation")
    assert_close(to_host64(y), ref_y, tol, "gelu")
    # shapes the direct-to-LDS kernel does not take are declined, nothing is written
    assert hip.load().br_hip_linear_gelu(ptr(x), ptr(w), None, ptr(u), ptr(y), dtype, rows, out, inn - 8, stream()) == -1
    assert hip.load().br_hip_linear_gelu(ptr(x), ptr(w), None, ptr(u), ptr(u), dtype, rows, out, inn, stream()) == -3
    torch.cuda.synchronize()


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("c_dt", [F32, F16])
@pytest.mark.parametrize("m,n,k,batch", [
    (1, 8, 8, 1),            # one row of one tile, K within a chunk
    (33, 40, 72, 1),         # 32 x 32 tiles, one past the first; K one chunk past a step
    (64, 64, 64, 1),
    (78, 1024, 520, 1),      # 32-row tiles, K dealt unevenly to the four waves
    (250, 64, 250, 3),       # attention products of 250 tokens: rows that are not 16-byte aligned
    (31, 65, 7, 2),          # everything odd
    (1000, 1032, 1000, 1),   # 64 x 64 tiles with ragged edges
    (1002, 4096, 1002, 1),   # 128 x 128 tiles with a ragged K
    (200, 512, 12345, 1),    # slices of a ragged K
    (4000, 4104, 136, 1),    # the same, ragged in every direction
    (8200, 2056, 1002, 1),
])
def test_gemm_small_and_ragged_products_are_exact_on_integers(ta, tb, c_dt, m, n, k, batch):
    """The kernels for small and ragged sizes through the staged entry, on operands of small integers: every
    partial sum is a whole number below 2^24, so the fp32 result is exact whatever the order of summation (and an
    fp16 result is its rounding).  Any element read past an operand's end, or missed, changes it."""
    print("case ta=%d tb=%d c=%d m=%d n=%d k=%d batch=%d" % (ta, tb, c_dt, m, n, k, batch), flush=True)
    rng = np.random.default_rng(m + n + k)
    a, b = operands(rng, ta, tb, m, n, k, batch)
    a = rng.integers(-3, 4, a.shape).astype(np.float32)
    b = rng.integers(-2, 3, b.shape).astype(np.float32)
    bias = rng.integers(-5, 6, n).astype(np.float32)
    da, db_, dbias = to_dev(a, F16), to_dev(b, F16), dev(bias)
    c0 = rng.integers(-9, 10, (batch, m, n)).astype(np.float32)
    c = to_dev(c0, c_dt)
    need = hip.load().br_hip_gemm_staged_workspace(ta, tb, m, n, k, F16, F16, batch)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda").fill_(255)   # NaN wherever nothing is written
    call("br_hip_gemm_staged", ta, tb, m, n, k, 1.0, ptr(da), F16, m if ta else k, m * k, ptr(db_), F16, k if tb else n,
         n * k, 1, ptr(c), c_dt, n, m * n, ptr(dbias), batch, hip.GEMM_F16, ptr(ws), need, stream())
    A, B = a.astype(np.float64), b.astype(np.float64)
    ref = np.matmul(A.transpose(0, 2, 1) if ta else A, B.transpose(0, 2, 1) if tb else B) + bias.astype(np.float64) + c0
    if c_dt == F16:
        ref = ref.astype(np.float16).astype(np.float64)
    assert np.array_equal(to_host64(c).reshape(batch, m, n), ref)


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("kernel,slices,m,n,k,batch", PLANNED)
def test_gemm_every_kernel_is_exact_on_integers(ta, tb, kernel, slices, m, n, k, batch):
    """Every kernel the plan knows, in each of its forms, with both 16-bit types and both types of C: bias and an old C
    added, the workspace full of NaNs.  Small integers: every partial sum is exact in fp32."""
    assert hip.gemm_kernel(ta, tb, m, n, k, batch=batch, staged=True) == (kernel, slices)
    torch.manual_seed(m + n + k)
    a = torch.randint(-3, 4, (batch, k, m) if ta else (batch, m, k), device="cuda").float()
    b = torch.randint(-2, 3, (batch, n, k) if tb else (batch, k, n), device="cuda").float()
    bias = torch.randint(-5, 6, (n,), device="cuda").float()
    c0 = torch.randint(-9, 10, (batch, m, n), device="cuda").float()
    want = torch.stack([(x.t() if ta else x) @ (y.t() if tb else y) for x, y in zip(a, b)]) + bias + c0
    for t, dt, compute, c_dt in ((torch.float16, F16, hip.GEMM_F16, F32), (torch.bfloat16, BF16, hip.GEMM_BF16, BF16)):
        print("case %s/%d ta=%d tb=%d m=%d n=%d k=%d c=%d" % (kernel, slices, ta, tb, m, n, k, c_dt), flush=True)
        da, db_, c = a.to(t), b.to(t), c0.clone().to(TORCH_T[c_dt])
        need = hip.load().br_hip_gemm_staged_workspace(ta, tb, m, n, k, dt, dt, batch)
        ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda").fill_(255)
        call("br_hip_gemm_staged", ta, tb, m, n, k, 1.0, ptr(da), dt, m if ta else k, m * k, ptr(db_), dt, k if tb else n,
             n * k, 1, ptr(c), c_dt, n, m * n, ptr(bias), batch, compute, ptr(ws), need, stream())
        torch.cuda.synchronize()
        assert torch.equal(c, want.to(c.dtype))


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k,batch", [
    (1, 4, 4, 1),
    (33, 36, 40, 2),         # 32 x 32 tiles, rows in 16-byte granules
    (64, 1024, 260, 1),      # K dealt unevenly to the four waves
    (512, 1028, 1024, 1),    # 32 x 64 tiles
    (1000, 1028, 36, 4),     # 32 x 64 tiles, many of them
    (31, 65, 7, 2),          # value by value: everything odd
    (333, 64, 333, 3),       # attention products of 333 tokens
    (1001, 2050, 70, 2),     # 32 x 64 tiles, value by value
    (128, 128, 128, 512),
    (256, 384, 68, 90),
])
def test_gemm_fp32_small_tiles_are_exact_on_integers(ta, tb, m, n, k, batch):
    """The fp32 kernel's tiles and both ways it loads its operands, on small integers: every partial sum is exact."""
    print("case ta=%d tb=%d m=%d n=%d k=%d batch=%d" % (ta, tb, m, n, k, batch), flush=True)
    rng = np.random.default_rng(m + n + k)
    a, b = operands(rng, ta, tb, m, n, k, batch)
    a = rng.integers(-3, 4, a.shape).astype(np.float32)
    b = rng.integers(-2, 3, b.shape).astype(np.float32)
    bias = rng.integers(-5, 6, n).astype(np.float32)
    c0 = rng.integers(-9, 10, (batch, m, n)).astype(np.float32)
    got, ref = run_gemm(ta, tb, m, n, k, a, b, F32, F32, F32, hip.GEMM_F32, batch=batch, bias=bias, c0=c0)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("kernel,waves,m,n,k,batch", FP32_PLANNED)
def test_gemm_every_fp32_kernel_is_exact_on_integers(ta, tb, kernel, waves, m, n, k, batch):
    assert hip.gemm_fp32_kernel(m, n, k, batch) == (kernel, waves)
    test_gemm_fp32_small_tiles_are_exact_on_integers(ta, tb, m, n, k, batch)


@pytest.mark.parametrize("wide", ["a", "b"])
@pytest.mark.parametrize("ta,tb", [(0, 1), (1, 0)])
def test_gemm_fp32_rows_far_apart(ta, tb, wide):
    """Rows of an fp32 operand 2^23 elements apart: past the 32-bit offsets of the small-tile kernel, on 128 x 128
    tiles.  Ragged sizes, small integers: exact."""
    m, n, k, ld = 130, 70, 36, 1 << 23
    print("case wide=%s ta=%d tb=%d" % (wide, ta, tb), flush=True)
    rng = np.random.default_rng(9)
    a = torch.from_numpy(rng.integers(-3, 4, (k, m) if ta else (m, k)).astype(np.float32)).cuda()
    b = torch.from_numpy(rng.integers(-2, 3, (n, k) if tb else (k, n)).astype(np.float32)).cuda()
    bias = torch.from_numpy(rng.integers(-5, 6, n).astype(np.float32)).cuda()
    want = (a.t() if ta else a) @ (b.t() if tb else b) + bias
    narrow = a if wide == "a" else b
    spread = torch.empty((narrow.shape[0], ld), device="cuda")
    spread[:, :narrow.shape[1]] = narrow
    pa, pb = (spread, b) if wide == "a" else (a, spread)
    c = torch.full((m, n), float("nan"), device="cuda")
    call("br_hip_gemm", ta, tb, m, n, k, 1.0, ptr(pa), F32, pa.shape[1], 0, ptr(pb), F32, pb.shape[1], 0, 0, ptr(c), F32, n,
         0, ptr(bias), 1, hip.GEMM_F32, stream())
    torch.cuda.synchronize()
    assert torch.equal(c, want)


@pytest.mark.parametrize("m,n,k", [(64, 96, 40), (64, 96, 511), (200, 768, 512), (520, 1028, 1024), (520, 1028, 1028), (64, 256, 2048),
                                   (64, 256, 2052), (512, 1024, 3072),
                                   (64, 256, 4096), (64, 256, 4100), (1000, 1100, 2120), (31, 65, 2049)])
def test_gemm_fp32_error_against_64_bits(m, n, k):
    """Products as sums of bf16 parts: apart and folded, four waves and eight, tiles of 32 rows, values one by one.  Rounding sums of 64
    products of random sign to 24 bits one after the other leaves 2^-25 sqrt(64 / 2) = 1.7e-7 of the result."""
    print("case m=%d n=%d k=%d" % (m, n, k), flush=True)
    torch.manual_seed(k)
    for ta, tb in ((0, 1), (1, 0)):
        a, b = torch.randn((k, m) if ta else (m, k), device="cuda"), torch.randn((n, k) if tb else (k, n), device="cuda")
        c = torch.full((m, n), float("nan"), device="cuda")
        call("br_hip_gemm", ta, tb, m, n, k, 1.0, ptr(a), F32, a.shape[1], 0, ptr(b), F32, b.shape[1], 0, 0, ptr(c), F32, n, 0, None, 1,
             hip.GEMM_F32, stream())
        want = (a.t() if ta else a).double().contiguous() @ (b.t() if tb else b).double().contiguous()
        assert ((c - want).norm() / want.norm()).item() <= 2.0e-7


@pytest.mark.parametrize("front", [0, 1])   # values in front of A: 1 puts it off 16-byte boundaries
@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("kernel,waves,m,n,k,batch", FP32_PLANNED)
def test_gemm_every_fp32_kernel_against_64_bits(kernel, waves, m, n, k, batch, ta, tb, front):
    """The bound of test_gemm_fp32_error_against_64_bits; 128 x 128 tiles add up K one after the other, of at most 80 values."""
    assert hip.gemm_fp32_kernel(m, n, k, batch) == (kernel, waves)
    print("case ta=%d tb=%d m=%d n=%d k=%d batch=%d front=%d" % (ta, tb, m, n, k, batch, front), flush=True)
    torch.manual_seed(k)
    buf, b = torch.randn(front + batch * m * k, device="cuda"), torch.randn((batch, n, k) if tb else (batch, k, n), device="cuda")
    a = buf[front:].view((batch, k, m) if ta else (batch, m, k))
    c = torch.full((batch, m, n), float("nan"), device="cuda")
    call("br_hip_gemm", ta, tb, m, n, k, 1.0, ptr(a), F32, a.shape[2], m * k, ptr(b), F32, b.shape[2], n * k, 0, ptr(c), F32, n, m * n, None,
         batch, hip.GEMM_F32, stream())
    want = torch.stack([(x.t() if ta else x).double().contiguous() @ (y.t() if tb else y).double().contiguous() for x, y in zip(a, b)])
    assert ((c - want).norm() / want.norm()).item() <= 2.0e-7


@pytest.mark.parametrize("k", [40, 512, 2100])
@pytest.mark.parametrize("m,n", [(32, 64), (200, 768), (1000, 2100)])
def test_gemm_fp32_values_that_parts_do_not_hold(m, n, k):
    """Infinities, NaN, a value that rounds past bf16's largest and operands of some 2^-115 come out as from fp32 instructions."""
    print("case m=%d n=%d k=%d" % (m, n, k), flush=True)
    torch.manual_seed(k)
    for odd in (True, False):
        a, b = torch.randn((m, k), device="cuda"), torch.randn((n, k), device="cuda")
        if odd:
            a[3, 5], a[7, 9], b[11, 2], a[20, 30] = math.inf, math.nan, -math.inf, 3.4e38
            b[:, 30] = 0.25
            b[12, 5] = 0.0
        else:
            a *= 2.0 ** -115
        c = torch.full((m, n), 5.0, device="cuda")
        call("br_hip_gemm", 0, 1, m, n, k, 1.0, ptr(a), F32, k, 0, ptr(b), F32, k, 0, 0, ptr(c), F32, n, 0, None, 1, hip.GEMM_F32, stream())
        want = (a.double() @ b.double().t().contiguous()).cpu()   # of bounded rows and columns: no sum is beyond fp32
        got = c.double().cpu()
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
        assert torch.equal(got[want.isinf()], want[want.isinf()])
        sure = want.isfinite()
        sure[20] &= not odd   # one value outweighs the others
        assert ((got - want)[sure].norm() / want[sure].norm()).item() <= 2.0e-7
        if odd:
            both = want[20].isfinite()
            assert ((got[20] - want[20])[both].norm() / want[20][both].norm()).item() <= 2.0e-7


# 32 x 32 tiles (four waves, eight), 32 x 64 (four, eight) and 64 x 64, apart and folded; sizes that are loaded value by value too
FP32_SIZES = [(32, 64, 40), (200, 768, 512), (500, 4100, 516), (1000, 2100, 2100), (500, 520, 512), (500, 520, 2052), (500, 4096, 516),
              (500, 2048, 2052)]


@pytest.mark.parametrize("kernel,m,n,k", [("flex 32x64", 333, 1025, 1025), ("flex 32x64", 500, 520, 2052), ("flex 64", 500, 4096, 333),
                                          ("flex 64", 500, 4096, 516), ("flex 64", 500, 2048, 2052), ("flex 64", 500, 2048, 2053)])
def test_gemm_fp32_values_that_parts_do_not_hold_on_the_larger_tiles(kernel, m, n, k):
    assert hip.gemm_fp32_kernel(m, n, k)[0] == kernel
    test_gemm_fp32_values_that_parts_do_not_hold(m, n, k)


@pytest.mark.parametrize("front", [0, 1])   # values in front of A: 1 puts it off 16-byte boundaries
@pytest.mark.parametrize("m,n,k", FP32_SIZES)
def test_gemm_fp32_small_operands_keep_their_bits(m, n, k, front):
    """Operands down to the smallest subnormal ones against such as bring the sums back to normal numbers, beside one of ordinary
    size that meets zeros alone; the bound of test_gemm_fp32_error_against_64_bits.  And times one: every bit."""
    print("case m=%d n=%d k=%d front=%d" % (m, n, k, front), flush=True)
    rng = np.random.default_rng(k)

    def product(a, b):
        da, db = dev(np.concatenate([np.zeros(front, np.float32), a.ravel()])), dev(b)
        c = torch.full((m, n), float("nan"), device="cuda")
        call("br_hip_gemm", 0, 1, m, n, k, 1.0, ctypes.c_void_p(da.data_ptr() + 4 * front), F32, k, 0, ptr(db), F32, k, 0, 0, ptr(c), F32,
             n, 0, None, 1, hip.GEMM_F32, stream())
        return host(c)

    for ea, eb in ((-115, 0), (-120, 30), (-125, 60), (-130, 10), (-140, 100), (40, -130)):
        a, b = rng.standard_normal((m, k)) * 2.0 ** ea, rng.standard_normal((n, k)) * 2.0 ** eb
        a[:, 0], b[:, 0] = 1, 0
        a, b = a.astype(np.float32), b.astype(np.float32)
        got, want = product(a, b), (dev(a).double() @ dev(b).double().t().contiguous()).cpu().numpy()
        assert np.linalg.norm(got - want) / np.linalg.norm(want) <= 2.0e-7, (ea, eb)
    if n >= k:
        for e in (-124, -126, -135):
            a = (rng.uniform(1, 4, (m, k)) * 2.0 ** e).astype(np.float32)
            assert np.array_equal(product(a, np.eye(n, k, dtype=np.float32))[:, :k], a), e


@pytest.mark.parametrize("n,inn,out,kernel", [(64, 256, 264, "flex 32"), (250, 1024, 3072, "flex 32x64"), (512, 1024, 1024, "flex 64")])
def test_fp32_pairs_of_small_operands_and_of_values_that_parts_do_not_hold(n, inn, out, kernel):
    print("case n=%d in=%d out=%d" % (n, inn, out), flush=True)
    assert hip.load().br_hip_gemm_pair_kernel(out, inn, n, 1, n, inn, out, 1, hip.GEMM_F32) == hip.GEMM_KERNELS.index(kernel)
    rng = np.random.default_rng(n)
    for odd in (False, True):
        dy, x, w = (rng.standard_normal(s) * 2.0 ** (0 if odd else e)
                    for s, e in (((1, n, out), -125), ((1, n, inn), 60), ((1, out, inn), 60)))
        if odd:
            dy[0, 3, 5], dy[0, 20, 30], w[0, 11, 2], x[0, 9, 7] = math.inf, 3.0e38, math.nan, -math.inf
            w[0, 30], x[0, 20] = 0.25, 0.25
        dy, x, w = (dev(t.astype(np.float32)) for t in (dy, x, w))
        dw, dx = torch.full((1, out, inn), float("nan"), device="cuda"), torch.full((1, n, inn), float("nan"), device="cuda")
        assert run_pair([(1, 0, dy, x, dw), (0, 0, dy, w, dx)], hip.GEMM_F32)
        for got, want in ((dw, pair_reference(1, 0, dy, x)), (dx, pair_reference(0, 0, dy, w))):
            got, want = got.double(), torch.where(want.abs() >= 2.0 ** 128, want.sign() * math.inf, want)
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got[want.isinf()], want[want.isinf()])
            big = want.abs() > 1e30 if odd else want.isnan()   # one value outweighs the others
            for part in (want.isfinite() & big, want.isfinite() & ~big):
                assert not part.any() or ((got - want)[part].norm() / want[part].norm()).item() <= 2.0e-7


def test_gemm_fp32_without_k_leaves_the_bias():
    bias, a = dev(np.arange(7, dtype=np.float32)), empty((5, 8))
    c = torch.full((5, 7), float("nan"), device="cuda")
    call("br_hip_gemm", 0, 1, 5, 7, 0, 1.0, ptr(a), F32, 8, 0, ptr(a), F32, 8, 0, 0, ptr(c), F32, 7, 0, ptr(bias), 1,
         hip.GEMM_F32, stream())
    assert np.array_equal(host(c), np.tile(np.arange(7, dtype=np.float32), (5, 1)))


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("c_dt", [F32, F16])
@pytest.mark.parametrize("m,n,k,batch", [
    (488, 4096, 520, 1),     # about as few K steps as the plan gives it, the last one ragged
    (960, 1800, 2056, 1),    # an odd number of steps, ragged columns
    (1002, 2040, 1096, 1),   # ragged in every direction
    (512, 1000, 1032, 4),    # batch entries
])
def test_gemm_tiles_on_a_ring_of_k_steps_are_exact_on_integers(ta, tb, c_dt, m, n, k, batch):
    """64 x 128 tiles, one workgroup per CU: waves that load beside waves that multiply."""
    assert hip.gemm_kernel(ta, tb, m, n, k, c_dt, batch, staged=True) == ("ring 64x128", 1)
    test_gemm_small_and_ragged_products_are_exact_on_integers(ta, tb, c_dt, m, n, k, batch)


@pytest.mark.parametrize("dtype", [F16, BF16])
def test_linear_gelu_epilogue_on_a_ring_of_k_steps(dtype):
    assert hip.gemm_kernel(0, 1, 1024, 2048, 2048) == ("ring 64x128", 1)
    test_linear_gelu_epilogue_writes_both_tensors(dtype, 1024, 2048, 2048)


@pytest.mark.parametrize("a_wide", [True, False])
def test_gemm_staged_rows_too_far_apart_for_slices(a_wide):
    """An operand whose rows lie 2^22 elements apart is beyond the offsets of the kernels that know slices of K: the
    product is not sliced (small integers: exact), also where its sizes alone would have it in slices."""
    print("case a_wide=%s" % a_wide, flush=True)
    m, n, k, ld = 4, 4, 8192, 1 << 22
    rng = np.random.default_rng(3)
    a = rng.integers(-3, 4, (m, k)).astype(np.float32)
    b = rng.integers(-2, 3, (n, k)).astype(np.float32)
    spread = torch.zeros((4, ld), dtype=torch.float16, device="cuda")
    spread[:, :k] = torch.from_numpy(a if a_wide else b).cuda().half()
    dense = to_dev(b if a_wide else a, F16)
    pa, lda, pb, ldb = (spread, ld, dense, k) if a_wide else (dense, k, spread, ld)
    c = torch.zeros((m, n), device="cuda")
    need = hip.load().br_hip_gemm_staged_workspace(0, 1, m, n, k, F16, F16, 1)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda").fill_(255)
    call("br_hip_gemm_staged", 0, 1, m, n, k, 1.0, ptr(pa), F16, lda, 0, ptr(pb), F16, ldb, 0, 0, ptr(c), F32, n, 0, None,
         1, hip.GEMM_F16, ptr(ws), need, stream())
    assert need > 0   # sliced by its sizes
    assert np.array_equal(to_host64(c), a.astype(np.float64) @ b.astype(np.float64).T)


@pytest.mark.parametrize("c_dt", [F32, F16, BF16])
@pytest.mark.parametrize("old", [0, 1])
@pytest.mark.parametrize("off,gap", [(0, 0), (0, 3), (1, 4)])   # rows of C on 16-byte addresses, each row on another, none
@pytest.mark.parametrize("slices,m,n,k", [(2, 488, 1024, 5120), (4, 40, 1024, 3072), (8, 40, 512, 3072), (15, 200, 1024, 8200),
                                          (16, 40, 512, 12288)])
def test_gemm_sum_of_slices_is_exact_on_integers(slices, m, n, k, off, gap, old, c_dt):
    """The second launch of a product in slices of K: every number of slices, bias, an old C, and a C it can and cannot
    write four elements at a time, with nothing beside it written."""
    print("case slices=%d m=%d n=%d k=%d off=%d gap=%d c=%d" % (slices, m, n, k, off, gap, c_dt), flush=True)
    assert hip.gemm_kernel(0, 1, m, n, k, staged=True)[1] == slices
    torch.manual_seed(k)
    dt = F16 if c_dt == F16 else BF16
    a, b = whole_numbers((m, k), 2, dt), whole_numbers((n, k), 1, dt)
    bias, before = whole_numbers((n,), 5, F32), whole_numbers((m, n), 9, c_dt)
    buf = torch.full((off + m * (n + gap) + 8,), 77.0, device="cuda", dtype=TORCH_T[c_dt])
    c = buf[off:off + m * (n + gap)].view(m, n + gap)
    c[:, :n] = before
    need = hip.load().br_hip_gemm_staged_workspace(0, 1, m, n, k, dt, dt, 1)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda").fill_(255)
    call("br_hip_gemm_staged", 0, 1, m, n, k, 0.5, ptr(a), dt, k, 0, ptr(b), dt, k, 0, old, ptr(c), c_dt, n + gap, 0, ptr(bias), 1,
         hip.GEMM_F16 if dt == F16 else hip.GEMM_BF16, ptr(ws), need, stream())
    torch.cuda.synchronize()
    want = 0.5 * (a.float() @ b.float().t()) + bias + (before.float() if old else 0)
    assert torch.equal(c[:, :n], want.to(c.dtype))
    c[:, :n] = 77
    assert bool((buf == 77).all())


@pytest.mark.parametrize("c_dt", [F32, F16])
@pytest.mark.parametrize("kernel,m,n,k", [("256", 4000, 4096, 72), ("256x128 groups", 1000, 4104, 4160), ("128", 500, 4100, 72),
                                          ("flex 32", 40, 40, 72)])
def test_gemm_into_a_slice_of_a_wide_tensor(kernel, m, n, k, c_dt):
    """C is a block of columns of a tensor of 2^21 columns: whole large tiles as planned, the rest on small ones, and
    nothing beside the block is written.  Alpha, bias and an old C; small integers: exact."""
    ld = 1 << 21
    print("case %s m=%d n=%d k=%d c=%d" % (kernel, m, n, k, c_dt), flush=True)
    assert hip.gemm_kernel(0, 0, m, n, k)[0] == kernel
    torch.manual_seed(k)
    a = torch.randint(-3, 4, (m, k), device="cuda").float()
    b = torch.randint(-2, 3, (k, n), device="cuda").float()
    bias = torch.randint(-5, 6, (n,), device="cuda").float()
    c0 = torch.randint(-9, 10, (m, n), device="cuda").float()
    ah, bh = a.half(), b.half()
    whole = torch.empty((m, ld), dtype=TORCH_T[c_dt], device="cuda")
    at = 4096
    whole[:, at - 300:at + n + 300] = 77
    block = whole[:, at:at + n]
    block.copy_(c0)
    call("br_hip_gemm", 0, 0, m, n, k, 2.0, ptr(ah), F16, k, 0, ptr(bh), F16, n, 0, 1, ptr(block), c_dt, ld, 0,
         ptr(bias), 1, hip.GEMM_F16, stream())
    torch.cuda.synchronize()
    assert torch.equal(block, (2 * (a @ b) + bias + c0).to(block.dtype))
    assert bool((whole[:, at - 300:at] == 77).all()) and bool((whole[:, at + n:at + n + 300] == 77).all())


def test_linear_gelu_epilogue_on_a_wide_output():
    """More than 2^21 outputs, ragged in both directions; u is exact (small integers), y the GELU of it."""
    rows, out, inn = 300, (1 << 21) + 8, 64
    torch.manual_seed(2)
    x = torch.randint(-2, 3, (rows, inn), device="cuda").half()
    w = torch.randint(-1, 2, (out, inn), device="cuda").half()
    u, y = (torch.full((rows, out), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2))
    call("br_hip_linear_gelu", ptr(x), ptr(w), None, ptr(u), ptr(y), F16, rows, out, inn, stream())
    torch.cuda.synchronize()
    for lo in range(0, out, 1 << 18):
        want = x.float() @ w[lo:lo + (1 << 18)].float().t()
        assert torch.equal(u[:, lo:lo + (1 << 18)].float(), want)
        err = (y[:, lo:lo + (1 << 18)].float() - torch.nn.functional.gelu(want, approximate="tanh")).abs()
        assert float((err / (1 + want.abs())).max()) < 1e-3   # half an fp16 ulp is 5e-4 of the value


@pytest.mark.parametrize("batch", [1, 3])
@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
def test_gemm_staged_takes_rows_of_a_padded_pitch_where_they_are(ta, tb, batch):
    """16-bit operands of odd sizes whose rows start on 16-byte boundaries: only a row that runs along an odd K is
    copied (its end has to be zero-filled).  NaNs in the padding, small integers: exact."""
    m, n, k = 1001, 1003, 65
    print("case ta=%d tb=%d batch=%d" % (ta, tb, batch), flush=True)
    torch.manual_seed(4)

    def padded(rows, cols, most):
        t = torch.full((batch, rows, (cols + 7) // 8 * 8), float("nan"), dtype=torch.float16, device="cuda")
        t[:, :, :cols] = torch.randint(-most, most + 1, (batch, rows, cols), device="cuda").half()
        return t
    a = padded(*((k, m) if ta else (m, k)), 3)
    b = padded(*((n, k) if tb else (k, n)), 2)
    c = torch.full((batch, m, n), float("nan"), device="cuda")
    need = hip.load().br_hip_gemm_staged_workspace(ta, tb, m, n, k, F16, F16, batch)
    ws = torch.full((need,), 0x7f, dtype=torch.uint8, device="cuda")
    call("br_hip_gemm_staged", ta, tb, m, n, k, 1.0, ptr(a), F16, a.shape[2], a[0].numel(), ptr(b), F16, b.shape[2],
         b[0].numel(), 0, ptr(c), F32, n, m * n, None, batch, hip.GEMM_F16, ptr(ws), need, stream())
    torch.cuda.synchronize()
    for i in range(batch):
        x, y = a[i, :, :m if ta else k].float(), b[i, :, :k if tb else n].float()
        assert torch.equal(c[i], (x.t() if ta else x) @ (y.t() if tb else y))
    assert bool((ws != 0x7f).any()) == (not ta or tb)


def test_gemm_of_more_batch_entries_than_a_launch_has_work_items():
    """1.9 million fp32 products of nine 32 x 32 tiles each are more than 2^32 work items, which a launch drops without
    an error."""
    m, k, batch = 65, 4, 1900000
    print("case batch=%d" % batch, flush=True)
    a, b = (torch.ones((batch, m * k), device="cuda") for _ in range(2))
    c = torch.zeros((batch, m * m), device="cuda")
    call("br_hip_gemm", 0, 1, m, m, k, 1.0, ptr(a), F32, k, m * k, ptr(b), F32, k, m * k, 0, ptr(c), F32, m, m * m, None,
         batch, hip.GEMM_F32, stream())
    torch.cuda.synchronize()
    assert float(c.min()) == float(c.max()) == k


def whole_numbers(shape, most, dtype):
    return torch.randint(-most, most + 1, shape, device="cuda").to(TORCH_T[dtype])


def run_pair(products, compute, sums=None, later=None):
    """br_hip_gemm_pair on (trans_a, trans_b, a, b, c) with [batch, rows, cols] tensors; whether it was one launch."""
    code = {torch.float32: F32, torch.float16: F16, torch.bfloat16: BF16}
    descs, sizes = [], []
    for ta, tb, a, b, c in products:
        m, n, k = c.shape[1], c.shape[2], a.shape[1] if ta else a.shape[2]
        descs.append(hip.Product(ta, tb, m, n, k, 2.0, ptr(a), code[a.dtype], a.shape[2], a[0].numel(), ptr(b), code[b.dtype],
                                 b.shape[2], b[0].numel(), ptr(c), code[c.dtype], n, m * n, c.shape[0]))
        sizes = sizes + [m, n, k, c.shape[0]] if tb or not ta else [m, n, k, c.shape[0]] + sizes   # the weight gradient's first
    first, second = (ctypes.byref(d) for d in descs)
    need = hip.load().br_hip_gemm_pair_workspace(first, second, compute)
    ws = torch.full((max(need, 16),), 0x7f, dtype=torch.uint8, device="cuda")
    args = (first, second, ctypes.byref(sums) if sums else None, ctypes.byref(later) if later else None, compute, ptr(ws), need)
    call("br_hip_gemm_pair", *args, stream())
    torch.cuda.synchronize()
    kernel = hip.load().br_hip_gemm_pair_joined(*args)
    assert kernel in (-1, hip.load().br_hip_gemm_pair_kernel(*sizes, compute))
    return kernel >= 0


def pair_reference(ta, tb, a, b):
    a, b = a.double(), b.double()
    return 2 * torch.bmm(a.transpose(1, 2).contiguous() if ta else a, b.transpose(1, 2).contiguous() if tb else b)


COMPUTE_T = {hip.GEMM_F16: F16, hip.GEMM_BF16: BF16, hip.GEMM_F32: F32}


@pytest.mark.parametrize("compute", [hip.GEMM_F16, hip.GEMM_BF16, hip.GEMM_F32])
@pytest.mark.parametrize("n,inn,out,x_dt", [
    (1, 8, 8, None), (64, 256, 1024, None), (65, 1032, 264, None), (333, 136, 520, F32), (40, 2560, 640, F32), (516, 640, 640, None),
    (830, 640, 2560, F32), (700, 4096, 4096, None)])
def test_two_products_of_a_linear_layer_in_one_launch_are_exact_on_integers(n, inn, out, x_dt, compute):
    """dW = dy^T x, dx = dy W and the column sums of dy, every tile the rule picks and its remainders; the largest is two
    launches.  x and W in the products' type or as fp32 that is converted first; dx in either type."""
    dt = COMPUTE_T[compute]
    print("case n=%d in=%d out=%d compute=%d" % (n, inn, out, compute), flush=True)
    torch.manual_seed(n)
    for dx_dt in {dt, F32}:
        dy, x, w = whole_numbers((1, n, out), 1, dt), whole_numbers((1, n, inn), 1, x_dt or dt), whole_numbers((1, out, inn), 1, x_dt or dt)
        dw = torch.full((1, out, inn), float("nan"), device="cuda")
        dx = torch.full((1, n, inn), float("nan"), device="cuda", dtype=TORCH_T[dx_dt])
        db = torch.full((out,), float("nan"), device="cuda")
        need = hip.load().br_hip_colsum_workspace(n, out)
        ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
        sums = hip.ColumnSums(ptr(dy), dt, ptr(db), n, out, 0.5, ptr(ws), need)
        assert run_pair([(1, 0, dy, x, dw), (0, 0, dy, w, dx)], compute, sums) == (n != 700 or compute == hip.GEMM_F32)
        assert torch.equal(dw, pair_reference(1, 0, dy, x).float())
        assert torch.equal(dx, pair_reference(0, 0, dy, w).to(dx.dtype))
        assert torch.equal(db, 0.5 * dy[0].float().sum(0))


@pytest.mark.parametrize("compute", [hip.GEMM_F16, hip.GEMM_BF16])
@pytest.mark.parametrize("n,inn,out,x_dt", [(1, 1024, 1024, None), (64, 2056, 2040, None), (128, 1024, 4096, None), (200, 512, 2048, F32),
                                            (257, 1024, 3080, None), (300, 520, 2056, F32)])
def test_weight_gradients_on_wide_tiles_beside_the_other_product_are_exact_on_integers(n, inn, out, x_dt, compute):
    """One K step of the wide tiles to five, whole tiles and remainders either way, eight waves with a step each and some without;
    column sums and partial sums beside them, dx in either type and either product first."""
    dt = COMPUTE_T[compute]
    print("case n=%d in=%d out=%d compute=%d" % (n, inn, out, compute), flush=True)
    assert hip.load().br_hip_gemm_pair_kernel(out, inn, n, 1, n, inn, out, 1, compute) == 10   # BR_GEMM_PAIR_WIDE
    torch.manual_seed(n)
    partials = whole_numbers((3, 65, 68), 1, F32)
    for dx_dt, turned in ((dt, False), (F32, True)):
        dy, x, w = whole_numbers((1, n, out), 1, dt), whole_numbers((1, n, inn), 1, x_dt or dt), whole_numbers((1, out, inn), 1, dt)
        dw = torch.full((1, out, inn), float("nan"), device="cuda")
        dx = torch.full((1, n, inn), float("nan"), device="cuda", dtype=TORCH_T[dx_dt])
        db, added = torch.full((out,), float("nan"), device="cuda"), torch.full((3, 68), float("nan"), device="cuda")
        need = hip.load().br_hip_colsum_workspace(n, out)
        ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
        sums = hip.ColumnSums(ptr(dy), dt, ptr(db), n, out, 0.5, ptr(ws), need)
        later = hip.PartialSums(ptr(partials), 3, 65, 68, (ctypes.c_void_p * 3)(*(added[i].data_ptr() for i in range(3))), 2.0)
        products = [(1, 0, dy, x, dw), (0, 0, dy, w, dx)]
        assert run_pair(products[::-1] if turned else products, compute, sums, later)
        assert torch.equal(dw, pair_reference(1, 0, dy, x).float())
        assert torch.equal(dx, pair_reference(0, 0, dy, w).to(dx.dtype))
        assert torch.equal(db, 0.5 * dy[0].float().sum(0)) and torch.equal(added, 2 * partials.sum(1))


@pytest.mark.parametrize("compute", [hip.GEMM_F16, hip.GEMM_BF16])
@pytest.mark.parametrize("n,inn,out", [(200, 512, 2048), (257, 1024, 3080), (300, 1024, 4096)])
def test_weight_gradients_on_wide_tiles_are_as_precise_as_on_small_ones(n, inn, out, compute):
    """dW is four sums over every fourth 64 tokens, as a small tile's four waves leave them, added up at the end.  A matrix instruction
    adds 16 products to a sum and is off by up to 0.65 x 2^-24 of what it leaves (2-norm; 0.6 measured from 16 tokens): all
    roundings of the four and of the three additions, each times the variance the sum then has."""
    dt, steps = COMPUTE_T[compute], -(-n // 64)
    print("case n=%d in=%d out=%d compute=%d" % (n, inn, out, compute), flush=True)
    assert hip.load().br_hip_gemm_pair_kernel(out, inn, n, 1, n, inn, out, 1, compute) == 10   # BR_GEMM_PAIR_WIDE
    torch.manual_seed(n)
    dy, x, w = (torch.randn(s, device="cuda").to(TORCH_T[dt]) for s in ((1, n, out), (1, n, inn), (1, out, inn)))
    dw, dx = torch.empty((1, out, inn), device="cuda"), torch.empty((1, n, inn), device="cuda")
    assert run_pair([(1, 0, dy, x, dw), (0, 0, dy, w, dx)], compute)
    want = pair_reference(1, 0, dy, x)
    waves = [[min(16, n - k) / n for t in range(w, steps, 4) for k in range(64 * t, min(64 * t + 64, n), 16)] for w in range(4)]
    variance = sum(sum(np.cumsum(w)) for w in waves) + sum(np.cumsum([sum(w) for w in waves])[1:])
    assert ((dw - want).norm() / want.norm()).item() <= 0.65 * 2.0 ** -24 * math.sqrt(variance)


def sums_of_four_waves(x):
    """Column sums in fp32 in the order that four waves of 8 rows at a time have: every 32nd row one after the other, the 8 rows of a wave
    by halves, the waves one after the other."""
    slots = np.zeros((32, x.shape[1]), np.float32)
    for first in range(0, x.shape[0], 32):
        rows = x[first:first + 32]
        slots[:len(rows)] += rows
    while len(slots) > 4:
        slots = slots[0::2] + slots[1::2]
    return ((slots[0] + slots[1]) + slots[2]) + slots[3]


@pytest.mark.parametrize("compute", [hip.GEMM_F16, hip.GEMM_BF16])
@pytest.mark.parametrize("n,inn,out", [(1, 1024, 1024), (33, 1024, 4096), (78, 1024, 4096), (200, 512, 2048), (300, 1024, 4096), (78, 256, 264)])
def test_column_sums_beside_two_products_have_one_order(n, inn, out, compute):
    """Beside wide tiles as beside small ones (the last): the bits of four waves' sums."""
    dt = COMPUTE_T[compute]
    print("case n=%d in=%d out=%d compute=%d" % (n, inn, out, compute), flush=True)
    assert (hip.load().br_hip_gemm_pair_kernel(out, inn, n, 1, n, inn, out, 1, compute) == 10) == (out > 264)   # BR_GEMM_PAIR_WIDE
    torch.manual_seed(n)
    dy, x, w = (torch.randn(s, device="cuda").to(TORCH_T[dt]) for s in ((1, n, out), (1, n, inn), (1, out, inn)))
    dw, dx, db = (torch.empty(s, device="cuda") for s in ((1, out, inn), (1, n, inn), (out,)))
    need = hip.load().br_hip_colsum_workspace(n, out)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    assert run_pair([(1, 0, dy, x, dw), (0, 0, dy, w, dx)], compute, hip.ColumnSums(ptr(dy), dt, ptr(db), n, out, 1.0, ptr(ws), need))
    assert np.array_equal(host(db), sums_of_four_waves(host(dy[0].float())))


@pytest.mark.parametrize("compute", [hip.GEMM_F16, hip.GEMM_BF16, hip.GEMM_F32])
@pytest.mark.parametrize("n", [64, 700])   # one launch, and (16-bit) two after the sums
@pytest.mark.parametrize("arrays,parts,cols", [(2, 1, 4), (3, 7, 68), (3, 39, 256), (2, 64, 1000), (3, 65, 60), (3, 256, 4096)])
def test_partial_sums_are_added_up_beside_two_products(arrays, parts, cols, n, compute):
    """Whole numbers, so exact; a partial last group of columns, fewer parts than slices and more, and no room outside."""
    torch.manual_seed(cols)
    inn = out = 256 if n == 64 else 4096
    dt = COMPUTE_T[compute]
    print("case n=%d arrays=%d parts=%d cols=%d compute=%d" % (n, arrays, parts, cols, compute), flush=True)
    dy, x, w = (whole_numbers(s, 1, dt) for s in ((1, n, out), (1, n, inn), (1, out, inn)))
    dw, dx = torch.empty((1, out, inn), device="cuda"), torch.empty((1, n, inn), device="cuda", dtype=TORCH_T[dt])
    partials = whole_numbers((arrays, parts, cols), 50, F32)
    sums = torch.full((arrays, cols + 4), float("nan"), device="cuda")
    outs = (ctypes.c_void_p * 3)(*[sums[i].data_ptr() for i in range(arrays)])
    later = hip.PartialSums(ptr(partials), arrays, parts, cols, outs, 0.5)
    assert run_pair([(1, 0, dy, x, dw), (0, 0, dy, w, dx)], compute, None, later) == (n == 64 or compute == hip.GEMM_F32)
    assert torch.equal(sums[:, :cols], 0.5 * partials.sum(1)) and sums[:, cols:].isnan().all()
    assert torch.equal(dw, pair_reference(1, 0, dy, x).float())
    assert torch.equal(dx, pair_reference(0, 0, dy, w).to(dx.dtype))
    sums.fill_(float("nan"))
    call("br_hip_finish_sums", ctypes.byref(later), stream())   # a launch of their own
    assert torch.equal(sums[:, :cols], 0.5 * partials.sum(1)) and sums[:, cols:].isnan().all()


@pytest.mark.parametrize("compute", [hip.GEMM_F16, hip.GEMM_BF16, hip.GEMM_F32])
@pytest.mark.parametrize("bh,t,hd,p_dt", [(2, 4, 64, None), (6, 40, 64, F32), (5, 50, 96, None), (3, 250, 128, None), (40, 120, 128, F32)])
def test_two_products_of_attention_in_one_launch_are_exact_on_integers(bh, t, hd, p_dt, compute):
    """dV = P^T dO with dP = dO V^T, and dQ = dS K with dK = dS^T Q in that order; rows of T values that are no multiple of a
    granule are copied once for both."""
    dt = COMPUTE_T[compute]
    print("case bh=%d t=%d hd=%d compute=%d" % (bh, t, hd, compute), flush=True)
    torch.manual_seed(t)
    p, d_o, v = whole_numbers((bh, t, t), 1, p_dt or dt), whole_numbers((bh, t, hd), 1, dt), whole_numbers((bh, t, hd), 1, p_dt or dt)
    dv, dq = (torch.full((bh, t, hd), float("nan"), device="cuda") for _ in range(2))
    dp = torch.full((bh, t, t), float("nan"), device="cuda")
    joined = compute != hip.GEMM_F32 or t % 4 == 0   # fp32 rows have to start on 16-byte boundaries
    assert run_pair([(1, 0, p, d_o, dv), (0, 1, d_o, v, dp)], compute) == joined
    assert torch.equal(dv, pair_reference(1, 0, p, d_o).float()) and torch.equal(dp, pair_reference(0, 1, d_o, v).float())
    dv.fill_(float("nan"))
    assert run_pair([(0, 0, p, v, dq), (1, 0, p, d_o, dv)], compute) == joined
    assert torch.equal(dq, pair_reference(0, 0, p, v).float()) and torch.equal(dv, pair_reference(1, 0, p, d_o).float())


@pytest.mark.parametrize("staged", [False, True])
def test_two_products_keep_their_order_where_one_overwrites_the_others_operand(staged):
    """dx over x, as the model's scripts have it: the weight gradient is formed from x as it was."""
    torch.manual_seed(7)
    n, inn, out = 72, 256, 512
    dy, w = whole_numbers((1, n, out), 1, F16), whole_numbers((1, out, inn), 1, F16)
    x = whole_numbers((1, n, inn), 1, F32 if staged else F16)
    dw = torch.empty((1, out, inn), device="cuda")
    want = pair_reference(1, 0, dy, x).float()
    # a copy of x is out of dx's way, x itself is not
    assert run_pair([(1, 0, dy, x, dw), (0, 0, dy, w, x)], hip.GEMM_F16) == staged
    assert torch.equal(dw, want) and torch.equal(x, pair_reference(0, 0, dy, w).to(x.dtype))


@pytest.mark.parametrize("over", [None, "sums.x", "x"])
@pytest.mark.parametrize("compute", [hip.GEMM_F16, hip.GEMM_F32])
def test_sums_beside_two_products_keep_their_order_where_they_meet(over, compute):
    """Partial sums, column sums and both products as the one-after-the-other calls leave them: the column sums are of what the
    partial sums have written, and so are the products, also of an operand that is converted first."""
    torch.manual_seed(9)
    dt = COMPUTE_T[compute]
    n, inn, out, rows, cols, parts = 64, 256, 256, 40, 256, 7
    print("case over=%s compute=%d" % (over, compute), flush=True)
    dy, x, w = whole_numbers((1, n, out), 1, dt), whole_numbers((1, n, inn), 1, F32), whole_numbers((1, out, inn), 1, dt)
    z = whole_numbers((rows, cols), 3, F32)
    partials = whole_numbers((2, parts, cols), 1, F32)
    dw, dx = torch.empty((1, out, inn), device="cuda"), torch.empty((1, n, inn), device="cuda")
    db, apart = torch.full((cols,), float("nan"), device="cuda"), torch.full((2, cols), float("nan"), device="cuda")
    first = {None: apart[0], "sums.x": z[3], "x": x[0, 5]}[over]
    outs = (ctypes.c_void_p * 3)(first.data_ptr(), apart[1].data_ptr())
    later = hip.PartialSums(ptr(partials), 2, parts, cols, outs, 1.0)
    need = hip.load().br_hip_colsum_workspace(rows, cols)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    sums = hip.ColumnSums(ptr(z), F32, ptr(db), rows, cols, 0.5, ptr(ws), need)
    # (column sums of another type than the products' are a launch of their own)
    assert run_pair([(1, 0, dy, x, dw), (0, 0, dy, w, dx)], compute, sums, later) == (over is None and compute == hip.GEMM_F32)
    added = partials.sum(1)
    assert torch.equal(first, added[0]) and torch.equal(apart[1], added[1]) and torch.equal(db, 0.5 * z.sum(0))
    assert torch.equal(dw, pair_reference(1, 0, dy, x).float()) and torch.equal(dx, pair_reference(0, 0, dy, w).float())


@pytest.mark.parametrize("compute", [hip.GEMM_F16, hip.GEMM_BF16, hip.GEMM_F32])
@pytest.mark.parametrize("rows,out,inn,x_dt,y_dt", [
    (24, 256, 256, F32, F32), (65, 40, 72, None, None), (130, 1000, 136, None, F32), (1000, 1024, 64, F32, F32), (1000, 2048, 256, None, F32),
    (2100, 1280, 128, F32, None), (33, 30, 20, F32, F32), (512, 2048, 2048, None, None)])
def test_linear_group_is_exact_on_integers(rows, out, inn, x_dt, y_dt, compute):
    """Three layers of one x as a batch, each with a bias of its own; the kernels of small and of large tiles, sizes that are no multiple
    of a granule among them."""
    dt = COMPUTE_T[compute]
    print("case rows=%d out=%d in=%d compute=%d" % (rows, out, inn, compute), flush=True)
    torch.manual_seed(rows)
    x, w = whole_numbers((rows, inn), 1, x_dt or dt), whole_numbers((3, out, inn), 1, dt)
    bias = whole_numbers((3, out), 5, F32)
    y = torch.full((3, rows, out), float("nan"), device="cuda", dtype=TORCH_T[y_dt or dt])
    need = hip.load().br_hip_linear_group_workspace(3, rows, out, inn, x_dt or dt, dt)
    ws = torch.full((max(need, 16),), 0x7f, dtype=torch.uint8, device="cuda")
    call("br_hip_linear_group", ptr(x), x_dt or dt, ptr(w), dt, ptr(bias), ptr(y), y_dt or dt, 3, rows, out, inn, compute, ptr(ws),
         need, stream())
    torch.cuda.synchronize()
    for i in range(3):
        assert torch.equal(y[i], (x.double() @ w[i].double().t() + bias[i].double()).to(y.dtype))


@pytest.mark.parametrize("compute", [hip.GEMM_F16, hip.GEMM_F32])
@pytest.mark.parametrize("rows,out,inn", [(24, 256, 256), (65, 44, 72), (78, 1024, 4096), (1000, 1024, 1024), (1000, 2048, 2048), (2048, 4096, 64), (33, 30, 20),
                                          (500, 4096, 384), (800, 2560, 1536)])   # two waves to a tile: with the sum, and followed by it
@pytest.mark.parametrize("over", [False, True])
def test_linear_with_the_sum_beside_it_is_exact_on_integers(rows, out, inn, over, compute):
    """y and y + r, the sum over r or apart: small tiles, a ring of K steps, slices of K, and large tiles followed by an
    addition."""
    dt = COMPUTE_T[compute]
    print("case rows=%d out=%d in=%d compute=%d" % (rows, out, inn, compute), flush=True)
    torch.manual_seed(rows)
    x, w = whole_numbers((rows, inn), 1, dt), whole_numbers((out, inn), 1, dt)
    bias, r = whole_numbers((out,), 5, F32), whole_numbers((rows, out), 9, F32)
    want = x.double() @ w.double().t() + bias.double()
    want_sum = want + r.double()
    y = torch.full((rows, out), float("nan"), device="cuda")
    total = r if over else torch.full_like(y, float("nan"))
    need = hip.load().br_hip_gemm_staged_workspace(0, 1, rows, out, inn, dt, dt, 1) if compute != hip.GEMM_F32 else 0
    ws = torch.full((max(need, 16),), 0x7f, dtype=torch.uint8, device="cuda")
    call("br_hip_linear_sum", ptr(x), dt, ptr(w), dt, ptr(bias), ptr(r), ptr(y), ptr(total), rows, out, inn, compute, ptr(ws), need,
         stream())
    torch.cuda.synchronize()
    assert torch.equal(y, want.float()) and torch.equal(total, want_sum.float())
