"""At most 128 rows per weight set through the SwiGLU and int8 forms of the
skinny kernels (narrow_dma_kernel to 16 rows, narrow_lds_kernel to 128) and
the workgroups of the 16-row kernels, on a context built with U15H_SKINNY=2
(every batch that fits them), against the tiled GEMM of one built with
U15H_SKINNY=0.  int32 accumulators and dequantised
outputs are equal bit for bit (exact sums, the same epilogue arithmetic);
bf16 sums run in another order, so outputs meet the reference's bars
(max-rel <= 1e-2, rel-L2 < 4e-3, tests/u15-kernels-test.cc:55), and equal
the exact result bit for bit on operands whose sums are exact in any order."""
import os

import numpy as np
import pytest
import torch

import oracle
import u15h
from helpers import dev_bf16, host_bits, host_f32, max_rel, rand_bf16_bits, rel_l2

pytestmark = pytest.mark.gpu

MAX_REL = 1e-2
REF_BAR = 4e-3


def ctx_with(skinny):
    """A context created with U15H_SKINNY=skinny (read at create)."""
    old = os.environ.get("U15H_SKINNY")
    os.environ["U15H_SKINNY"] = str(skinny)
    try:
        return u15h.Ops(0)
    finally:
        if old is None:
            del os.environ["U15H_SKINNY"]
        else:
            os.environ["U15H_SKINNY"] = old


@pytest.fixture(scope="module")
def tiled():
    o = ctx_with(0)
    yield o
    torch.cuda.synchronize()
    o.close()


@pytest.fixture(scope="module")
def ops():
    o = ctx_with(2)
    yield o
    torch.cuda.synchronize()
    o.close()


def small_ints(rng, shape, top):
    """bf16 bits of integers in [-top, top]: products and sums are exact."""
    return oracle.f32_to_bf16(rng.integers(-top, top + 1, shape).astype(np.float32))


# (rows, K, N): both kernels' row edges, one K-block, fewer K-blocks than
# waves, columns that leave lanes, waves or whole fragments past N, and
# shapes of every 16-row plan: 4 and 8 waves, 1, 2 and 4 K shares.
SHAPES = [(1, 64, 8), (1, 192, 24), (1, 4096, 1024), (3, 1024, 2600), (16, 2048, 6152), (2, 8192, 264), (16, 8192, 136),
          (4, 4096, 2568),
          (17, 128, 72), (32, 4096, 200), (33, 1088, 1000), (64, 2048, 4104), (65, 256, 520),
          (96, 4096, 1032), (97, 640, 136), (128, 4096, 4096), (128, 64, 8)]


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_swiglu_exact_sums(ops, tiled, M, K, N):
    """gate and up sums are small integers, so every order rounds the same:
    equal bits to the tiled kernel, for separate and interleaved weights."""
    rng = np.random.default_rng(M + K + N)
    x = dev_bf16(small_ints(rng, (M, K), 2))
    wg = dev_bf16(small_ints(rng, (N, K), 1))
    wu = dev_bf16(small_ints(rng, (N, K), 1))
    h = torch.full((M, N), 7.0, dtype=torch.bfloat16, device="cuda")
    ref, fused = torch.full_like(h, 3.0), torch.full_like(h, 5.0)
    wf = torch.stack([wg, wu], 1).reshape(2 * N, K).contiguous()
    ops.mot_gate_up_swiglu(x, M, 0, K, wg, wu, None, None, h)
    ops.swiglu_fused(x, wf, fused, M, K, N)
    tiled.mot_gate_up_swiglu(x, M, 0, K, wg, wu, None, None, ref)
    torch.cuda.synchronize()
    assert torch.equal(h.view(torch.int16), ref.view(torch.int16))
    assert torch.equal(fused.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("Mu,Mg", [(1, 0), (5, 16), (0, 60), (20, 90), (128, 128)])
def test_swiglu_both_groups(ops, tiled, Mu, Mg):
    """Random rows of both weight sets in one call (the larger group picks
    the build) against the tiled kernel and the oracle."""
    K, N, M = 2048, 1064, Mu + Mg
    rng = np.random.default_rng(Mu + Mg)
    xb = rand_bf16_bits(rng, (M, K))
    W = [rand_bf16_bits(rng, (N, K), 0.03) for _ in range(4)]
    x, w = dev_bf16(xb), [dev_bf16(b) for b in W]
    h = torch.full((M, N), 7.0, dtype=torch.bfloat16, device="cuda")
    t = torch.empty_like(h)
    ops.mot_gate_up_swiglu(x, Mu, Mg, K, *w, h)
    tiled.mot_gate_up_swiglu(x, Mu, Mg, K, *w, t)
    torch.cuda.synchronize()
    assert rel_l2(host_f32(h), host_f32(t)) < REF_BAR
    assert max_rel(host_f32(h), host_f32(t)) <= MAX_REL
    gate = oracle.mot_linear_bf16(xb, W[0], W[2], Mu, Mg)
    up = oracle.mot_linear_bf16(xb, W[1], W[3], Mu, Mg)
    ref = oracle.swiglu_bf16(oracle.f32_to_bf16(gate), oracle.f32_to_bf16(up))
    assert rel_l2(host_f32(h), ref) < REF_BAR


@pytest.mark.parametrize("M,K,N", [s for s in SHAPES if s[1] % 128 == 0])
def test_int8_equals_the_tiled_kernel(ops, tiled, M, K, N):
    """Accumulators at the extremes (codes +-127) and dequantised outputs,
    both groups, two projections: bit for bit."""
    rng = np.random.default_rng(M + K + N)
    Mu = M // 3
    Mg = M - Mu

    def codes(*shape):
        c = rng.integers(-127, 128, shape).astype(np.int8)
        c.reshape(-1)[::5] = 127
        return torch.from_numpy(c).cuda()

    def scales(n):
        return torch.from_numpy(rng.random(n).astype(np.float32) * 1e-3).cuda()
    xq, sx = codes(M, K), scales(M)
    base = []
    for n in (N, 16):
        base.append(dict(wq_und=codes(n, K), wq_gen=codes(n, K), sw_und=scales(n),
                         sw_gen=scales(n)))
    for call, dtype in (("mot_gemm_i8_i32", torch.int32), ("mot_gemm_i8", torch.bfloat16)):
        got = []
        for o in (ops, tiled):
            projs = [dict(p, y=torch.full((M, p["wq_und"].shape[0]), 7, dtype=dtype,
                                          device="cuda")) for p in base]
            args = (xq,) if call.endswith("i32") else (xq, sx)
            getattr(o, call)(*args, Mu, Mg, K, projs)
            got.append([p["y"] for p in projs])
        torch.cuda.synchronize()
        for a, b in zip(*got):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("N", [8, 1024, 2568, 6144])
@pytest.mark.parametrize("M,K", [(1, 64), (4, 4096), (7, 4096), (16, 1984), (3, 8192),
                                 (16, 12288)])
def test_bf16_workgroup_plans(ops, M, K, N):
    """The 16-row kernel's plans (4 or 8 waves, 1 to 4 K shares by the rows,
    K and the column blocks), with bias, on exact sums: equal bits to the
    exact result."""
    rng = np.random.default_rng(M + K + N)
    xb, wb = small_ints(rng, (M, K), 2), small_ints(rng, (N, K), 1)
    bb = small_ints(rng, (N,), 3)
    y = torch.full((M, N), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.linear(dev_bf16(xb), dev_bf16(wb), dev_bf16(bb), y, M, K, N)
    torch.cuda.synchronize()
    f = oracle.bf16_to_f32
    exact = f(xb).astype(np.float64) @ f(wb).astype(np.float64).T + f(bb)
    assert np.array_equal(host_bits(y), oracle.f32_to_bf16(exact.astype(np.float32)))


@pytest.mark.parametrize("bits,group", [(8, 64), (8, 32), (4, 64), (4, 32)])
@pytest.mark.parametrize("M,K,N,shift", [
    (1, 64, 8, 0), (5, 192, 24, 0), (16, 320, 328, 0), (1, 4096, 328, 1), (3, 1984, 2568, 0),
    (16, 2048, 2568, 1), (1, 448, 6144, 0), (9, 1024, 6152, 1), (2, 1024, 6144, 0),
    (4, 4096, 2568, 1), (1, 8192, 136, 0), (16, 8192, 136, 1), (3, 12288, 24, 1)])
def test_pack_order_equals_the_expansion(ops, bits, group, M, K, N, shift):
    """narrow_pack_kernel's plans (8 and 4 waves, K shares; a K that ends
    inside a 128-byte line of codes; scales an odd number of groups per row,
    or `shift` elements off dword alignment, which take the 16-bit loads or
    the register kernel): bit-equal to u15h_linear on the expansion, also
    where a scale is infinite or NaN."""
    rng = np.random.default_rng(M + K + N + bits)
    codes = rng.integers(0, 1 << 32, (N, K * bits // 32), dtype=np.uint64).astype(np.uint32)
    sc = rng.random((N, K // group)).astype(np.float32) * 0.01
    bi = rng.standard_normal((N, K // group)).astype(np.float32) * 0.1
    sc[3, -1], bi[5, 0] = np.inf, np.nan

    def dev(a):
        flat = torch.zeros(a.size + 8, dtype=torch.bfloat16, device="cuda")
        t = flat[shift:shift + a.size].view(a.shape)
        t.copy_(dev_bf16(oracle.f32_to_bf16(a)))
        return t
    qw = (torch.from_numpy(codes.view(np.int32)).cuda(), dev(sc), dev(bi), bits, group)
    x = dev_bf16(rand_bf16_bits(rng, (M, K)))
    b = dev_bf16(rand_bf16_bits(rng, (N,)))
    y, y2 = (torch.full((M, N), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    w = torch.empty(N, K, dtype=torch.bfloat16, device="cuda")
    ops.linear_q(x, qw, b, y, M, K, N)
    ops.dequant_affine(qw, N, K, w)
    ops.linear(x, w, b, y2, M, K, N)
    torch.cuda.synchronize()
    nan = torch.isnan(y2)
    assert torch.equal(torch.isnan(y), nan) and bool(nan[:, [3, 5]].all())
    assert int(nan.sum()) == 2 * M
    assert torch.equal(y.view(torch.int16)[~nan], y2.view(torch.int16)[~nan])


@pytest.mark.parametrize("bits,group", [(8, 64), (4, 32)])
@pytest.mark.parametrize("M", [96, 97, 128, 129])
def test_packs_up_to_the_skinny_rows(ops, bits, group, M):
    """96 to 128 rows read the pack directly with the default floor: bit-equal
    to u15h_linear on the expansion, as at 129 rows and with the floor set
    (which expands)."""
    K, N = 1024, 520
    rng = np.random.default_rng(M + bits)
    codes = rng.integers(0, 1 << 32, (N, K * bits // 32), dtype=np.uint64).astype(np.uint32)
    sc, bi = (dev_bf16(rand_bf16_bits(rng, (N, K // group), 0.01)) for _ in range(2))
    qw = (torch.from_numpy(codes.view(np.int32)).cuda(), sc, bi, bits, group)
    x = dev_bf16(rand_bf16_bits(rng, (M, K)))
    os.environ["U15H_Q_MIN_M"] = "96"
    try:
        floor = u15h.Ops(0)
    finally:
        del os.environ["U15H_Q_MIN_M"]
    w = torch.empty(N, K, dtype=torch.bfloat16, device="cuda")
    ops.dequant_affine(qw, N, K, w)
    ys = [torch.full((M, N), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
    ops.linear_q(x, qw, None, ys[0], M, K, N)
    floor.linear_q(x, qw, None, ys[1], M, K, N)
    ops.linear(x, w, None, ys[2], M, K, N)
    torch.cuda.synchronize()
    floor.close()
    assert torch.equal(ys[0].view(torch.int16), ys[2].view(torch.int16))
    assert torch.equal(ys[1].view(torch.int16), ys[2].view(torch.int16))
