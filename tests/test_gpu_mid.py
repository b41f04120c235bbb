"""The mid-size tiles (mid_gemm_kernel: 128, 192 or 256 rows x 128 weight
rows) against the 256 x 256 tiles of a context built with U15H_MID=0: equal
bits on operands whose sums are exact in any order, for every epilogue, at
row and column counts around the tiles' edges, K tails, whole rounds, split
tails, and both groups with and without bias; and the planner's choice
against the tiled kernel and the oracle on random operands."""
import os

import numpy as np
import pytest
import torch

import oracle
import u15h
from helpers import dev_bf16, host_f32, max_rel, rand_bf16_bits, rel_l2

pytestmark = pytest.mark.gpu


def ctx_with(**env):
    old = {k: os.environ.get(k) for k in env}
    os.environ.update({k: str(v) for k, v in env.items()})
    try:
        return u15h.Ops(0)
    finally:
        for k, v in old.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v


@pytest.fixture(scope="module")
def contexts():
    made = {bm: ctx_with(U15H_MID=bm) for bm in (0, 128, 192, 256)}
    made["one"] = ctx_with(U15H_MID=192, U15H_SPLIT=0, U15H_PERSIST=0)
    yield made
    torch.cuda.synchronize()
    for o in made.values():
        o.close()


def ints(rng, shape, top):
    return dev_bf16(oracle.f32_to_bf16(rng.integers(-top, top + 1, shape).astype(np.float32)))


@pytest.mark.parametrize("Mu,Mg,K,N", [
    (0, 129, 64, 8), (129, 0, 72, 136), (43, 157, 192, 264), (0, 333, 1088, 1000),
    (128, 192, 640, 2056), (191, 193, 4096, 128), (257, 0, 2048, 520), (1, 1023, 256, 4104),
    (100, 1500, 320, 264)])
@pytest.mark.parametrize("bm", [128, 192, 256, "one"])
def test_exact_sums_equal_the_256_tiles(contexts, bm, Mu, Mg, K, N):
    rng = np.random.default_rng(Mu + Mg + K + N)
    M = Mu + Mg
    x, bias = ints(rng, (M, K), 2), [ints(rng, (N,), 3) for _ in range(2)]
    w = [ints(rng, (N, K), 1) for _ in range(4)]
    xq = torch.from_numpy(rng.integers(-127, 128, (M, K)).astype(np.int8)).cuda()
    wq = [torch.from_numpy(rng.integers(-127, 128, (N, K)).astype(np.int8)).cuda()
          for _ in range(2)]
    sx, s0, s1 = (torch.from_numpy(rng.random(n).astype(np.float32)).cuda() for n in (M, N, N))

    def run(o):
        def out(dtype=torch.bfloat16, n=N):
            return torch.full((M, n), 7, dtype=dtype, device="cuda")
        ys = [out(), out(), out()]
        o.mot_linear(x, Mu, Mg, K, [
            dict(w_und=w[0], w_gen=w[1], bias_und=bias[0], bias_gen=bias[1], y=ys[0]),
            dict(w_und=w[2], w_gen=w[3], y=ys[1])])
        o.mot_gate_up_swiglu(x, Mu, Mg, K, *w, ys[2])
        if K % 128 == 0:
            proj = dict(wq_und=wq[0], wq_gen=wq[1], sw_und=s0, sw_gen=s1)
            ys += [out(torch.int32), out()]
            o.mot_gemm_i8_i32(xq, Mu, Mg, K, [dict(proj, y=ys[3])])
            o.mot_gemm_i8(xq, sx, Mu, Mg, K, [dict(proj, y=ys[4])])
        torch.cuda.synchronize()
        return ys
    for a, b in zip(run(contexts[bm]), run(contexts[0])):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("M,K,N", [(130, 4096, 1032), (333, 4096, 4096), (1100, 1024, 2056)])
def test_planned_tiles(ops, contexts, M, K, N):
    """The default context's choice (a mid-size tile at these shapes:
    test_plan.py) on random operands, with bias, at the reference's bars."""
    rng = np.random.default_rng(M + K + N)
    xb, wb = rand_bf16_bits(rng, (M, K)), rand_bf16_bits(rng, (N, K), 0.02)
    bb = rand_bf16_bits(rng, (N,), 0.5)
    x, w, b = dev_bf16(xb), dev_bf16(wb), dev_bf16(bb)
    y, t = (torch.full((M, N), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    ops.linear(x, w, b, y, M, K, N)
    contexts[0].linear(x, w, b, t, M, K, N)
    torch.cuda.synchronize()
    assert rel_l2(host_f32(y), host_f32(t)) < 4e-3
    rows = np.array([0, M // 2, M - 1], np.int32)
    ref = oracle.linear_bf16(xb, wb, bb, row_ids=rows)
    a = host_f32(y)[rows]
    assert max_rel(a, ref) <= 1e-2 and rel_l2(a, ref) < 4e-3


@pytest.mark.parametrize("Mu,Mg,K,N", [(128, 4096, 256, 4096), (1, 2048, 192, 8192),
                                       (50, 4096, 320, 4096), (77, 4096, 256, 4096)])
def test_few_rows_apart_from_whole_rounds(ops, contexts, Mu, Mg, K, N):
    """A group of at most 128 rows beside one whose 256 x 256 tiles fill whole
    rounds of 256 CUs runs in a launch of its own (test_plan.py): equal bits
    on exact sums to the one grouped launch, for every epilogue, and in the
    allocation-free call."""
    rng = np.random.default_rng(Mu + Mg + K)
    M = Mu + Mg
    x = ints(rng, (M, K), 2)
    w = [ints(rng, (N, K), 1) for _ in range(4)]
    b = [ints(rng, (N,), 3) for _ in range(2)]

    def run(o, call):
        y = torch.full((M, N), 7, dtype=torch.bfloat16, device="cuda")
        if call == "swiglu":
            o.mot_gate_up_swiglu(x, Mu, Mg, K, *w, y)
        else:
            o.mot_linear(x, Mu, Mg, K, [dict(w_und=w[0], w_gen=w[1], bias_und=b[0],
                                             bias_gen=b[1], y=y)], noalloc=call == "noalloc")
        torch.cuda.synchronize()
        return y.view(torch.int16)
    for call in ("linear", "noalloc", "swiglu"):
        assert torch.equal(run(ops, call), run(contexts[0], call))
    if K % 128 == 0:
        xq, q0, q1 = (torch.from_numpy(rng.integers(-127, 128, s).astype(np.int8)).cuda()
                      for s in ((M, K), (N, K), (N, K)))
        ys = [torch.empty(M, N, dtype=torch.int32, device="cuda") for _ in range(2)]
        for o, y in zip((ops, contexts[0]), ys):
            o.mot_gemm_i8_i32(xq, Mu, Mg, K, [dict(wq_und=q0, wq_gen=q1, y=y)])
        torch.cuda.synchronize()
        assert torch.equal(*ys)


@pytest.mark.parametrize("bm", [128, 192, 256, None])
@pytest.mark.parametrize("M,K,N", [(129, 64, 8), (191, 320, 1000), (256, 2048, 520),
                                   (257, 192, 136), (384, 4096, 264), (385, 448, 128)])
@pytest.mark.parametrize("bits,group", [(4, 32), (4, 64), (8, 32), (8, 64)])
def test_packs_on_the_mid_tiles(ops, contexts, bits, group, M, K, N, bm):
    """Packs of more than 128 rows, read by the tiles (to 256 rows at 4 bits,
    384 at 8) or expanded, with bias: bit-equal to u15h_linear on the
    expansion, at tile edges, one K stage, odd stage counts and splits."""
    pack_equals_expansion(ops if bm is None else contexts[bm], bits, group, M, K, N)


@pytest.mark.parametrize("bits,group,M,K,N", [(4, 32, 224, 87488, 256), (8, 64, 192, 210624, 128)])
def test_packs_of_long_k(ops, bits, group, M, K, N):
    """Sizes where the mid-size and the 256 x 256 tiles' estimates are close:
    the tiles are picked once."""
    pack_equals_expansion(ops, bits, group, M, K, N)


def pack_equals_expansion(o, bits, group, M, K, N):
    rng = np.random.default_rng(M + K + bits + group)
    codes = rng.integers(0, 1 << 32, (N, K * bits // 32), dtype=np.uint64).astype(np.uint32)
    sc, bi = (dev_bf16(rand_bf16_bits(rng, (N, K // group), 0.01)) for _ in range(2))
    qw = (torch.from_numpy(codes.view(np.int32)).cuda(), sc, bi, bits, group)
    x, b = dev_bf16(rand_bf16_bits(rng, (M, K))), dev_bf16(rand_bf16_bits(rng, (N,), 0.5))
    w = torch.empty(N, K, dtype=torch.bfloat16, device="cuda")
    o.dequant_affine(qw, N, K, w)
    y, t = (torch.full((M, N), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    o.linear_q(x, qw, b, y, M, K, N)
    o.linear(x, w, b, t, M, K, N)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), t.view(torch.int16))


@pytest.mark.parametrize("bm", [128, 192, 256])
@pytest.mark.parametrize("M,K,N", [(129, 320, 1000), (200, 4096, 136)])
@pytest.mark.parametrize("bits,group", [(4, 32), (4, 64), (8, 32), (8, 64)])
def test_packs_with_odd_scales(contexts, bits, group, M, K, N, bm):
    """Scales and biases off dword alignment, and an infinite scale and a NaN
    bias: the same bits as u15h_linear on the expansion, NaN where it has
    NaN."""
    rng = np.random.default_rng(M + K + bits + group)
    codes = rng.integers(0, 1 << 32, (N, K * bits // 32), dtype=np.uint64).astype(np.uint32)
    sc = rng.random((N, K // group)).astype(np.float32) * 0.01
    bi = rng.standard_normal((N, K // group)).astype(np.float32) * 0.1
    sc[3, -1], bi[5, 0] = np.inf, np.nan

    def dev(a):
        flat = torch.zeros(a.size + 8, dtype=torch.bfloat16, device="cuda")
        t = flat[1:1 + a.size].view(a.shape)
        t.copy_(dev_bf16(oracle.f32_to_bf16(a)))
        return t
    qw = (torch.from_numpy(codes.view(np.int32)).cuda(), dev(sc), dev(bi), bits, group)
    x = dev_bf16(rand_bf16_bits(rng, (M, K)))
    w = torch.empty(N, K, dtype=torch.bfloat16, device="cuda")
    o = contexts[bm]
    o.dequant_affine(qw, N, K, w)
    y, t = (torch.full((M, N), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    o.linear_q(x, qw, None, y, M, K, N)
    o.linear(x, w, None, t, M, K, N)
    torch.cuda.synchronize()
    nan = torch.isnan(t)
    assert torch.equal(torch.isnan(y), nan) and bool(nan[:, [3, 5]].all())
    assert int(nan.sum()) == 2 * M
    assert torch.equal(y.view(torch.int16)[~nan], t.view(torch.int16)[~nan])


@pytest.mark.parametrize("call,Mu,Mg,K,N", [
    ("linear", 0, 2800, 4096, 3072), ("linear", 333, 1, 2048, 12288),
    ("swiglu", 333, 1, 2048, 6144), ("i8", 333, 257, 8192, 10240),
    ("swiglu", 97, 0, 1536, 128), ("i8", 97, 0, 3072, 128), ("pack", 97, 0, 1536, 256)])
def test_first_call_of_a_context_under_capture(ops, call, Mu, Mg, K, N):
    """Mid-size tiles with a split tail where the 256 x 256 ones have none, few
    rows on tiles, and a pack that is expanded when not captured: captured as
    a context's first call.  Replays with eager work between them equal the
    eager result."""
    g = torch.Generator(device="cuda").manual_seed(Mu + Mg + K)
    M = Mu + Mg

    def rnd(*shape):
        return torch.empty(*shape, dtype=torch.bfloat16, device="cuda").normal_(generator=g)

    def codes(*shape):
        return torch.randint(-127, 128, shape, generator=g, dtype=torch.int8, device="cuda")
    y = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    if call == "pack":
        rows = torch.randint(-2**31, 2**31 - 1, (N, K // 8), generator=g, dtype=torch.int32,
                             device="cuda")
        x, qw = rnd(M, K), (rows, rnd(N, K // 32), rnd(N, K // 32), 4, 32)

        def run(o):
            o.linear_q(x, qw, None, y, M, K, N)
    elif call == "i8":
        xq, q0, q1 = codes(M, K), codes(N, K), codes(N, K)
        sx, s0, s1 = (torch.rand(n, generator=g, device="cuda") for n in (M, N, N))

        def run(o):
            o.mot_gemm_i8(xq, sx, Mu, Mg, K, [dict(wq_und=q0, wq_gen=q1, sw_und=s0, sw_gen=s1,
                                                   y=y)])
    else:
        x, w = rnd(M, K), [rnd(N, K) for _ in range(4 if call == "swiglu" else 2)]

        def run(o):
            if call == "swiglu":
                o.mot_gate_up_swiglu(x, Mu, Mg, K, *w, y)
            else:
                o.mot_linear(x, Mu, Mg, K, [dict(w_und=w[0], w_gen=w[1], y=y)])
    run(ops)
    torch.cuda.synchronize()
    want = y.clone()
    o = u15h.Ops(0)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(o)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))
        run(ops)
    torch.cuda.synchronize()
    o.close()
