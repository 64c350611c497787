"""Parity of the HIP path (through the C ABI) against the oracle, on an MI355X.

Bars: dequantised weights bit-exact; matmul outputs within 1e-3 relative L2 of
the float64 oracle (the fp32-accumulating kernels land near 1e-6, asserted at
2e-5 for fp32 outputs so that a dropped group or a wrong scale cannot hide)."""
import numpy as np
import pytest

from cyb_amd import QMatMul, formats, synth
from cyb_amd.backend import CybqError

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = 1e-3          # the operator's stated tolerance
TIGHT = 2e-5        # what fp32 accumulation actually delivers
FAST = 5e-4         # prefill FAST mode: weights rounded once to f16 (expected ~2e-4)
SUMS = 1e-6         # prefill EXACT mode on integer operands: nothing but fp32 sums of up to 14336 products (measured 5e-8 .. 2e-7)


@pytest.fixture(params=["exact", "fast"])
def prefill_mode(request, backend):
    backend.set_prefill_mode(request.param)
    yield request.param
    backend.set_prefill_mode("fast")


def _bar(mode):
    return TIGHT if mode == "exact" else FAST

TDT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def _quant(oracle, bits, N, K, cfg=21):
    w = synth.weights(cfg, N, K)
    return oracle.quantize(w, bits)


def _x(M, K, dt, cfg=21, outliers=0.0):
    x = torch.from_numpy(synth.activations(cfg, M, K, outliers=outliers)).cuda().to(TDT[dt])
    return x


def _run(backend, qw, x, ydt="f32"):
    M = x.shape[0]
    y = torch.full((M, qw.N), float("nan"), dtype=TDT[ydt], device="cuda")
    backend.matmul(qw, x, y)
    torch.cuda.synchronize()
    return y


def _random_weight(backend, bits, N, K, seed):
    """Every value of q, scales of 0 .. 0.01: the weight and its dequantised values in float64, on the device."""
    rng = np.random.default_rng(seed)
    q = rng.integers(-(1 << (bits - 1)), 1 << (bits - 1), size=(N, K), dtype=np.int8)
    s = (rng.random((N, K // 32), dtype=np.float32) * 0.01).astype(np.float16)
    wd = torch.from_numpy(s).cuda().double().repeat_interleave(32, dim=1) * torch.from_numpy(q).cuda()
    return backend.upload_quantized(q, s.view(np.uint16), bits), wd


# ------------------------------------------------------------------ dequant

@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("layout", [formats.PLANAR, formats.BLOCK_AOS])
@pytest.mark.parametrize("shape", [(1, 32), (17, 160), (16, 128), (100, 4096), (1024, 4096)])
def test_dequant_bit_exact(backend, oracle, bits, layout, shape):
    N, K = shape
    q, s = _quant(oracle, bits, N, K)
    qw = backend.upload_quantized(q, s, bits, layout)
    out = torch.empty((N, K), dtype=torch.float32, device="cuda")
    backend.dequant(qw, out)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy().view(np.uint32), oracle.dequant(q, s).view(np.uint32))
    assert qw.algorithmic_bytes == formats.weight_bytes(bits, N, K)
    qw.free()


# (a slot of the upload ring holds whole 16-row strips, 4 MiB: one short piece, several pieces with a ragged last strip,
# pieces of exactly one strip, and a strip that does not fit a slot at all)
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("layout", [formats.PLANAR, formats.BLOCK_AOS])
def test_upload_many_is_bit_exact_across_pieces(backend, bits, layout):
    rng = np.random.default_rng(5)
    tensors, want = [], []
    for N, K in [(1, 32), (17, 160), (4111, 4096), (2050, 2080), (33, 262144), (19, 524288 + 32)]:
        q = rng.integers(-8 if bits == 4 else -128, 8 if bits == 4 else 128, size=(N, K), dtype=np.int8)
        s = (rng.random((N, K // 32), dtype=np.float32) * 0.01).astype(np.float16).view(np.uint16)
        planar = layout == formats.PLANAR
        tensors.append((bits, layout, N, K, formats.pack_planar(q, bits) if planar else formats.pack_blocks(q, s, bits), s if planar else None, None))
        want.append(formats.dequantize(q, s))
    for ws in (backend.upload_many(tensors), backend.upload_many(tensors[::-1])[::-1]):
        for w, ref in zip(ws, want):
            out = torch.empty(ref.shape, dtype=torch.float32, device="cuda")
            backend.dequant(w, out)
            torch.cuda.synchronize()
            assert np.array_equal(out.cpu().numpy().view(np.uint32), ref.view(np.uint32)), ref.shape
            w.free()
    bad = list(tensors[0])
    bad[3] = 48                                                # K % 32: nothing of the list is made
    with pytest.raises(CybqError):
        backend.upload_many([tensors[1], tuple(bad)])
    assert backend.upload_many([]) == []


@pytest.mark.parametrize("bits", [4, 8])
def test_dequant_exhaustive_scales_and_values(backend, oracle, bits):
    # every finite f16 scale against every representable q (extremes included)
    scales = np.arange(65536, dtype=np.uint16)
    fin = np.isfinite(scales.view(np.float16))
    scales = scales[fin]
    qs = np.arange(-8, 8) if bits == 4 else np.arange(-128, 128)
    reps = -(-len(qs) // 32)
    qrow = np.resize(qs, reps * 32).astype(np.int8)
    q = np.tile(qrow, (len(scales), 1))
    s = np.repeat(scales[:, None], reps, axis=1)
    qw = backend.upload_quantized(q, s, bits)
    out = torch.empty(q.shape, dtype=torch.float32, device="cuda")
    backend.dequant(qw, out)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy().view(np.uint32), oracle.dequant(q, s).view(np.uint32))


# ------------------------------------------------------------ decode (M <= 16)

@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("xdt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 7, 8, 16])
def test_decode_matches_oracle(backend, oracle, bits, xdt, M):
    N, K = 272, 1024
    q, s = _quant(oracle, bits, N, K)
    qw = backend.upload_quantized(q, s, bits)
    x = _x(M, K, xdt, outliers=0.001)
    y = _run(backend, qw, x).cpu().numpy()
    ref = oracle.matmul_f64(q, s, x.float().cpu().numpy())
    err = oracle.rel_l2(y, ref)
    assert err < TIGHT, err
    # and against the fp32-accumulating CPU path itself
    y32 = oracle.matmul_f32(q, s, x.float().cpu().numpy())
    assert oracle.rel_l2(y, y32.astype(np.float64)) < TIGHT


@pytest.mark.parametrize("shape", [(1, 32), (5, 64), (16, 128), (33, 160), (1000, 2080), (48, 32768)])
def test_decode_ragged_shapes(backend, oracle, shape):
    N, K = shape
    q, s = _quant(oracle, 4, N, K)
    qw = backend.upload_quantized(q, s, 4, formats.BLOCK_AOS)
    for M in (1, 5, 16):
        x = _x(M, K, "f16")
        y = _run(backend, qw, x).cpu().numpy()
        assert not np.isnan(y).any()
        assert oracle.rel_l2(y, oracle.matmul_f64(q, s, x.float().cpu().numpy())) < TIGHT


def test_decode_seven_strips_per_workgroup(backend, oracle):
    # N = 7 * 16 * 256: on a 256-CU part the batched-rows kernel gives every workgroup seven strips
    N, K = 28672, 256
    q, s = _quant(oracle, 4, N, K)
    qw = backend.upload_quantized(q, s, 4)
    for M in (4, 16):
        x = _x(M, K, "f16")
        y = _run(backend, qw, x).cpu().numpy()
        assert oracle.rel_l2(y, oracle.matmul_f64(q, s, x.float().cpu().numpy())) < TIGHT
    r = torch.from_numpy(synth.activations(34, 16, N)).cuda()
    y2 = torch.empty((16, N), dtype=torch.float32, device="cuda")
    backend.matmul_ex(qw, x, y2, "add", r)
    torch.cuda.synchronize()
    assert torch.equal(y2, torch.from_numpy(y).cuda() + r)
    # gate / up pairs of that width: eight strips (four pairs) per workgroup
    h = N // 2
    pair = backend.fuse_pairs(backend.upload_quantized(q[:h], s[:h], 4), backend.upload_quantized(q[h:], s[h:], 4))
    for M in (3, 8, 16):
        y3 = torch.empty((M, h), dtype=torch.float32, device="cuda")
        backend.matmul_ex(pair, x[:M].contiguous(), y3, "swiglu")
        torch.cuda.synchronize()
        yd = torch.from_numpy(y[:M]).cuda().double()
        ref = torch.nn.functional.silu(yd[:, :h]) * yd[:, h:]
        assert ((y3.double() - ref).norm() / ref.norm()).item() < TIGHT, M


@pytest.mark.parametrize("bits,xdt", [(4, "f16"), (4, "bf16"), (8, "f16"), (8, "bf16")])
@pytest.mark.parametrize("N", [14336, 28672, 8192])
def test_decode_batched_rows_wide_shapes(backend, oracle, bits, xdt, N):
    """Wide outputs give a workgroup of the batched-rows kernel 4, 7 or 2 strips; which shape runs
    depends on block type and activation type (register budget), and the x load pattern on the
    batch (up to 4 / 8 / 16 rows per load).  K = 384 is three K tiles: a partly filled slab."""
    K = 384
    q, s = _quant(oracle, bits, N, K, cfg=23)
    qw = backend.upload_quantized(q, s, bits)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    y1 = None
    try:
        for M in (16, 8, 5, 4):
            x = _x(16, K, xdt, cfg=24)[:M].contiguous()
            ref = x.double() @ wd.T
            backend.set_gemv_tuning(0, 0, 0)              # whichever kernel the library picks for this batch
            y = _run(backend, qw, x)
            err = ((y.double() - ref).norm() / ref.norm()).item()
            assert err < TIGHT, (M, err)
            # within the batched-rows kernel a row's bits do not depend on the batch it travels in
            # (nor on the x load pattern that follows from it)
            backend.set_gemv_tuning(0, 1, 0)
            y = _run(backend, qw, x)
            if y1 is None:
                y1 = y
            else:
                assert torch.equal(y, y1[:M]), M
    finally:
        backend.set_gemv_tuning(0, 0, 0)


@pytest.mark.parametrize("bits,xdt", [(4, "f16"), (4, "bf16"), (8, "f16"), (8, "bf16")])
@pytest.mark.parametrize("shape", [(14336, 384), (28672, 384), (8192, 384), (512, 4096 + 128), (80, 14336), (33, 160)])
def test_decode_17_to_32_rows_in_one_pass(backend, oracle, bits, xdt, shape):
    """17 .. 32 rows of 16-bit activations run the batched-rows kernel with two row blocks: the
    weights stream once.  A row's bits are those of the same kernel at 16 rows or fewer."""
    N, K = shape
    q, s = _quant(oracle, bits, N, K, cfg=27)
    qw = backend.upload_quantized(q, s, bits)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    x = _x(32, K, xdt, cfg=28)
    try:
        backend.set_gemv_tuning(0, 1, 0)                 # the batched-rows kernel for the 16-row halves too
        lo, hi = _run(backend, qw, x[:16].contiguous()), _run(backend, qw, x[16:].contiguous())
        backend.set_gemv_tuning(0, 0, 0)
        for M in (32, 17, 24):
            y = _run(backend, qw, x[:M].contiguous())
            ref = x[:M].double() @ wd.T
            err = ((y.double() - ref).norm() / ref.norm()).item()
            assert err < TIGHT, (M, err)
            assert torch.equal(y[:16], lo), M
            assert torch.equal(y[16:], hi[:M - 16]), M
    finally:
        backend.set_gemv_tuning(0, 0, 0)
    if N % 32 == 0 and K == 384:
        # epilogues in the same kernel: residual add, and SwiGLU over a gate / up pair
        M = 21
        r = torch.from_numpy(synth.activations(35, M, N)).cuda()
        y = _run(backend, qw, x[:M].contiguous())
        y2 = torch.empty((M, N), dtype=torch.float32, device="cuda")
        backend.matmul_ex(qw, x[:M].contiguous(), y2, "add", r)
        torch.cuda.synchronize()
        assert torch.equal(y2, y + r)
        h = N // 2
        g = backend.upload_quantized(q[:h], s[:h], bits)
        u = backend.upload_quantized(q[h:], s[h:], bits)
        pair = backend.fuse_pairs(g, u)
        y3 = torch.empty((M, h), dtype=torch.float32, device="cuda")
        backend.matmul_ex(pair, x[:M].contiguous(), y3, "swiglu")
        torch.cuda.synchronize()
        yd = y.double()
        ref = torch.nn.functional.silu(yd[:, :h]) * yd[:, h:]
        assert ((y3.double() - ref).norm() / ref.norm()).item() < TIGHT


# the kernel whose workgroups stay: four or eight waves of two to four K tiles, the last one missing for some waves or ragged;
# an odd number of strips, the last one ragged; one, two and three rounds of pairs; both row blocks
@pytest.mark.parametrize("bits,xdt", [(4, "f16"), (4, "bf16"), (8, "f16"), (8, "bf16")])
@pytest.mark.parametrize("shape", [(6144, 1024), (6149, 1056), (10241, 1888), (6160, 2048), (6149, 2080), (17000, 2592), (10241, 3104), (6144, 4096)])
def test_decode_rows_streamed_by_staying_workgroups(backend, bits, xdt, shape):
    N, K = shape
    g = torch.Generator(device="cuda").manual_seed(N + K)
    w = torch.empty((N, K), device="cuda").normal_(0.0, 0.02, generator=g)
    qd = torch.empty(N * K * bits // 8, dtype=torch.uint8, device="cuda")
    sd = torch.empty(N * (K // 32), dtype=torch.int16, device="cuda")
    backend.quantize(bits, w, N, K, qd, sd)
    qw = backend.weight_from_device(bits, N, K, qd, sd)
    backend.dequant(qw, w)
    wd = w.double()
    x = torch.empty((32, K), device="cuda").normal_(generator=g).to(TDT[xdt])
    r = torch.empty((32, N), device="cuda").normal_(generator=g)
    gamma = (1.0 + 0.25 * torch.empty(K, device="cuda").normal_(generator=g)).to(torch.float16)
    plain = x.double() @ wd.t()
    rstd = 1.0 / torch.sqrt((x.double() ** 2).mean(dim=1, keepdim=True) + 1e-5)
    normed = ((x.float() * gamma.float()).to(TDT[xdt]).double() @ wd.t()) * rstd
    rel = lambda a, b: ((a.double() - b).norm() / b.norm()).item()
    full = torch.empty((32, N), device="cuda")
    backend.matmul(qw, x, full)
    for M in (3, 8, 9, 16, 17, 32):
        y = torch.full((M, N), float("nan"), device="cuda")
        backend.matmul(qw, x[:M].contiguous(), y)
        assert rel(y, plain[:M]) < TIGHT, M
        backend.matmul_ex(qw, x[:M].contiguous(), y, "add", r[:M].contiguous())
        assert rel(y, plain[:M] + r[:M].double()) < TIGHT, M
        if M <= 16 or xdt == "f16":           # (17 bf16 rows or more with a norm are not this kernel's)
            backend.matmul_norm(qw, x[:M].contiguous(), gamma, 1e-5, y)
            # (K of four tiles per wave: registers for x or for gamma, not both; those calls are FAST ones)
            four = -(-K // 128) > (12 if K <= 1920 else 24)
            assert rel(y, normed[:M]) < (FAST if M > 16 and four else TIGHT), M
    half = N // 32 * 16
    qb, sb = half * K * bits // 8, half * (K // 32)
    pair = backend.fuse_pairs(backend.weight_from_device(bits, half, K, qd[:qb], sd[:sb]),
                              backend.weight_from_device(bits, half, K, qd[qb:2 * qb], sd[sb:2 * sb]))
    for M in (5, 16, 30):
        y = torch.full((M, half), float("nan"), device="cuda")
        backend.matmul_ex(pair, x[:M].contiguous(), y, "swiglu")
        assert rel(y, torch.nn.functional.silu(plain[:M, :half]) * plain[:M, half:2 * half]) < TIGHT, M


# two kernels share these shapes by row count: full rounds of four and two strips up to 16 rows and staying workgroups beyond (an odd
# last strip, a ragged K tile, waves with three and four K tiles), the reverse for gate / up pairs (four waves too),
# seven strips per CU, several rounds per CU, and shapes that one kernel has for itself; a few strips more than CUs, with two strips to a
# workgroup from 17 rows or from three
@pytest.mark.parametrize("bits,N,K,pair", [(4, 14336, 4096, False), (4, 14341, 4064, False), (4, 8180, 3104, False), (4, 32000, 3200, False),
                                           (4, 28672, 4096, False), (4, 32784, 3200, False), (4, 10241, 3104, False), (4, 20480, 4096, True),
                                           (4, 6176, 3104, True), (4, 20480, 1792, True), (4, 6176, 1664, True), (8, 14336, 4096, False),
                                           (8, 8224, 3104, True), (4, 6144, 928, False), (4, 28640, 2048, True), (4, 28656, 4096, False), (8, 6144, 928, False),
                                           (4, 4130, 1024, False), (4, 5120, 4096, False), (4, 6127, 12320, False)])
@pytest.mark.parametrize("xdt", ["f16", "bf16"])
def test_a_row_keeps_its_bits_from_3_to_32_rows(backend, bits, N, K, pair, xdt):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    rows, parts, wd = N // 2 if pair else N, [], []
    for _ in range(2 if pair else 1):
        w = torch.empty((rows, K), device="cuda").normal_(0.0, 0.02, generator=g)
        qd = torch.empty(rows * K * bits // 8, dtype=torch.uint8, device="cuda")
        sd = torch.empty(rows * (K // 32), dtype=torch.int16, device="cuda")
        backend.quantize(bits, w, rows, K, qd, sd)
        parts.append(backend.weight_from_device(bits, rows, K, qd, sd))
        backend.dequant(parts[-1], w)
        wd.append(w.double())
    qw = backend.fuse_pairs(*parts) if pair else parts[0]
    x = torch.empty((32, K), device="cuda").normal_(generator=g).to(TDT[xdt])
    ref = x.double() @ wd[0].t()
    if pair:
        ref = torch.nn.functional.silu(ref) * (x.double() @ wd[1].t())
    try:
        for mode in ("stream", "exact"):
            backend.set_decode_mode(mode)
            full = torch.full((32, rows), float("nan"), device="cuda")
            backend.matmul_ex(qw, x, full, "swiglu" if pair else "none")
            assert ((full.double() - ref).norm() / ref.norm()).item() < TIGHT, mode
            for M in (3, 4, 8, 9, 16, 17, 24):
                y = torch.full((M, rows), float("nan"), device="cuda")
                backend.matmul_ex(qw, x[:M].contiguous(), y, "swiglu" if pair else "none")
                assert torch.equal(y, full[:M]), (mode, M)
    finally:
        backend.set_decode_mode("stream")


# a folded norm on wide outputs, up to 16 rows, every load pattern: two, three and four K tiles per wave with waves that
# have one less, four waves, ragged K and N, a half-filled last pair; more than two steps per workgroup.  gamma is a power of two, so x * gamma is
# exact and what is left is the sums: up to 128 products per fp32 step, for bf16 rows with the bias in them (8 .. 128 times the weights), 1e-6 and
# less; f16 rows meet the exact integers in either mode, whatever kernel has the shape: the same bits, and a weight of zeros gives exact zeros
@pytest.mark.parametrize("bits,N,K,pair", [(4, 6149, 4064, False), (4, 12288, 3104, True), (4, 20000, 4096, True), (4, 32784, 4096, False),
                                           (4, 14341, 3488, False), (4, 6176, 2080, True), (4, 28689, 3072, False), (4, 8200, 1120, False),
                                           (4, 6149, 1664, False), (8, 6149, 4064, False), (8, 12320, 1120, True)])
@pytest.mark.parametrize("xdt", ["f16", "bf16"])
def test_staying_workgroups_with_a_folded_norm(backend, bits, N, K, pair, xdt):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    rows, parts, wd = N // 2 if pair else N, [], []
    for _ in range(2 if pair else 1):
        w = torch.empty((rows, K), device="cuda").normal_(0.0, 0.02, generator=g)
        qd = torch.empty(rows * K * bits // 8, dtype=torch.uint8, device="cuda")
        sd = torch.empty(rows * (K // 32), dtype=torch.int16, device="cuda")
        backend.quantize(bits, w, rows, K, qd, sd)
        parts.append(backend.weight_from_device(bits, rows, K, qd, sd))
        backend.dequant(parts[-1], w)
        wd.append(w.double())
    qw = backend.fuse_pairs(*parts) if pair else parts[0]
    gamma = torch.exp2(torch.randint(-1, 2, (K,), device="cuda", generator=g).float())
    zero = backend.weight_from_device(bits, rows, K, torch.zeros_like(qd), sd)
    first = {}
    try:
        for mode in ("stream", "exact"):
            backend.set_decode_mode(mode)
            for i, M in enumerate((3, 4, 5, 8, 9, 16)):
                x = torch.empty((M, K), device="cuda").normal_(generator=g.manual_seed(M)).to(TDT[xdt])
                xn = x.double() * gamma.double() / (x.double().square().mean(1, keepdim=True) + 1e-5).sqrt()
                ref = xn @ wd[0].t()
                if pair:
                    ref = torch.nn.functional.silu(ref) * (xn @ wd[1].t())
                y = torch.full((M, rows), float("nan"), device="cuda")
                gd = (torch.float16, torch.float32, torch.bfloat16)[i % 3]
                backend.matmul_norm(qw, x, gamma.to(gd), 1e-5, y, "swiglu" if pair else "none")
                # (a pair's error is u silu'(g) dg + silu(g) du with |silu'| <= 1.1 and |silu(g)| <= |g|, against |silu(g) u|, which for normal g is
                # about 0.6 |g u|: at most 2.1 / 0.6 = 3.5 times that of its sums)
                assert ((y.double() - ref).norm() / ref.norm()).item() < (7e-6 if pair else 2e-6), (mode, M)
                if xdt == "f16":
                    assert torch.equal(y, first.setdefault(M, y)), (mode, M)
                    y0 = torch.full((M, rows), float("nan"), device="cuda")
                    backend.matmul_norm(zero, x, gamma.to(gd), 1e-5, y0)
                    assert (y0 == 0).all(), (mode, M)
    finally:
        backend.set_decode_mode("stream")


# fp32 rows in the batched-rows kernel (decode tuning 1 forces it) and wherever the library sends them: one, two and four strips to a workgroup, two and
# four K tiles per wave, slabs partly filled, one K tile, ragged K and N, each load pattern.  The two halves of a row keep 22 bits of every value
# (2^-23 of it left out at most) and the sums are fp32: 1e-6; a pair's error is at most 3.5 times that (above).  A row has the same bits in
# the LDS kernel (decode tuning 2), alone and in any batch, and as one of many in EXACT mode; with a norm in any batch of 3 .. 16 and in EXACT mode
@pytest.mark.parametrize("bits,N,K", [(4, 33, 96), (4, 500, 1056), (4, 4096, 2048 + 32), (4, 6149, 4064), (4, 12304, 3104), (4, 4101, 14336), (4, 300, 12384), (8, 33, 160),
                                      (8, 4096, 4096 + 96), (8, 12304, 1120), (8, 6160, 8192)])
def test_batched_rows_of_fp32(backend, bits, N, K):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    w = torch.empty((N, K), device="cuda").normal_(0.0, 0.02, generator=g)
    qd = torch.empty(N * K * bits // 8, dtype=torch.uint8, device="cuda")
    sd = torch.empty(N * (K // 32), dtype=torch.int16, device="cuda")
    backend.quantize(bits, w, N, K, qd, sd)
    qw = backend.weight_from_device(bits, N, K, qd, sd)
    backend.dequant(qw, w)
    x = torch.empty((16, K), device="cuda").normal_(generator=g)
    gamma = 1.0 + 0.25 * torch.empty(K, device="cuda").normal_(generator=g)
    res = torch.empty((16, N), device="cuda").normal_(generator=g)
    rms = (x.double().square().mean(1, keepdim=True) + 1e-5).sqrt()
    plain, normed = x.double() @ w.double().t(), (x.double() * gamma.double() / rms) @ w.double().t()
    rel = lambda y, ref: ((y.double() - ref).norm() / ref.norm()).item()
    half = N // 2 // 16 * 16
    parts = [backend.weight_from_device(bits, half, K, qd[i * half * K * bits // 8:], sd[i * half * (K // 32):]) for i in (0, 1)] if half else []
    pair = backend.fuse_pairs(*parts) if half else None
    first = {}
    try:
        for tuning in (1, 0, 2):
            backend.set_gemv_tuning(0, tuning, 0)
            for M in (16, 9, 8, 5, 4, 3, 2, 1):
                y = torch.full((M, N), float("nan"), device="cuda")
                backend.matmul(qw, x[:M].contiguous(), y)
                assert rel(y, plain[:M]) < 1e-6, (tuning, M)
                assert torch.equal(y, first.setdefault("plain", y)[:M]), (tuning, M)
                y = torch.full((M, N), float("nan"), device="cuda")
                backend.matmul_norm(qw, x[:M].contiguous(), gamma, 1e-5, y, "add", res[:M].contiguous())
                assert rel(y, normed[:M] + res[:M].double()) < 1e-6, (tuning, M)
                if tuning != 2 and M > 2:
                    assert torch.equal(y, first.setdefault("normed", y)[:M]), (tuning, M)
                if pair is not None:
                    y = torch.full((M, half), float("nan"), device="cuda")
                    backend.matmul_ex(pair, x[:M].contiguous(), y, "swiglu")
                    ref = torch.nn.functional.silu(plain[:M, :half]) * plain[:M, half:2 * half]
                    assert rel(y, ref) < 3.5e-6, (tuning, M)
                    assert torch.equal(y, first.setdefault("pair", y)[:M]), (tuning, M)
        backend.set_gemv_tuning(0, 0, 0)
        backend.set_prefill_mode("exact")
        for M in (17, 18, 35):
            rows = torch.arange(M, device="cuda") % 16
            y = torch.full((M, N), float("nan"), device="cuda")
            backend.matmul(qw, x[rows].contiguous(), y)
            assert torch.equal(y, first["plain"][rows]), M
            backend.matmul_norm(qw, x[rows].contiguous(), gamma, 1e-5, y, "add", res[rows].contiguous())
            assert torch.equal(y, first["normed"][rows]), M
    finally:
        backend.set_gemv_tuning(0, 0, 0)
        backend.set_prefill_mode("fast")


# a few strips more than CUs, or than twice as many (256 CUs: two and four strips to a workgroup), and K split over workgroups up to one per CU: an odd
# last strip, ragged N and K, up to 32 rows
@pytest.mark.parametrize("bits,N,K", [(4, 4096, 12288), (4, 4100, 12288), (4, 4112, 2048), (4, 6128, 4096 + 32), (4, 4130, 1024), (4, 8200, 4128), (4, 10224, 4128),
                                      (8, 4130, 2080), (8, 6128, 4128)])
@pytest.mark.parametrize("xdt", ["f16", "bf16", "f32"])
def test_decode_a_few_strips_more_than_cus(backend, bits, N, K, xdt):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    w = torch.empty((N, K), device="cuda").normal_(0.0, 0.02, generator=g)
    qd = torch.empty(N * K * bits // 8, dtype=torch.uint8, device="cuda")
    sd = torch.empty(N * (K // 32), dtype=torch.int16, device="cuda")
    backend.quantize(bits, w, N, K, qd, sd)
    qw = backend.weight_from_device(bits, N, K, qd, sd)
    backend.dequant(qw, w)
    for M in (3, 8, 16) + ((17, 32) if xdt != "f32" else ()):
        x = torch.empty((M, K), device="cuda").normal_(generator=g).to(TDT[xdt])
        r = torch.empty((M, N), device="cuda").normal_(generator=g)
        y = torch.full((M, N), float("nan"), device="cuda")
        backend.matmul_ex(qw, x, y, "add", r)
        ref = x.double() @ w.double().t() + r.double()
        assert ((y.double() - ref).norm() / ref.norm()).item() < TIGHT, M


# with the same operands (f16 rows and exact integers; Q8) the staying workgroups and the batched-rows kernel (decode tuning 5: the
# former never) give the same bits: every epilogue and output type, a folded norm where both load the rows alike
# (Q4 bf16 rows: another order of sums; the test above has the shapes that the kernels share)
@pytest.mark.parametrize("xdt,bits,N,K", [("f16", 4, 6144, 4096), ("f16", 4, 10241, 3104), ("f16", 4, 8192, 2560), ("f16", 4, 6160, 2048),
                                          ("f16", 4, 6149, 1056)] + [(t, 8, n, k) for t in ("f16", "bf16")
                                                                     for n, k in ((14336, 4096), (6149, 2080), (20480, 1792))])
def test_staying_workgroups_against_the_batched_rows_kernel(backend, bits, N, K, xdt):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    w = torch.empty((N, K), device="cuda").normal_(0.0, 0.02, generator=g)
    qd = torch.empty(N * K * bits // 8, dtype=torch.uint8, device="cuda")
    sd = torch.empty(N * (K // 32), dtype=torch.int16, device="cuda")
    backend.quantize(bits, w, N, K, qd, sd)
    qw = backend.weight_from_device(bits, N, K, qd, sd)
    gamma = (1.0 + 0.25 * torch.empty(K, device="cuda").normal_(generator=g)).to(torch.float16)
    try:
        backend.set_decode_mode("exact")
        for M in (5, 8, 9, 16, 17, 32):
            x = torch.empty((M, K), device="cuda").normal_(generator=g).to(TDT[xdt])
            for ydt in ("f32", "f16", "bf16"):
                r = torch.empty((M, N), device="cuda").normal_(generator=g).to(TDT[ydt])
                outs = []
                for tuning in (0, 5):
                    backend.set_gemv_tuning(0, tuning, 0)
                    ys = [torch.full((M, N), float("nan"), dtype=TDT[ydt], device="cuda") for _ in range(3)]
                    backend.matmul(qw, x, ys[0])
                    backend.matmul_ex(qw, x, ys[1], "add", r)
                    if M <= 16 and K > 1920:             # (four waves load up to 16 rows in one form)
                        backend.matmul_norm(qw, x, gamma, 1e-5, ys[2])
                    torch.cuda.synchronize()
                    outs.append(ys)
                for a, b in zip(*outs):
                    assert torch.equal(a, b) or a.isnan().all() and b.isnan().all(), (M, ydt)
    finally:
        backend.set_gemv_tuning(0, 0, 0)
        backend.set_decode_mode("stream")


# a folded norm: the squares of a row are summed as the row is loaded, and the workgroups that stay load 3 .. 8 rows in one form
@pytest.mark.parametrize("bits,N,K", [(4, 6149, 2080), (4, 12288, 3072), (4, 20000, 4096), (8, 6149, 4064), (8, 8192, 2048)])
@pytest.mark.parametrize("xdt", ["f16", "bf16"])
def test_a_row_keeps_its_bits_from_3_to_8_rows_with_a_folded_norm(backend, bits, N, K, xdt):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    qd = torch.randint(0, 256, (N * K * bits // 8,), dtype=torch.uint8, device="cuda", generator=g)
    sd = (0.01 * torch.rand(N * (K // 32), device="cuda", generator=g)).half().view(torch.int16)
    w = backend.weight_from_device(bits, N, K, qd, sd)
    x = torch.empty((8, K), device="cuda").normal_(generator=g).to(TDT[xdt])
    gamma = 1.0 + 0.25 * torch.empty(K, device="cuda").normal_(generator=g)
    full = torch.full((8, N), float("nan"), device="cuda")
    backend.matmul_norm(w, x, gamma, 1e-5, full)
    for M in (3, 4, 5):
        y = torch.full((M, N), float("nan"), device="cuda")
        backend.matmul_norm(w, x[:M].contiguous(), gamma, 1e-5, y)
        assert torch.equal(y, full[:M]), M


# f16 rows that meet the exact integers in either decode mode, two strips to a workgroup or not: fewer than one and a half strips per CU (the
# shortest K from 17 rows), and pairs of seven strips per CU or eight and more.  The same bits in both modes, and zeros from zeros
@pytest.mark.parametrize("N,K,pair", [(4112, 160, False), (4224, 1024, False), (5120, 4096, False), (6127, 2080, False), (4224, 12320, False),
                                      (28672, 4096, True), (32800, 3104, True), (40000, 3616, True)])
def test_f16_rows_with_integers_in_either_mode(backend, N, K, pair):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    rows = N // 2 if pair else N
    qd = torch.randint(0, 256, (rows * K // 2,), dtype=torch.uint8, device="cuda", generator=g)
    sd = (0.01 * torch.rand(rows * (K // 32), device="cuda", generator=g)).half().view(torch.int16)
    ws = [[backend.weight_from_device(4, rows, K, q, sd) for _ in range(2 if pair else 1)] for q in (qd, torch.zeros_like(qd))]
    w, zero = [backend.fuse_pairs(*p) if pair else p[0] for p in ws]
    try:
        for M in (3, 8, 9, 16) + (() if pair else (17, 32)):
            x = torch.empty((M, K), device="cuda").normal_(generator=g).half()
            ys = []
            for mode in ("stream", "exact"):
                backend.set_decode_mode(mode)
                for v in (w, zero):
                    y = torch.full((M, rows), float("nan"), device="cuda")
                    backend.matmul_ex(v, x, y, "swiglu" if pair else "none")
                    ys.append(y)
            assert torch.equal(ys[0], ys[2]) and (ys[1] == 0).all() and (ys[3] == 0).all(), M
    finally:
        backend.set_decode_mode("stream")


@pytest.mark.parametrize("N", [8192, 12288])
def test_decode_modes_in_the_batched_rows_kernel(backend, oracle, N):
    """3 .. 32 f16 rows on outputs wide enough for two / four strips per workgroup: STREAM feeds the Q4
    weights as f16 subnormals there too (bias off through the MFMA's C operand, one bias product per K
    tile for all strips), EXACT the integer operands; both inside the tight bar, and not the same bits."""
    K = 640
    q, s = _quant(oracle, 4, N, K, cfg=29)
    qw = backend.upload_quantized(q, s, 4)
    qz = backend.upload_quantized(np.zeros((N, K), np.int8), s, 4)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    x = _x(32, K, "f16", cfg=30)
    try:
        for M in (3, 8, 16, 24, 32):
            xm = x[:M].contiguous()
            ref = xm.double() @ wd.T
            outs = {}
            for mode in ("stream", "exact"):
                backend.set_decode_mode(mode)
                y = _run(backend, qw, xm)
                err = ((y.double() - ref).norm() / ref.norm()).item()
                assert err < (TIGHT if mode == "stream" else 1e-6), (M, mode, err)
                outs[mode] = y
                z = _run(backend, qz, xm)
                if mode == "exact":
                    assert not z.any()
                else:
                    assert z.abs().max().item() < 1e-4 * ref.abs().mean().item()
            assert not torch.equal(outs["stream"], outs["exact"]), M
            # bf16 rows on the same strips: biased operands, the bias product shared by a tile's strips
            xb = _x(M, K, "bf16", cfg=31)
            yb = _run(backend, qw, xb)
            refb = xb.double() @ wd.T
            assert ((yb.double() - refb).norm() / refb.norm()).item() < TIGHT, M
            assert _run(backend, qz, xb).abs().max().item() < 1e-4 * refb.abs().mean().item()      # (the bias cancels to rounding)
    finally:
        backend.set_decode_mode("stream")


@pytest.mark.parametrize("xdt", ["f16", "bf16"])
def test_decode_long_k_split_over_workgroups(backend, oracle, xdt):
    """About one strip per CU and a long K: from twelve rows on the batched-rows kernel splits K four ways over
    workgroups, partial sums meet in slabs and the workgroup that arrives last adds them in split order.
    Ragged N (a last strip of 8 rows, a strip group of one strip) and a K whose tiles do not divide by four;
    against float64, run to run (the ticket is back at zero), across batch sizes, with the residual epilogue,
    with exact operands, and against the kernel without the split."""
    N, K = 193 * 16 - 8, 97 * 128
    q, s = _quant(oracle, 4, N, K, cfg=45)
    qw = backend.upload_quantized(q, s, 4)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    x = _x(32, K, xdt, cfg=46)
    ref = x.double() @ wd.T
    try:
        y32 = _run(backend, qw, x)
        assert ((y32.double() - ref).norm() / ref.norm()).item() < TIGHT
        for _ in range(3):
            assert torch.equal(_run(backend, qw, x), y32)
        for M in (12, 16, 17, 24):                       # one and two row blocks: a row keeps its bits
            assert torch.equal(_run(backend, qw, x[:M].contiguous()), y32[:M]), M
        backend.set_gemv_tuning(0, 4, 0)                 # the split from three rows on (the narrower x load patterns)
        for M in (3, 5, 8):
            assert torch.equal(_run(backend, qw, x[:M].contiguous()), y32[:M]), M
        backend.set_gemv_tuning(0, 3, 0)                 # never split: another order of summation, the same sums
        y_plain = _run(backend, qw, x)
        assert not torch.equal(y_plain, y32)
        assert ((y_plain.double() - y32.double()).norm() / ref.norm()).item() < 2e-6
        backend.set_gemv_tuning(0, 0, 0)
        r = torch.from_numpy(synth.activations(47, 32, N)).cuda()
        ya = torch.empty((32, N), dtype=torch.float32, device="cuda")
        backend.matmul_ex(qw, x, ya, "add", r)
        torch.cuda.synchronize()
        assert torch.equal(ya, y32 + r)
        for ydt in ("f16", "bf16"):
            assert torch.equal(_run(backend, qw, x, ydt), y32.to(TDT[ydt]))
        backend.set_decode_mode("exact")
        ye = _run(backend, qw, x[:16].contiguous())
        assert ((ye.double() - ref[:16]).norm() / ref[:16].norm()).item() < (1e-6 if xdt == "f16" else TIGHT)
        # recorded into a graph (no allocation, no memset: the ticket resets itself) and replayed
        backend.set_decode_mode("stream")
        yg = torch.zeros((32, N), dtype=torch.float32, device="cuda")
        side = torch.cuda.Stream()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            backend.matmul(qw, x, yg, stream=torch.cuda.current_stream().cuda_stream)
        for _ in range(3):
            yg.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(yg, y32)
            assert torch.equal(_run(backend, qw, x), y32)            # eager calls between the replays
    finally:
        backend.set_gemv_tuning(0, 0, 0)
        backend.set_decode_mode("stream")
    qw.free()


def test_decode_long_k_uses_several_slabs(backend, oracle):
    # M * K * 2 B exceeds the kernel's LDS budget: x is staged slab by slab
    N, K = 64, 14336
    q, s = _quant(oracle, 4, N, K)
    qw = backend.upload_quantized(q, s, 4)
    for M, xdt in ((16, "f16"), (8, "f32"), (3, "bf16")):
        x = _x(M, K, xdt)
        y = _run(backend, qw, x).cpu().numpy()
        assert oracle.rel_l2(y, oracle.matmul_f64(q, s, x.float().cpu().numpy())) < TIGHT


@pytest.mark.parametrize("bits", [4, 8])
def test_decode_every_kernel_variant(backend, oracle, bits):
    # the launch heuristics pick among one-shot (4 / 8 / 16 tiles in flight) and
    # streaming (2 / 4 tiles per batch) variants; force each of them
    N, K = 80, 4096
    q, s = _quant(oracle, bits, N, K)
    qw = backend.upload_quantized(q, s, bits)
    try:
        for M in (1, 2, 4, 9):
            x = _x(M, K, "f16")
            ref = oracle.matmul_f64(q, s, x.float().cpu().numpy())
            for waves in (1, 2, 4, 8, 16):
                for unroll in (0, 2, 4):
                    backend.set_gemv_tuning(waves, 2, unroll)       # the LDS kernel, every variant
                    y = _run(backend, qw, x).cpu().numpy()
                    err = oracle.rel_l2(y, ref)
                    assert err < TIGHT, (M, waves, unroll, err)
                backend.set_gemv_tuning(waves, 1, 0)                # the x-in-registers kernel
                y2 = _run(backend, qw, x).cpu().numpy()
                assert oracle.rel_l2(y2, ref) < TIGHT, (M, waves)
                assert np.array_equal(y2, _run(backend, qw, x).cpu().numpy()), (M, waves)   # reproducible
    finally:
        backend.set_gemv_tuning(0, 0, 0)


def test_decode_batched_rows_equal_single_rows_bitwise(backend, oracle):
    """Within one kernel a row's bits do not depend on the batch it travels in."""
    N, K = 512, 4096
    q, s = _quant(oracle, 4, N, K)
    qw = backend.upload_quantized(q, s, 4)
    x = _x(16, K, "f16")
    try:
        for kernel, batch in ((2, 4), (2, 16), (1, 16), (1, 7)):      # LDS kernel, x-in-registers kernel
            backend.set_gemv_tuning(0, kernel, 0)
            yb = _run(backend, qw, x[:batch].contiguous())
            for m in (0, batch // 2, batch - 1):
                y1 = _run(backend, qw, x[m:m + 1].contiguous())
                assert torch.equal(y1[0], yb[m]), (kernel, batch, m)
            assert torch.equal(_run(backend, qw, x[:batch].contiguous()), yb)     # and run to run
    finally:
        backend.set_gemv_tuning(0, 0, 0)
    # the automatic choice (LDS kernel for one or two rows, registers beyond) is deterministic too
    y16 = _run(backend, qw, x)
    assert torch.equal(_run(backend, qw, x), y16)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("shape", [(64, 128), (48, 160), (100, 4096 + 96), (4096, 4096), (256, 14336), (64, 11008),
                                   (32, 16384), (16, 24576), (16, 32768)])
@pytest.mark.parametrize("xdt", ["f16", "bf16"])
def test_one_row_kernel_shapes(backend, oracle, bits, shape, xdt):
    """One and two f16 / bf16 rows (subnormal weight operands - bf16: 128 + u -, bias removed inside the accumulation; the 16
    rows of an activation operand are 1 / 2 batch rows x 16 / 8 scale groups): whole and ragged
    sets of K tiles, one to three sets per wave, and K beyond what the kernel serves (3 and 4 rows
    take the batched-rows kernel)."""
    N, K = shape
    q, s = _quant(oracle, bits, N, K)
    qw = backend.upload_quantized(q, s, bits, formats.BLOCK_AOS if N % 32 else formats.PLANAR)
    x4 = _x(4, K, xdt, outliers=0.001)
    ref = oracle.matmul_f64(q, s, x4.float().cpu().numpy())
    for M in (1, 2, 3, 4):
        x = x4[:M].contiguous()
        y = _run(backend, qw, x)
        assert oracle.rel_l2(y.cpu().numpy(), ref[:M]) < TIGHT, M
        assert torch.equal(_run(backend, qw, x), y)                 # reproducible
        for ydt in ("f16", "bf16"):
            assert torch.equal(_run(backend, qw, x, ydt), y.to(TDT[ydt]))
        # fused epilogues of the same kernel: residual add, and SwiGLU where the rows pair up
        r = torch.from_numpy(synth.activations(36, M, N)).cuda()
        y2 = torch.empty((M, N), dtype=torch.float32, device="cuda")
        backend.matmul_ex(qw, x, y2, "add", r)
        torch.cuda.synchronize()
        assert torch.equal(y2, y + r), M
    if N % 32 == 0 and N >= 64:
        h = N // 2
        pair = backend.fuse_pairs(backend.upload_quantized(q[:h], s[:h], bits), backend.upload_quantized(q[h:], s[h:], bits))
        for M in (1, 2, 4):
            y3 = torch.empty((M, h), dtype=torch.float32, device="cuda")
            backend.matmul_ex(pair, x4[:M].contiguous(), y3, "swiglu")
            torch.cuda.synchronize()
            rd = torch.from_numpy(ref[:M]).cuda()
            want = torch.nn.functional.silu(rd[:, :h]) * rd[:, h:]
            assert ((y3.double() - want).norm() / want.norm()).item() < TIGHT, M


@pytest.mark.parametrize("bits", [4, 8])
def test_decode_modes(backend, oracle, bits):
    """STREAM (default) and EXACT weight operands for one f16 row: both inside the tight bar;
    EXACT returns exact zeros for a tensor of zeros."""
    N, K = 320, 4096
    q, s = _quant(oracle, bits, N, K)
    qw = backend.upload_quantized(q, s, bits)
    qz = backend.upload_quantized(np.zeros((N, K), np.int8), s, bits)
    x = _x(1, K, "f16")
    ref = oracle.matmul_f64(q, s, x.float().cpu().numpy())
    scale = float(np.abs(ref).mean())
    try:
        errs = {}
        for mode in ("stream", "exact"):
            backend.set_decode_mode(mode)
            errs[mode] = oracle.rel_l2(_run(backend, qw, x).cpu().numpy(), ref)
            assert errs[mode] < TIGHT, (mode, errs)
            z = _run(backend, qz, x).cpu().numpy()
            if mode == "exact":
                assert not z.any()
            else:
                assert np.abs(z).max() < 1e-4 * scale       # the bias cancels to rounding, not to the bit
        assert errs["exact"] < 1e-6
    finally:
        backend.set_decode_mode("stream")
    with pytest.raises(CybqError):
        backend.set_decode_mode("loose")


def test_decode_lds_kernel_largest_request(backend, oracle):
    """fp32 activations, 10..16 rows, K long enough for 16 waves: the slab of x is one tile per
    wave whatever the budget says (up to 146 KB of LDS); and exact-mode fp32 prefill walks it."""
    K = 14336
    for N in (64, 4096):
        q, s = _quant(oracle, 4, N, K)
        qw = backend.upload_quantized(q, s, 4)
        for M in (12, 16):
            x = _x(M, K, "f32")
            y = _run(backend, qw, x).cpu().numpy()
            assert oracle.rel_l2(y, oracle.matmul_f64(q, s, x.cpu().numpy())) < TIGHT, (N, M)
    backend.set_prefill_mode("exact")
    try:
        x = _x(40, K, "f32")
        y = _run(backend, qw, x).cpu().numpy()
        assert oracle.rel_l2(y, oracle.matmul_f64(q, s, x.cpu().numpy())) < TIGHT
    finally:
        backend.set_prefill_mode("fast")


def test_known_answers_from_the_committed_fixture(backend):
    """tests/golden/matmul_small.json through the C ABI: both interchange layouts, f16 activations."""
    from tests.test_oracle_matmul import _golden_cases
    for name, bits, q, s, x, want in _golden_cases():
        for layout in (formats.PLANAR, formats.BLOCK_AOS):
            qw = backend.upload_quantized(q, s, bits, layout)
            xt = torch.from_numpy(x).cuda().to(torch.float16)
            y = _run(backend, qw, xt).double().cpu().numpy()
            assert np.linalg.norm(y - want) <= TIGHT * np.linalg.norm(want), (name, layout)
            if name == "by_hand_q4":
                assert np.allclose(y, [[16.0, 32.0, 48.0, 64.0]], rtol=1e-6)


def test_decode_special_cases(backend, oracle):
    N, K = 64, 256
    ones = np.full((N, K // 32), 0x3C00, np.uint16)
    # q = 0 -> 0 ; q = 1, d = 1 -> row sums of x
    qw0 = backend.upload_quantized(np.zeros((N, K), np.int8), ones, 4)
    x = _x(4, K, "f16")
    assert not _run(backend, qw0, x).any()
    qw1 = backend.upload_quantized(np.ones((N, K), np.int8), ones, 4)
    y = _run(backend, qw1, x).cpu().numpy()
    want = x.double().sum(dim=1).cpu().numpy()
    assert np.allclose(y, np.repeat(want[:, None], N, axis=1), rtol=1e-5, atol=1e-4)
    # one-hot x picks a dequantised column exactly
    q, s = _quant(oracle, 4, N, K)
    qw = backend.upload_quantized(q, s, 4)
    wd = oracle.dequant(q, s)
    for k in (0, 7, 8, 31, 32, 255):
        e = torch.zeros((1, K), dtype=torch.float16, device="cuda")
        e[0, k] = 1.0
        assert np.array_equal(_run(backend, qw, e).cpu().numpy()[0], wd[:, k])
    # extreme weights: every nibble value in every slot position
    qe = np.resize(np.arange(-8, 8), (N, K)).astype(np.int8)
    qe[1::2] = qe[1::2, ::-1]
    qwe = backend.upload_quantized(qe, s, 4)
    xe = _x(2, K, "f16")
    assert oracle.rel_l2(_run(backend, qwe, xe).cpu().numpy(),
                         oracle.matmul_f64(qe, s, xe.float().cpu().numpy())) < TIGHT


@pytest.mark.parametrize("ydt", ["f16", "bf16"])
def test_output_dtypes_round_once(backend, oracle, ydt):
    N, K = 128, 512
    q, s = _quant(oracle, 4, N, K)
    qw = backend.upload_quantized(q, s, 4)
    for M in (2, 40):
        x = _x(M, K, "bf16" if M > 16 else "f16")
        y32 = _run(backend, qw, x)
        y16 = _run(backend, qw, x, ydt)
        assert torch.equal(y16, y32.to(TDT[ydt]))


def test_config1_q8_fp32_activations(backend, oracle):
    q, s = _quant(oracle, 8, 2048, 2048, cfg=1)
    qw = backend.upload_quantized(q, s, 8, formats.BLOCK_AOS)
    x = _x(1, 2048, "f32", cfg=1)
    y = _run(backend, qw, x).cpu().numpy()
    assert oracle.rel_l2(y, oracle.matmul_f64(q, s, x.cpu().numpy())) < TIGHT


@pytest.mark.parametrize("shape", [(4096, 4096), (4096, 1024), (4096, 14336), (14336, 4096)])
def test_config2_and_3_full_size(backend, oracle, shape):
    K, N = shape
    q, s = _quant(oracle, 4, N, K, cfg=2)
    qw = backend.upload_quantized(q, s, 4)
    assert qw.algorithmic_bytes == formats.weight_bytes(4, N, K)
    for M in (1, 4, 8, 16):
        x = _x(M, K, "f16", cfg=3, outliers=0.001)
        y = _run(backend, qw, x).cpu().numpy()
        ref = oracle.matmul_f64(q, s, x[: min(M, 2)].float().cpu().numpy())
        assert oracle.rel_l2(y[: min(M, 2)], ref) < TIGHT
        # remaining rows: float64 library matmul on the dequantised weights
        full = x.double().cpu().numpy() @ oracle.dequant(q, s).astype(np.float64).T
        assert oracle.rel_l2(y, full) < TIGHT


# ------------------------------------------------------------ prefill (M > 16)

@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("xdt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("M", [17, 64, 300])
def test_prefill_matches_oracle(backend, oracle, prefill_mode, bits, xdt, M):
    N, K = 240, 512
    q, s = _quant(oracle, bits, N, K)
    qw = backend.upload_quantized(q, s, bits)
    x = _x(M, K, xdt)
    y = _run(backend, qw, x).cpu().numpy()
    assert not np.isnan(y).any()
    err = oracle.rel_l2(y, oracle.matmul_f64(q, s, x.float().cpu().numpy()))
    # fp32 activations: exact through the decode kernel's hi/lo split up to 32 rows and in EXACT mode;
    # FAST prefill rounds them to f16 in the staging pass like any other
    exact_path = M <= (16 if xdt == "f32" else 32) or prefill_mode == "exact"
    assert err < (TIGHT if (xdt == "f32" and exact_path) else _bar(prefill_mode)), err
    if prefill_mode == "fast" and M > (16 if xdt == "f32" else 64):
        # the rounded-weight kernel really ran (up to 32 rows of 16-bit activations take the exact decode
        # kernel, and up to 64 on a weight as small as this one)
        assert err > 1e-6


@pytest.mark.parametrize("shape", [(17, 32), (112, 160), (113, 96), (130, 2080)])
def test_prefill_ragged_shapes(backend, oracle, prefill_mode, shape):
    N, K = shape
    q, s = _quant(oracle, 4, N, K)
    qw = backend.upload_quantized(q, s, 4)
    for M in (17, 257):
        x = _x(M, K, "bf16")
        y = _run(backend, qw, x).cpu().numpy()
        assert not np.isnan(y).any()
        assert oracle.rel_l2(y, oracle.matmul_f64(q, s, x.float().cpu().numpy())) < _bar(prefill_mode)


@pytest.mark.parametrize("xdt", ["bf16", "f32"])
def test_prefill_fast_mode_activation_range(backend, oracle, xdt):
    # FAST turns bf16 / fp32 activations into f16 operands behind a power-of-two scale per row:
    # rows of any magnitude keep the mode's accuracy, outliers far beyond f16's range survive
    N, K = 128, 1024
    q, s = _quant(oracle, 4, N, K)
    qw = backend.upload_quantized(q, s, 4)
    x = _x(40, K, xdt)
    x[0, 5] = 3.0e5
    x[1, 77] = -9.0e5
    x[2] *= 1e-3
    x[3] *= 300.0
    x[4] *= 1e-4
    x[5] *= 1e-5
    x[6] *= 1e-6
    x[7] *= 1e-12
    x[8] *= 1e12
    x[9] = 0.0
    x[10, 1:] = 0.0
    x[11] *= 1e-36                 # largest magnitude below 2^-113: the row's power of two stops at 2^126
    if xdt == "f32":               # a row of fp32 subnormals (made on the host: bit patterns, not device arithmetic)
        x[12] = torch.from_numpy(synth.activations(21, 40, K)[12] * np.float32(1e-40)).cuda()
    backend.set_prefill_mode("fast")
    y = _run(backend, qw, x).cpu().numpy()
    assert np.isfinite(y).all()
    assert not y[9].any()
    ref = oracle.matmul_f64(q, s, x.float().cpu().numpy())
    for rows in ([0], [1], [2], [3], [4], [5], [6], [7], [8], [10], [11], list(range(13, 40))):
        assert oracle.rel_l2(y[rows], ref[rows]) < FAST, rows
    # (the subnormal row: its operands keep what f16 holds below 2^126 times the row, and the result is itself
    # an fp32 subnormal - finite, and as close as those two allow; with bf16 it is an ordinary row)
    assert oracle.rel_l2(y[[12]], ref[[12]]) < (2e-2 if xdt == "f32" else FAST)
    # a folded norm sees the same rows (gamma of mixed magnitudes)
    gamma = torch.from_numpy(np.abs(synth.activations(22, 1, K))[0] * 10.0 + 1e-3).cuda()
    yn = torch.empty((40, N), dtype=torch.float32, device="cuda")
    backend.matmul_norm(qw, x, gamma, 1e-30, yn)           # 40 rows: the prefill kernel
    torch.cuda.synchronize()
    xf = x[:9].double().cpu().numpy()
    rstd = 1.0 / np.sqrt((xf ** 2).mean(axis=1, keepdims=True) + 1e-30)
    refn = oracle.matmul_f64(q, s, (xf * gamma.double().cpu().numpy()).astype(np.float32)) * rstd
    for r in range(9):
        assert oracle.rel_l2(yn[r:r + 1].cpu().numpy(), refn[r:r + 1]) < 2 * FAST, r


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("xdt", ["f16", "bf16", "f32"])
def test_scales_beyond_f16_products(backend, oracle, bits, xdt):
    """scale * q would leave f16's range: such tensors take the decode kernels (scale in fp32) on both
    sides of the prefill boundary - whether the handle was built from host buffers (scanned on the host)
    or from device buffers (scanned by the repack kernel)."""
    N, K = 64, 256
    q, s = _quant(oracle, bits, N, K)
    s = s.copy()
    s[::3, ::2] = np.float16(30000.0).view(np.uint16)
    qd = torch.from_numpy(formats.pack_planar(q, bits)).cuda()
    sd = torch.from_numpy(s.view(np.int16)).cuda()
    handles = [backend.upload_quantized(q, s, bits, formats.BLOCK_AOS), backend.weight_from_device(bits, N, K, qd, sd)]
    for qw in handles:
        for M in (4, 32, 33, 100):
            x = _x(M, K, xdt)
            y = _run(backend, qw, x).cpu().numpy()
            assert np.isfinite(y).all(), M
            assert oracle.rel_l2(y, oracle.matmul_f64(q, s, x.float().cpu().numpy())) < TIGHT, M
    # pairs built from a wide tensor stay wide
    if bits == 4:
        pair = backend.fuse_pairs(handles[1], handles[1])
        x = _x(40, K, "f16")
        y = torch.empty((40, N), dtype=torch.float32, device="cuda")
        backend.matmul_ex(pair, x, y, "swiglu")
        torch.cuda.synchronize()
        assert torch.isfinite(y).all()
        pair.free()
    for qw in handles:
        qw.free()


def test_prefill_rows_agree_with_decode_rows(backend, oracle, prefill_mode):
    N, K = 448, 1024
    q, s = _quant(oracle, 4, N, K)
    qw = backend.upload_quantized(q, s, 4)
    x = _x(64, K, "bf16")
    yp = _run(backend, qw, x)
    yd = _run(backend, qw, x[:16].contiguous())
    num = (yp[:16] - yd).double().norm() / yd.double().norm()
    assert num.item() < _bar(prefill_mode)
    assert torch.equal(_run(backend, qw, x), yp)            # deterministic


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("shape", [(200, 4352), (37, 8192 + 96), (500, 2048)])
def test_prefill_few_tiles_split_k(backend, oracle, prefill_mode, bits, shape):
    # fewer output tiles than CUs and a long K: the K range is split over workgroups
    # (K tiles not divisible by the split, ragged N and M) and the partial sums are
    # added by a second kernel, which also does the output conversion
    N, K = shape
    q, s = _quant(oracle, bits, N, K)
    qw = backend.upload_quantized(q, s, bits)
    for M in (17, 130, 300):
        x = _x(M, K, "bf16")
        y = _run(backend, qw, x)
        assert not torch.isnan(y).any()
        err = oracle.rel_l2(y.cpu().numpy(), oracle.matmul_f64(q, s, x.float().cpu().numpy()))
        assert err < _bar(prefill_mode), (M, err)
        assert torch.equal(_run(backend, qw, x), y)                       # fixed summation order
        for ydt in ("f16", "bf16"):
            assert torch.equal(_run(backend, qw, x, ydt), y.to(TDT[ydt]))   # rounded once


# rows that are no multiple of four elements: the slab-adding pass steps back at the end of a row (its smallest row, one thread, several
# workgroups); outputs at any element, in place, and with a factor per row
@pytest.mark.parametrize("N", [3, 5, 1001, 4090])
@pytest.mark.parametrize("ydt", ["f32", "f16", "bf16"])
def test_prefill_split_k_on_ragged_rows(backend, oracle, N, ydt):
    M, K, dt = 257, 8320, TDT[ydt]
    q, s = _quant(oracle, 4, N, K, cfg=53)
    qw = backend.upload_quantized(q, s, 4)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    x = _x(M, K, "bf16", cfg=54)
    gamma = torch.linspace(0.5, 1.5, K, device="cuda")
    ref = x.double() @ wd.T
    rstd = 1.0 / torch.sqrt((x.double() ** 2).mean(dim=1, keepdim=True) + 1e-5)
    normed = ((x.double() * gamma.double()) @ wd.T) * rstd
    bar = FAST + {"f32": 0.0, "f16": 5e-4, "bf16": 4e-3}[ydt]          # (one rounding of the result)
    for off in (0, 1):                                                  # y and the residual at an odd element of their buffers
        room = torch.full((M * N + 9,), 7.0, dtype=dt, device="cuda")
        y = room[off:off + M * N].view(M, N)
        backend.matmul(qw, x, y)
        assert ((y.double() - ref).norm() / ref.norm()).item() < bar
        r = y.clone()
        backend.matmul_ex(qw, x, y, "add", y)                           # in place: r + x W^T
        want = r.double() + ref
        assert ((y.double() - want).norm() / want.norm()).item() < bar
        if ydt == "f32":
            assert torch.equal(y, r + r)
        backend.matmul_norm(qw, x, gamma, 1e-5, y)
        assert ((y.double() - normed).norm() / normed.norm()).item() < bar + 2e-4      # (x * gamma rounded to f16)
        assert (room[:off] == 7.0).all() and (room[off + M * N:] == 7.0).all()
    qw.free()


def test_prefill_more_rows_than_the_stage_holds(backend, oracle, prefill_mode):
    # 4200 x 16384 activations are 131 MiB: they pass through the 128 MiB staging area
    # in two row chunks
    N, K, M = 48, 16384, 4200
    q, s = _quant(oracle, 4, N, K)
    qw = backend.upload_quantized(q, s, 4)
    x = _x(M, K, "bf16")
    y = _run(backend, qw, x)
    assert not torch.isnan(y).any()
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    full = x.double() @ wd.T
    for lo, hi in ((0, 1000), (3900, 4096), (4096, M)):                     # rows of both chunks
        err = ((y[lo:hi].double() - full[lo:hi]).norm() / full[lo:hi].norm()).item()
        assert err < _bar(prefill_mode), (lo, err)
    rows = [0, 4095, 4096, M - 1]
    ref = oracle.matmul_f64(q, s, x[rows].float().cpu().numpy())
    assert oracle.rel_l2(y[rows].cpu().numpy(), ref) < _bar(prefill_mode)


@pytest.mark.parametrize("M", [128, 512, 2048])
@pytest.mark.parametrize("shape", [(4096, 14336), (14336, 4096)])
def test_config4_full_size(backend, oracle, prefill_mode, M, shape):
    K, N = shape
    q, s = _quant(oracle, 4, N, K, cfg=4)
    qw = backend.upload_quantized(q, s, 4)
    x = _x(M, K, "bf16", cfg=4)
    y = _run(backend, qw, x)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    full = (x.double() @ wd.T)
    err = ((y.double() - full).norm() / full.norm()).item()
    assert err < _bar(prefill_mode), err
    # the oracle itself on a few rows
    rows = [0, M // 2, M - 1]
    ref = oracle.matmul_f64(q, s, x[rows].float().cpu().numpy())
    assert oracle.rel_l2(y[rows].cpu().numpy(), ref) < _bar(prefill_mode)
    # linearity in x: f(2x) == 2 f(x) exactly (powers of two commute with every rounding)
    if prefill_mode == "exact":
        y2 = _run(backend, qw, (x * 2).contiguous())
        assert torch.equal(y2, y * 2)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("xdt", ["f16", "bf16"])
def test_prefill_512_row_workgroups(backend, oracle, bits, xdt):
    """FAST mode, N a multiple of 112 and enough rows for 512-row workgroups to fill the chip: a wave
    multiplies four row blocks per weight operand.  Row counts that are whole tiles, leave a last
    tile more than half full, or fall back to 256-row tiles; residual add and folded RMSNorm ride along."""
    N, K = 14336, 384
    q, s = _quant(oracle, bits, N, K, cfg=41)
    qw = backend.upload_quantized(q, s, bits)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    for M in (1024, 1300, 1100):
        x = _x(M, K, xdt, cfg=42)
        y = _run(backend, qw, x)
        ref = x.double() @ wd.T
        assert ((y.double() - ref).norm() / ref.norm()).item() < FAST, M
        assert torch.equal(_run(backend, qw, x), y)                 # reproducible
        # a row's bits depend neither on its place in a workgroup's tile nor on the tile shape
        # (600 rows run as 256-row tiles)
        assert torch.equal(_run(backend, qw, x[M - 600:].contiguous()), y[M - 600:]), M
    M = 1024
    x = _x(M, K, xdt, cfg=42)
    r = torch.from_numpy(synth.activations(43, M, N)).cuda()
    y2 = torch.empty((M, N), dtype=torch.float32, device="cuda")
    backend.matmul_ex(qw, x, y2, "add", r)
    torch.cuda.synchronize()
    assert torch.equal(y2, _run(backend, qw, x) + r)
    gamma = (1.0 + 0.1 * torch.from_numpy(synth.activations(44, 1, K))[0]).cuda()
    y3 = torch.empty((M, N), dtype=torch.float32, device="cuda")
    backend.matmul_norm(qw, x, gamma, 1e-5, y3)
    torch.cuda.synchronize()
    xd = x.double()
    xn = xd * torch.rsqrt((xd * xd).mean(dim=1, keepdim=True) + 1e-5) * gamma.double()
    ref = xn @ wd.T
    assert ((y3.double() - ref).norm() / ref.norm()).item() < 2 * FAST


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("shape", [(14336, 384, 512), (4096, 384, 2048), (6144, 160, 1100), (14336, 384, 100), (28672, 160, 128),
                                   (14344, 160, 520), (14342, 96, 515),
                                   (4096, 416, 512), (6144, 160, 500), (8000, 96, 512), (4096, 160, 200), (6150, 96, 250),
                                   (8000, 96, 230), (8704, 96, 192), (3840, 96, 320), (4096, 160, 64), (14336, 288, 50)])
def test_prefill_role_split_kernel(backend, oracle, bits, shape):
    """FAST mode with enough 256-row tiles to fill the chip: some waves of a workgroup only multiply,
    the others only fetch and dequantise weights.  Seven and eight column blocks per tile, a ragged
    last row tile, every activation and output type, residual add and folded RMSNorm.  The last two
    shapes: up to 128 rows on a wide output run 128 x 64 tiles without a K split (role-split for one
    round of tiles, the plain kernel for more); then N that ends inside a column block, with rows of y
    that are 16-byte aligned and rows that are not (element-wise stores).  From (4096, 416, 512) on:
    narrow outputs with a short K in one round of 128-row or 64-row tiles that are 4, 6 and 8 column
    blocks wide (K of 3.25 and 2.25 tiles: a remainder behind the whole rounds of the K loops), then
    two decode passes over 64 rows of a small weight and the 64-row tiles of a wide output."""
    N, K, M = shape
    q, s = _quant(oracle, bits, N, K, cfg=45)
    qw = backend.upload_quantized(q, s, bits)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    r = torch.from_numpy(synth.activations(47, M, N)).cuda()
    for xdt, ydt in (("bf16", "f32"), ("f16", "bf16"), ("f32", "f16")):
        x = _x(M, K, xdt, cfg=46)
        ref = x.double() @ wd.T
        y = _run(backend, qw, x, ydt)
        bar = FAST if ydt == "f32" else 4e-3            # (a 16-bit output rounds every element once more)
        assert ((y.double() - ref).norm() / ref.norm()).item() < bar, (xdt, ydt)
        assert torch.equal(_run(backend, qw, x, ydt), y)             # reproducible
        y2 = torch.empty((M, N), dtype=TDT[ydt], device="cuda")
        backend.matmul_ex(qw, x, y2, "add", r.to(TDT[ydt]))
        torch.cuda.synchronize()
        want = ref + r.to(TDT[ydt]).double()
        assert ((y2.double() - want).norm() / want.norm()).item() < bar, (xdt, ydt)
    x = _x(M, K, "bf16", cfg=46)
    gamma = (1.0 + 0.1 * torch.from_numpy(synth.activations(48, 1, K))[0]).cuda()
    y3 = torch.empty((M, N), dtype=torch.float32, device="cuda")
    backend.matmul_norm(qw, x, gamma, 1e-5, y3)
    torch.cuda.synchronize()
    xd = x.double()
    ref = (xd * torch.rsqrt((xd * xd).mean(dim=1, keepdim=True) + 1e-5) * gamma.double()) @ wd.T
    assert ((y3.double() - ref).norm() / ref.norm()).item() < 2 * FAST


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("shape", [(14336, 2048, 64), (8200, 4096 + 128, 33), (8198, 4096 + 256, 47), (14336, 4096, 48),
                                   (28672, 2048, 40), (8192, 8192, 64),
                                   (4096, 4096, 128), (6144 - 16, 4096 + 128, 100), (1024, 4096, 512), (2048, 4096, 300),
                                   (4102, 8192, 70), (8192, 2048, 65),
                                   (1024, 4096 + 128, 60), (4096, 4096, 64), (1030, 2048, 130)])
def test_prefill_few_rows_waves_split_k(backend, oracle, bits, shape):
    """FAST mode, K of 16 .. 64 tiles, one round of workgroups that is at least a quarter full: the kernel whose
    four waves split K and share nothing until the end (no LDS on the way, one partial-sum exchange).  33 .. 64
    rows on outputs from 8192 columns (more than a round of workgroups on the widest); from (4096, 4096, 128)
    on, narrow outputs with up to 512 rows: one to eight workgroups of 64 rows per column group, one, two or
    four column blocks wide (the last three shapes: one), a ragged last row part.  K tile counts that do not
    divide by four (waves with unequal shares), N that ends inside a column block with rows of y aligned and
    not, every activation and output type, residual add, folded RMSNorm; the other kernels (the same call with
    this kernel switched off: the tiled ones, or two decode passes on a small weight at up to 64 rows) agree
    within the mode's tolerance; a row's bits do not depend on the rows it travels with; reproducible."""
    N, K, M = shape
    q, s = _quant(oracle, bits, N, K, cfg=61)
    qw = backend.upload_quantized(q, s, bits)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    r = torch.from_numpy(synth.activations(63, M, N)).cuda()
    try:
        for xdt, ydt in (("bf16", "f32"), ("f16", "bf16"), ("f32", "f16"), ("f16", "f32")):
            x = _x(M, K, xdt, cfg=62)
            ref = x.double() @ wd.T
            y = _run(backend, qw, x, ydt)
            bar = FAST if ydt == "f32" else 4e-3            # (a 16-bit output rounds every element once more)
            assert ((y.double() - ref).norm() / ref.norm()).item() < bar, (xdt, ydt)
            assert torch.equal(_run(backend, qw, x, ydt), y)             # reproducible
            backend.set_gemm_tuning(2)                                     # the tiled kernels on the same call
            y_tiled = _run(backend, qw, x, ydt)
            backend.set_gemm_tuning(0)
            assert ((y.double() - y_tiled.double()).norm() / ref.norm()).item() < 2 * bar, (xdt, ydt)
            if ydt == "f32":
                assert not torch.equal(y, y_tiled)                         # (another order of summation: it did run)
            y2 = torch.empty((M, N), dtype=TDT[ydt], device="cuda")
            backend.matmul_ex(qw, x, y2, "add", r.to(TDT[ydt]))
            torch.cuda.synchronize()
            want = ref + r.to(TDT[ydt]).double()
            assert ((y2.double() - want).norm() / want.norm()).item() < bar, (xdt, ydt)
        parts = (M + 63) // 64                      # fewer rows, the same number of 64-row parts: the same kernel shape
        fewer = 64 * (parts - 1) + 37
        x = _x(64 * parts, K, "f16", cfg=62)
        y_all = _run(backend, qw, x)
        y_fewer = _run(backend, qw, x[:fewer].contiguous())
        assert torch.equal(y_all[:fewer], y_fewer)
        x = _x(M, K, "bf16", cfg=62)
        gamma = (1.0 + 0.1 * torch.from_numpy(synth.activations(64, 1, K))[0]).cuda()
        y3 = torch.empty((M, N), dtype=torch.float32, device="cuda")
        backend.matmul_norm(qw, x, gamma, 1e-5, y3)
        torch.cuda.synchronize()
        xd = x.double()
        ref = (xd * torch.rsqrt((xd * xd).mean(dim=1, keepdim=True) + 1e-5) * gamma.double()) @ wd.T
        assert ((y3.double() - ref).norm() / ref.norm()).item() < 2 * FAST
    finally:
        backend.set_gemm_tuning(0)
    qw.free()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("shape", [(4096, 14336, 45), (992, 65 * 128, 64), (16, 16384 + 32, 128), (1030, 9216 + 64, 100),
                                   (2048, 8192 + 32, 33), (4096, 65 * 128 - 32, 17), (8224, 65 * 128, 40), (10000, 8192 + 128, 60),
                                   (500, 96 * 128, 48), (500, 96 * 128 + 32, 33), (2050, 112 * 128, 32), (3850, 65 * 128, 31), (3850, 96 * 128, 19)])
def test_prefill_few_rows_long_k_shares(backend, oracle, bits, shape):
    """FAST mode, up to 128 rows, K of more than 64 tiles: each wave of the few-row kernel, or each workgroup of eight
    strips, walks one share of K as the tiled kernels' K split does, so the results are the tiled kernels' bit for bit.  Eight,
    seven, four, three shares, both sides of 96 tiles, of 32 and 48 rows and of one column block per workgroup, the fewest K tiles, a last share shorter than the others, one strip, N that ends inside a column block and is no multiple of four,
    y off its vector alignment, every epilogue; 17 rows are fp32 (16-bit rows that few keep the decode kernels)."""
    N, K, M = shape
    q, s = _quant(oracle, bits, N, K, cfg=65)
    qw = backend.upload_quantized(q, s, bits)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    r = torch.from_numpy(synth.activations(66, M, N)).cuda()
    try:
        for xdt, ydt in (("bf16", "f32"), ("f16", "bf16"), ("f32", "f16")) if M > 32 else (("f32", "f32"), ("f32", "bf16")):
            x = _x(M, K, xdt, cfg=67)
            ref = x.double() @ wd.T
            bar = FAST if ydt == "f32" else 4e-3            # (a 16-bit output rounds every element once more)
            y = _run(backend, qw, x, ydt)
            assert ((y.double() - ref).norm() / ref.norm()).item() < bar, (xdt, ydt)
            assert torch.equal(_run(backend, qw, x, ydt), y)             # reproducible
            backend.set_gemm_tuning(2)
            y_tiled = _run(backend, qw, x, ydt)
            backend.set_gemm_tuning(0)
            assert torch.equal(y, y_tiled), (xdt, ydt)
            want = ref + r.to(TDT[ydt]).double()
            for off in (0, 1):
                y2 = torch.empty(M * N + 1, dtype=TDT[ydt], device="cuda")[off:off + M * N].view(M, N)
                r2 = torch.empty_like(y2).copy_(r)
                backend.matmul_ex(qw, x, y2, "add", r2)
                torch.cuda.synchronize()
                assert ((y2.double() - want).norm() / want.norm()).item() < bar, (xdt, ydt, off)
        if M > 32:
            x = _x(M, K, "f16", cfg=67)
            gamma = (1.0 + 0.1 * torch.from_numpy(synth.activations(68, 1, K))[0]).cuda()
            y3 = torch.empty((M, N), dtype=torch.float32, device="cuda")
            backend.matmul_norm(qw, x, gamma, 1e-5, y3, "add", r)
            torch.cuda.synchronize()
            xd = x.double()
            ref = (xd * torch.rsqrt((xd * xd).mean(dim=1, keepdim=True) + 1e-5) * gamma.double()) @ wd.T + r.double()
            assert ((y3.double() - ref).norm() / ref.norm()).item() < 2 * FAST
            if N % 16 == 0:
                pair = backend.fuse_pairs(qw, qw)
                y4 = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
                backend.matmul_ex(pair, x, y4, "swiglu")
                torch.cuda.synchronize()
                z = xd @ wd.T
                ref = torch.nn.functional.silu(z) * z
                assert ((y4.double() - ref).norm() / ref.norm()).item() < 4e-3
                pair.free()
    finally:
        backend.set_gemm_tuning(0)
    qw.free()


@pytest.mark.parametrize("bits,N,K,M", [(4, 16400, 17 * 128, 49), (4, 16384 + 64, 18 * 128 - 32, 64), (4, 33000, 19 * 128 - 96, 63),
                                        (4, 49172, 16 * 128, 50), (8, 16400, 20 * 128, 17), (8, 24002, 21 * 128 + 64, 48), (8, 16448, 62 * 128, 64), (4, 17000, 63 * 128 + 32, 33)])
def test_prefill_few_rows_two_column_groups_per_workgroup(backend, oracle, bits, N, K, M):
    """More than a round of workgroups: two column groups to a workgroup that walk the K tiles together.  A last group that is not full or
    has no partner, K tiles that leave waves without one in the last step, N that is no multiple of 16 or 4: bit for bit the kernel with a
    group to a workgroup; against float64; the epilogues."""
    q, s = _quant(oracle, bits, N, K, cfg=137)
    qw = backend.upload_quantized(q, s, bits)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    r = torch.from_numpy(synth.activations(138, M, N)).cuda()
    try:
        for xdt in ("bf16", "f16") if M > 32 else ("f32",):
            x = _x(M, K, xdt, cfg=139)
            y = _run(backend, qw, x)
            ref = x.double() @ wd.T
            assert ((y.double() - ref).norm() / ref.norm()).item() < FAST
            backend.set_gemm_tuning(1)
            assert torch.equal(_run(backend, qw, x), y), xdt
            backend.set_gemm_tuning(0)
            y2 = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
            backend.matmul_ex(qw, x, y2, "add", r.bfloat16())
            want = ref + r.bfloat16().double()
            assert ((y2.double() - want).norm() / want.norm()).item() < 4e-3
        if N % 16 == 0:
            h = torch.arange(N // 2 // 16 * 16, device="cuda")
            half = backend.upload_quantized(q[: N // 2 // 16 * 16], s[: N // 2 // 16 * 16], bits)
            pair = backend.fuse_pairs(half, half)
            gamma = (1.0 + 0.1 * torch.from_numpy(synth.activations(140, 1, K))[0]).cuda()
            y3 = torch.empty((M, len(h)), dtype=torch.float32, device="cuda")
            y4 = torch.empty_like(y3)
            backend.matmul_norm(pair, x, gamma, 1e-5, y3, "swiglu")
            backend.set_gemm_tuning(1)
            backend.matmul_norm(pair, x, gamma, 1e-5, y4, "swiglu")
            torch.cuda.synchronize()
            assert torch.equal(y3, y4)
            pair.free()
            half.free()
    finally:
        backend.set_gemm_tuning(0)
    qw.free()


# (FAST needs K outside 2048 .. 8192 or more than 512 rows to get past the few-row kernel)
COLS = [("exact", 1030, 33 * 128 - 32, 67), ("exact", 1024, 128, 97), ("exact", 4096, 4096, 128), ("exact", 14336, 288, 193),
        ("exact", 520, 12 * 128 + 64, 260), ("exact", 9000, 640, 80), ("exact", 14400, 2048, 33),
        ("fast", 1030, 9 * 128 - 32, 100), ("fast", 520, 128, 129), ("fast", 24640, 70 * 128 + 64, 48), ("fast", 30000, 1056, 64),
        ("fast", 2064, 12288, 200), ("fast", 16400, 8320, 96), ("fast", 1040, 1920, 250)]


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("mode,N,K,M", COLS)
def test_prefill_waves_side_by_side(backend, oracle, bits, mode, N, K, M):
    """The kernel whose waves stand side by side and share out every K tile: one K tile, fewer than the copies reach ahead, a last
    K tile that is a quarter, half, three quarters full, K shared out over workgroups, each of its row and column counts, a last row
    and column tile that are not full, N that is no multiple of 16 or 4, y off its vector alignment, every epilogue.  Against
    float64; against the tiled kernels (another order of summation: it did run); reproducible."""
    q, s = _quant(oracle, bits, N, K, cfg=131)
    qw = backend.upload_quantized(q, s, bits)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    r = torch.from_numpy(synth.activations(133, M, N)).cuda()
    bar = TIGHT if mode == "exact" else FAST
    backend.set_prefill_mode(mode)
    try:
        for xdt in ("bf16", "f16"):
            x = _x(M, K, xdt, cfg=132)
            xd = x.double()
            z = xd @ wd.T
            y = _run(backend, qw, x)
            assert ((y.double() - z).norm() / z.norm()).item() < bar, xdt
            assert torch.equal(_run(backend, qw, x), y)
            backend.set_gemm_tuning(3)
            y_tiled = _run(backend, qw, x)
            backend.set_gemm_tuning(0)
            assert ((y - y_tiled).double().norm() / z.norm()).item() < (2e-6 if mode == "exact" else 2 * bar), xdt
            if M > 64 or mode == "fast":                   # (up to 64 rows a small weight is two decode passes there)
                assert K <= 256 or not torch.equal(y, y_tiled), xdt
            for ydt, off in (("f32", 1), ("bf16", 0), ("f16", 3)):
                y2 = torch.empty(M * N + 4, dtype=TDT[ydt], device="cuda")[off:off + M * N].view(M, N)
                r2 = torch.empty_like(y2).copy_(r)
                backend.matmul_ex(qw, x, y2, "add", r2)
                want = z + r2.double()
                assert ((y2.double() - want).norm() / want.norm()).item() < (bar if ydt == "f32" else 4e-3), (xdt, ydt)
            gamma = (1.0 + 0.1 * torch.from_numpy(synth.activations(134, 1, K))[0]).cuda()
            y3 = torch.empty((M, N), dtype=torch.float32, device="cuda")
            backend.matmul_norm(qw, x, gamma, 1e-5, y3)
            ref = (xd * torch.rsqrt((xd * xd).mean(dim=1, keepdim=True) + 1e-5) * gamma.double()) @ wd.T
            assert ((y3.double() - ref).norm() / ref.norm()).item() < (4e-3 if mode == "exact" else 2 * FAST), xdt    # (x * gamma rounded)
            if N % 16 == 0:
                pair = backend.fuse_pairs(qw, qw)
                y4 = torch.empty((M, N), dtype=torch.float32, device="cuda")
                backend.matmul_ex(pair, x, y4, "swiglu")
                ref = torch.nn.functional.silu(z) * z
                assert ((y4.double() - ref).norm() / ref.norm()).item() < 4 * bar, xdt
                pair.free()
    finally:
        backend.set_gemm_tuning(0)
        backend.set_prefill_mode("fast")
    qw.free()


# FAST, f16: shapes past the two decode passes (more than 6144 x 4096 weights or 64 rows) with K outside the few-row kernel's; over 64 K tiles
# eight whole-tile waves on 3, 4, 3, 4, 6 and 8 row blocks.  33 bf16 rows of Q4 at K = 9024: exact operands on a small weight.
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("mode,N,K,M", [("exact", 1030, 128, 97), ("exact", 530, 352, 65), ("exact", 14336, 288, 193), ("exact", 4096, 1056, 130),
                                        ("exact", 96, 4096, 519), ("fast", 520, 96, 129), ("fast", 1030, 9 * 128 - 32, 100), ("fast", 24640, 1056, 47),
                                        ("fast", 1030, 70 * 128 + 64, 33), ("fast", 1030, 192 * 128 + 64, 33), ("fast", 1030, 192 * 128 + 64, 60),
                                        ("fast", 1030, 71 * 128 + 96, 90), ("fast", 1030, 66 * 128 + 32, 128), ("fast", 4090, 65 * 128 + 32, 90),
                                        ("fast", 4090, 65 * 128 + 32, 120)])
def test_prefill_rows_read_in_place(backend, bits, mode, N, K, M):
    """Rows that are operands as they stand are multiplied from where the caller has them: the bits of the same call behind a staging
    launch, over row counts and K that leave a last row block and a last K tile of every fill, whatever lies behind the last row."""
    qw, wd = _random_weight(backend, bits, N, K, 141)
    backend.set_prefill_mode(mode)
    try:
        for xdt in ("f16", "bf16"):
            big = torch.full((M + 40, K), float("nan"), dtype=TDT[xdt], device="cuda")
            x = big[:M].copy_(_x(M, K, xdt, cfg=142))
            y = _run(backend, qw, x)
            backend.set_gemm_tuning(4)
            staged = _run(backend, qw, x)
            backend.set_gemm_tuning(0)
            ref = x.double() @ wd.T
            assert ((y.double() - ref).norm() / ref.norm()).item() < (SUMS if mode == "exact" else FAST), xdt
            assert torch.equal(y, staged), xdt
    finally:
        backend.set_gemm_tuning(0)
        backend.set_prefill_mode("fast")
    qw.free()


def test_prefill_rows_read_in_place_behind_a_chunk(backend):
    """f16 rows of a long K beyond what the scratch holds: a last chunk of 20 rows is eight whole-tile waves on two row blocks."""
    N, K = 2080, 32768
    rows = (((256 - 8) << 20) // 2 - (1 << 20)) // (2 * K) // 256 * 256      # what the first half of the scratch holds behind its last MiB
    M = rows + 20
    qw, wd = _random_weight(backend, 8, N, K, 143)
    g = torch.Generator(device="cuda").manual_seed(144)
    x = torch.empty((M + 8, K), device="cuda").normal_(generator=g).half()
    x[M:] = float("nan")
    try:
        y = _run(backend, qw, x[:M])
        backend.set_gemm_tuning(4)
        assert torch.equal(_run(backend, qw, x[:M]), y)
    finally:
        backend.set_gemm_tuning(0)
    ref = x[rows:M].double() @ wd.T
    assert ((y[rows:].double() - ref).norm() / ref.norm()).item() < FAST
    qw.free()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("xdt", ["bf16", "f16"])
@pytest.mark.parametrize("shift", [-8, 0, 8, 512 * 1024])
def test_prefill_rows_that_y_overlaps_are_staged(backend, bits, xdt, shift):
    """y written over the rows it is made from, at the same place, eight elements off either way or half of them on: 176 workgroups without
    a split of K, eleven row tiles, which would overwrite each other's rows if they were read in place."""
    N = K = M = 1024
    qw, _ = _random_weight(backend, bits, N, K, 145)
    backend.set_prefill_mode("exact")
    try:
        x = _x(M, K, xdt, cfg=146)
        backend.set_gemm_tuning(4)
        apart = _run(backend, qw, x, xdt)
        backend.set_gemm_tuning(0)
        assert torch.equal(_run(backend, qw, x, xdt), apart)
        both = torch.zeros((2 * M * K + 16,), dtype=TDT[xdt], device="cuda")
        xo, yo = both[8:8 + M * K].view(M, K), both[8 + shift:8 + shift + M * N].view(M, N)
        xo.copy_(x)
        backend.matmul(qw, xo, yo)
        torch.cuda.synchronize()
        assert torch.equal(yo, apart)
    finally:
        backend.set_gemm_tuning(0)
        backend.set_prefill_mode("fast")
    qw.free()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("N,K,M", [(1536, 128, 2000), (1530, 352, 1999), (1441, 544, 2000), (5600, 1184, 250), (5590, 96, 193)])
def test_prefill_six_column_blocks_per_workgroup(backend, oracle, bits, N, K, M):
    """Shapes whose tiles of six column blocks fill most of a round (128 rows, the last two 64): two of the blocks are shared out in halves
    among the four waves that stage weights.  One to ten K tiles, a last tile of every fill, a last column tile that is not whole."""
    q, s = _quant(oracle, bits, N, K, cfg=151)
    qw = backend.upload_quantized(q, s, bits)
    w = torch.empty((N, K), dtype=torch.float32, device="cuda")
    backend.dequant(qw, w)
    try:
        backend.set_gemm_tuning(2)                                     # (a short K is gemm_cols.hip's otherwise)
        for xdt in ("bf16", "f16"):
            x = _x(M, K, xdt, cfg=152)
            y = _run(backend, qw, x)
            ref = x.double() @ w.double().t()
            assert ((y.double() - ref).norm() / ref.norm()).item() < FAST, xdt
    finally:
        backend.set_gemm_tuning(0)
    qw.free()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("N,K,M", [(14364, 640, 327), (30164, 1248, 174), (7768, 1120, 1015), (15093, 512, 579)])
def test_prefill_exact_on_wide_outputs_of_a_short_k(backend, oracle, bits, N, K, M):
    """EXACT calls between the tiled kernels and the one whose waves stand side by side, which has most of them: what fp32 sums leave.  Q8 under
    bf16 rows on the tiled ones, which have two of them by the estimates: the rounding of a second operand, 2^-17 of the weight."""
    rng = np.random.default_rng(161)
    q = rng.integers(-8 if bits == 4 else -128, 8 if bits == 4 else 128, size=(N, K), dtype=np.int8)
    s = (rng.random((N, K // 32), dtype=np.float32) * 0.01).astype(np.float16).view(np.uint16)
    qw = backend.upload_quantized(q, s, bits)
    w = torch.empty((N, K), dtype=torch.float32, device="cuda")
    backend.dequant(qw, w)
    backend.set_prefill_mode("exact")
    try:
        for xdt in ("bf16", "f16"):
            x = _x(M, K, xdt, cfg=162)
            ref = x.double() @ w.double().t()
            for tuning in (0, 3):
                backend.set_gemm_tuning(tuning)
                y = _run(backend, qw, x)
                rounded = bits == 8 and xdt == "bf16" and (tuning == 3 or N in (14364, 7768))
                assert ((y.double() - ref).norm() / ref.norm()).item() < (2.0 ** -17 if rounded else SUMS), (xdt, tuning)
    finally:
        backend.set_gemm_tuning(0)
        backend.set_prefill_mode("fast")
    qw.free()


@pytest.mark.parametrize("N,K,M", [(300, 4096, 1537), (272, 4064, 1545), (530, 1056, 2047), (1024, 2080, 2048), (64, 32, 1551), (300, 4096, 1536), (300, 4128, 2048)])
def test_prefill_rows_staged_eight_to_a_workgroup(backend, oracle, N, K, M):
    """bf16 rows at and around the counts that are staged eight to a workgroup: last workgroups of one to eight rows, last pieces of every fill,
    rows of very different magnitudes (each has a power of two of its own)."""
    q, s = _quant(oracle, 4, N, K, cfg=171)
    qw = backend.upload_quantized(q, s, 4)
    w = torch.empty((N, K), dtype=torch.float32, device="cuda")
    backend.dequant(qw, w)
    x = _x(M, K, "f32", cfg=172)
    x *= torch.pow(2.0, (torch.arange(M, device="cuda") % 61 - 30).float())[:, None]
    x = x.to(torch.bfloat16)
    y = _run(backend, qw, x)
    ref = x.double() @ w.double().t()
    err = (y.double() - ref).norm(dim=1) / ref.norm(dim=1)
    # a row by itself: the mode's 2e-4 and, where N outputs are few, their spread; a row with a neighbour's power of two would be off by half and more
    assert err.max().item() < 1e-2 and err.mean().item() < FAST
    qw.free()


@pytest.mark.parametrize("mode,bits,N,K,M", [("exact", 4, 592, 352, 83), ("exact", 8, 592, 352, 83), ("exact", 4, 1024, 4096, 256), ("exact", 8, 96, 4096, 519),
                                             ("fast", 4, 512, 8224, 48), ("fast", 4, 6160, 512, 40)])
def test_prefill_exact_rows_of_any_magnitude(backend, mode, bits, N, K, M):
    """bf16 rows up to the type's largest against scales that bring them back, groups of scale zero and groups past the end of K among
    them: the sums of a group stay in range wherever its contribution to y does, in EXACT mode and where FAST mode takes exact operands
    (33 .. 64 rows of Q4, K over 4096, or short on a wide output)."""
    rng = np.random.default_rng(181)
    q = rng.integers(-(1 << (bits - 1)), 1 << (bits - 1), (N, K)).astype(np.int8)
    s = (rng.random((N, K // 32)) * 0.004 + 0.0005).astype(np.float16)
    s[:, 1::7] = 0
    qw = backend.upload_quantized(q, s.view(np.uint16), bits)
    wd = torch.from_numpy(np.repeat(s.astype(np.float64), 32, axis=1) * q).cuda()
    powers = (0, 30, 33, 34, 35, 36, -30, -34, -36)
    x = synth.activations(182, M, K).astype(np.float64) * (10.0 ** np.array([powers[m % len(powers)] for m in range(M)]))[:, None]
    x[0, 5] = 3.3e38                                           # one element
    x[9, :256] = 2e36 * np.sign(q[0, :256] + 0.5)              # eight groups of one sign against column 0
    x[18] = 0.0
    x = torch.from_numpy(x.astype(np.float32)).cuda().bfloat16()
    backend.set_prefill_mode(mode)
    try:
        y = _run(backend, qw, x).double()
    finally:
        backend.set_prefill_mode("fast")
    ref = x.double() @ wd.T
    assert torch.isfinite(y).all() and not y[18].any()
    norm = ref.norm(dim=1)
    norm[18] = 1.0
    # fp32 sums (1e-7): a row of 1e-36 has products down to 2^-149 of a sum of 2^-120
    assert ((y - ref).norm(dim=1) / norm).max().item() < 1e-6
    qw.free()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("xdt", ["bf16", "f16"])
def test_prefill_exact_operands_over_all_scales(backend, bits, xdt):
    """EXACT mode: subnormal, negative and large scales alike, every output column with scales of one binade of its own (the largest keeps
    scale * q inside f16): integer operands with the scale on the sums, and the tiled kernel's two operands, which add up to scale * q."""
    N, K, M = 37 * 16, 384, 80
    rng = np.random.default_rng(7)
    top = 11 if bits == 4 else 7                            # 2^12 * 8, 2^8 * 128
    e = np.arange(N) % (top + 25) - 24
    s = ((2.0 ** e)[:, None] * (1 + rng.random((N, K // 32))) * rng.choice([-1, 1], (N, K // 32))).astype(np.float16).view(np.uint16)
    q = rng.integers(-(1 << (bits - 1)), 1 << (bits - 1), (N, K)).astype(np.int8)
    qw = backend.upload_quantized(q, s, bits)
    wd = torch.from_numpy(np.repeat(s.view(np.float16).astype(np.float64), 32, axis=1) * q).cuda()
    x = _x(M, K, xdt, cfg=135)
    ref = x.double() @ wd.T
    # two operands: a Q8 weight's second bf16 operand is rounded to eight bits, 2^-17 of the weight; an f16 operand of the smallest
    # scales is a subnormal with up to ten leading zeros, and the matrix pipe aligns its 24 bits by exponent fields: 2^(10 - 24)
    two = 6.2e-5 if xdt == "f16" else 1e-5 if bits == 8 else 2e-6
    backend.set_prefill_mode("exact")
    try:
        for tuning, bar in ((0, SUMS), (3, two)):
            backend.set_gemm_tuning(tuning)
            y = _run(backend, qw, x).double()
            assert ((y - ref).norm(dim=0) / ref.norm(dim=0)).max().item() < bar, tuning
    finally:
        backend.set_gemm_tuning(0)
        backend.set_prefill_mode("fast")
    qw.free()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("N,M,pair", [(28672, 300, True), (28672, 257, True), (32 * 1083, 512, True), (20000, 300, False),
                                      (24998, 700, False), (20016, 512, False)])
def test_prefill_role_split_wide_outputs_and_pairs(backend, oracle, bits, N, M, pair):
    """FAST mode, enough 256-row tiles to fill the chip: the role-split kernel, for SwiGLU pairs as well.  A last tile that
    is not full, N that is no multiple of 16 or 4, ragged rows, residual add and folded norm; every column against float64."""
    K = 288                                             # (a last K tile that is a quarter full)
    half = N // 2 if pair else N
    q, s = _quant(oracle, bits, half, K, cfg=71)
    qw = backend.upload_quantized(q, s, bits)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    x = _x(M, K, "bf16", cfg=72)
    ref = x.double() @ wd.T
    if pair:
        q2, s2 = _quant(oracle, bits, half, K, cfg=73)
        q2w = backend.upload_quantized(q2, s2, bits)
        up = x.double() @ torch.from_numpy(oracle.dequant(q2, s2)).cuda().double().T
        fused = backend.fuse_pairs(qw, q2w)
        for ydt in ("f32", "bf16"):
            y = torch.full((M, half), float("nan"), dtype=TDT[ydt], device="cuda")
            backend.matmul_ex(fused, x, y, "swiglu")
            torch.cuda.synchronize()
            want = torch.nn.functional.silu(ref) * up
            assert ((y.double() - want).norm(dim=0) / want.norm(dim=0)).max().item() < (3e-3 if ydt == "f32" else 6e-3)    # column by column
            assert ((y.double() - want).norm() / want.norm()).item() < (2 * FAST if ydt == "f32" else 4e-3)
        for w in (q2w, fused):
            w.free()
    else:
        y = _run(backend, qw, x)
        assert ((y.double() - ref).norm(dim=0) / ref.norm(dim=0)).max().item() < 3e-3
        assert ((y.double() - ref).norm() / ref.norm()).item() < FAST
        assert torch.equal(_run(backend, qw, x), y)
        r = torch.from_numpy(synth.activations(74, M, N)).cuda()
        gamma = (1.0 + 0.1 * torch.from_numpy(synth.activations(75, 1, K))[0]).cuda()
        y2 = torch.empty_like(y)
        backend.matmul_norm(qw, x, gamma, 1e-5, y2, "add", r)
        torch.cuda.synchronize()
        xd = x.double()
        want = (xd * torch.rsqrt((xd * xd).mean(dim=1, keepdim=True) + 1e-5) * gamma.double()) @ wd.T + r.double()
        assert ((y2.double() - want).norm() / want.norm()).item() < 2 * FAST
    qw.free()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("N,K,M,xdt", [(16656, 2048, 24, "f32"), (16660, 2048 + 32, 48, "bf16"), (17024, 4096, 33, "f16"), (33000, 2048, 40, "bf16")])
def test_prefill_few_rows_two_workgroups_per_cu(backend, oracle, bits, N, K, M, xdt):
    """Up to 48 rows and more column groups than CUs: the few-row kernel with fewer weight tiles in flight, two workgroups
    per CU.  Just past one round, several rounds, N inside a column block, K tiles that no wave count divides; and the
    bits of the rows equal those of a call of 17 rows less (fp32: two rows less)."""
    q, s = _quant(oracle, bits, N, K, cfg=81)
    qw = backend.upload_quantized(q, s, bits)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    x = _x(M, K, xdt, cfg=82)
    y = _run(backend, qw, x)
    ref = x.double() @ wd.T
    assert ((y.double() - ref).norm(dim=0) / ref.norm(dim=0)).max().item() < 4e-3
    assert ((y.double() - ref).norm() / ref.norm()).item() < FAST
    fewer = 33 if M > 33 else M - 2 if xdt == "f32" else M
    assert torch.equal(_run(backend, qw, x[:fewer].contiguous()), y[:fewer])
    qw.free()


@pytest.mark.parametrize("xdt", ["bf16", "f32"])
@pytest.mark.parametrize("K", [512 - 32, 4096 + 32, 8192, 8192 + 32, 16384 + 64, 32768 + 512])
def test_prefill_row_scaling_pass_rows_per_workgroup(backend, oracle, K, xdt):
    """The row-scaling pass gives a workgroup one, two or four rows by K and the number of rows: last rows of a workgroup
    missing, K that ends inside a piece, rows that stay in registers and rows that are read again, rows of very different
    size, with a folded norm; and the same rows in calls of the sizes at which the rule changes."""
    N = 48
    q, s = _quant(oracle, 4, N, K, cfg=83)
    qw = backend.upload_quantized(q, s, 4)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    gamma = (1.0 + 0.1 * torch.from_numpy(synth.activations(84, 1, K))[0]).cuda()
    for M in (33, 47, 49, 127, 130, 513):
        x = (_x(M, K, "f32", cfg=85) * torch.logspace(-6, 6, M, device="cuda")[:, None]).to(TDT[xdt])
        xd = x.double()
        for y, ref in ((_run(backend, qw, x), xd @ wd.T), (torch.empty((M, N), device="cuda"), None)):
            if ref is None:
                backend.matmul_norm(qw, x, gamma, 1e-30, y)
                torch.cuda.synchronize()
                ref = (xd * torch.rsqrt((xd * xd).mean(dim=1, keepdim=True) + 1e-30) * gamma.double()) @ wd.T
            # row by row: 48 sums of K products, weights (and fp32 rows, or x * gamma) rounded to f16 (2^-11 each)
            assert ((y.double() - ref).norm(dim=1) / ref.norm(dim=1)).max().item() < 2e-3, M
    qw.free()


@pytest.mark.parametrize("xdt,M", [("bf16", 384), ("bf16", 385), ("f32", 512), ("f32", 513)])
@pytest.mark.parametrize("K", [8192 + 32, 16384 + 64])
def test_prefill_row_scaling_pass_where_two_rows_become_four(backend, oracle, K, xdt, M):
    N = 48
    q, s = _quant(oracle, 4, N, K, cfg=86)
    qw = backend.upload_quantized(q, s, 4)
    x = (_x(M, K, "f32", cfg=87) * torch.logspace(-6, 6, M, device="cuda")[:, None]).to(TDT[xdt])
    ref = x.double() @ torch.from_numpy(oracle.dequant(q, s)).cuda().double().T
    # (row by row; the bar of the test above)
    assert ((_run(backend, qw, x).double() - ref).norm(dim=1) / ref.norm(dim=1)).max().item() < 2e-3
    qw.free()


@pytest.mark.parametrize("shape", [(14336, 4096, 17), (4096, 4096, 32), (8200, 2048 + 128, 24)])
def test_prefill_fp32_rows_17_to_32_fast_mode(backend, oracle, shape):
    """fp32 activations leave the decode kernels at 17 rows; in FAST mode they are rounded to f16 by the staging
    pass and, where the shape fits, multiplied by the kernel whose waves split K (a 64-row workgroup mostly
    empty).  Against float64, against the tiled kernels, residual add, reproducible."""
    N, K, M = shape
    q, s = _quant(oracle, 4, N, K, cfg=65)
    qw = backend.upload_quantized(q, s, 4)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    x = _x(M, K, "f32", cfg=66)
    ref = x.double() @ wd.T
    try:
        y = _run(backend, qw, x)
        assert ((y.double() - ref).norm() / ref.norm()).item() < FAST
        assert torch.equal(_run(backend, qw, x), y)
        backend.set_gemm_tuning(2)
        y_tiled = _run(backend, qw, x)
        backend.set_gemm_tuning(0)
        assert ((y.double() - y_tiled.double()).norm() / ref.norm()).item() < 2 * FAST
        assert not torch.equal(y, y_tiled)                                 # (another order of summation: it did run)
        r = torch.from_numpy(synth.activations(67, M, N)).cuda()
        y2 = torch.empty((M, N), dtype=torch.float32, device="cuda")
        backend.matmul_ex(qw, x, y2, "add", r)
        torch.cuda.synchronize()
        assert ((y2.double() - (ref + r.double())).norm() / (ref + r.double()).norm()).item() < FAST
    finally:
        backend.set_gemm_tuning(0)
    qw.free()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("shape", [(7168, 4096, 48, "bf16"), (2048, 4096 + 128, 100, "f16"), (14336, 2048, 33, "bf16"),
                                   (1040, 4096, 24, "f32"), (4096, 2048, 64, "bf16")])
def test_prefill_few_rows_swiglu(backend, oracle, bits, shape):
    """The SwiGLU epilogue of the kernel whose waves split K (FAST mode): a workgroup holds gate / up column blocks
    in pairs and the wave that finishes a row block writes silu(gate) * up.  One workgroup per 64 rows, two row
    parts, more than one round of workgroups, fp32 rows below 33, with a folded RMSNorm; against float64 and
    against the tiled kernels on the same call."""
    N, K, M, xdt = shape
    qg, sg = _quant(oracle, bits, N, K, cfg=81)
    qu, su = _quant(oracle, bits, N, K, cfg=82)
    wg, wu = backend.upload_quantized(qg, sg, bits), backend.upload_quantized(qu, su, bits)
    wf = backend.fuse_pairs(wg, wu)
    dg = torch.from_numpy(oracle.dequant(qg, sg)).cuda().double()
    du = torch.from_numpy(oracle.dequant(qu, su)).cuda().double()
    try:
        for ydt in ("f32", "bf16"):
            x = _x(M, K, xdt, cfg=83)
            g, u = x.double() @ dg.T, x.double() @ du.T
            ref = g / (1.0 + torch.exp(-g)) * u
            bar = 2 * FAST if ydt == "f32" else 6e-3
            y = torch.full((M, N), float("nan"), dtype=TDT[ydt], device="cuda")
            backend.matmul_ex(wf, x, y, "swiglu")
            y_again = torch.empty_like(y)
            backend.matmul_ex(wf, x, y_again, "swiglu")
            backend.set_gemm_tuning(2)
            y_tiled = torch.empty_like(y)
            backend.matmul_ex(wf, x, y_tiled, "swiglu")
            backend.set_gemm_tuning(0)
            torch.cuda.synchronize()
            assert not torch.isnan(y.float()).any()
            assert ((y.double() - ref).norm() / ref.norm()).item() < bar, ydt
            assert torch.equal(y, y_again)
            assert ((y.double() - y_tiled.double()).norm() / ref.norm()).item() < 2 * bar, ydt
            if ydt == "f32":
                assert not torch.equal(y, y_tiled)                         # (another kernel: it did run)
        x = _x(M, K, "bf16", cfg=84)
        gamma = (1.0 + 0.1 * torch.from_numpy(synth.activations(85, 1, K))[0]).cuda()
        xd = x.double()
        xn = xd * torch.rsqrt((xd * xd).mean(dim=1, keepdim=True) + 1e-5) * gamma.double()
        g, u = xn @ dg.T, xn @ du.T
        ref = g / (1.0 + torch.exp(-g)) * u
        y = torch.empty((M, N), dtype=torch.float32, device="cuda")
        backend.matmul_norm(wf, x, gamma, 1e-5, y, "swiglu")
        torch.cuda.synchronize()
        assert ((y.double() - ref).norm() / ref.norm()).item() < 4 * FAST
    finally:
        backend.set_gemm_tuning(0)
    for t in (wf, wg, wu):
        t.free()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("shape", [(14336, 4096, 32), (2064, 2048 + 128, 17), (4096, 8192, 25)])
def test_folded_norm_17_to_32_rows_fast_mode(backend, oracle, bits, shape):
    """17 .. 32 rows of 16-bit activations with a folded RMSNorm leave the one-pass decode kernel; in FAST mode,
    where the shape fits, the staging pass folds gamma in and the kernel whose waves split K multiplies (two row
    blocks per workgroup).  Against float64, against the two decode passes that take the call otherwise, with a
    residual add, 16-bit outputs; reproducible; a row's bits do not depend on the rows it travels with."""
    N, K, M = shape
    q, s = _quant(oracle, bits, N, K, cfg=71)
    qw = backend.upload_quantized(q, s, bits)
    wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
    r = torch.from_numpy(synth.activations(73, M, N)).cuda()
    try:
        for xdt, gdt, ydt in (("bf16", torch.float16, "f32"), ("f16", torch.float32, "bf16"), ("bf16", torch.bfloat16, "f16")):
            x = _x(M, K, xdt, cfg=72)
            gamma = (1.0 + 0.1 * torch.from_numpy(synth.activations(74, 1, K))[0]).cuda().to(gdt)
            xd = x.double()
            ref = (xd * torch.rsqrt((xd * xd).mean(dim=1, keepdim=True) + 1e-5) * gamma.double()) @ wd.T
            bar = 2 * FAST if ydt == "f32" else 4e-3
            y = torch.empty((M, N), dtype=TDT[ydt], device="cuda")
            backend.matmul_norm(qw, x, gamma, 1e-5, y)
            torch.cuda.synchronize()
            assert ((y.double() - ref).norm() / ref.norm()).item() < bar, (xdt, ydt)
            y_again = torch.empty_like(y)
            backend.matmul_norm(qw, x, gamma, 1e-5, y_again)
            backend.set_gemm_tuning(2)                                     # two passes of the batched-rows decode kernel
            y_two = torch.empty_like(y)
            backend.matmul_norm(qw, x, gamma, 1e-5, y_two)
            backend.set_gemm_tuning(0)
            fewer = torch.empty((17, N), dtype=TDT[ydt], device="cuda")
            backend.matmul_norm(qw, x[:17].contiguous(), gamma, 1e-5, fewer)
            y_add = torch.empty_like(y)
            backend.matmul_norm(qw, x, gamma, 1e-5, y_add, epilogue="add", residual=r.to(TDT[ydt]))
            torch.cuda.synchronize()
            assert torch.equal(y, y_again)
            assert ((y.double() - y_two.double()).norm() / ref.norm()).item() < 2 * bar, (xdt, ydt)
            if ydt == "f32":
                assert not torch.equal(y, y_two)                           # (rounded operands, another order: it did run)
            assert torch.equal(y[:17], fewer)
            want = ref + r.to(TDT[ydt]).double()
            assert ((y_add.double() - want).norm() / want.norm()).item() < bar, (xdt, ydt)
    finally:
        backend.set_gemm_tuning(0)
    qw.free()


def test_lm_head_shape(backend, oracle):
    """The LM head of a Llama-3-sized vocabulary (decide/pipeline.md:51): 128256 rows, K = 4096, Q4 -
    8016 strips, several rounds of workgroups per CU.  Weights are made and quantised on the device;
    every output is checked against a float64 product over the exactly dequantised tensor (chunks of
    rows), a sample of rows against the oracle from the packed bytes."""
    N, K, bits = 128256, 4096, 4
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1234)
    w = torch.empty((N, K), dtype=torch.float32, device="cuda").normal_(0.0, 0.02, generator=gen)
    qd = torch.empty(N * K // 2, dtype=torch.uint8, device="cuda")
    sd = torch.empty(N * (K // 32), dtype=torch.int16, device="cuda")
    backend.quantize(bits, w, N, K, qd, sd)
    qw = backend.weight_from_device(bits, N, K, qd, sd)
    torch.cuda.synchronize()
    backend.dequant(qw, w)                       # w now holds scale * q, bit-exact (tested elsewhere)
    torch.cuda.synchronize()
    rows = torch.arange(0, N, 997, device="cuda")
    qrows = formats.unpack_planar(qd.view(N, K // 2)[rows].cpu().numpy().reshape(-1), bits, len(rows), K)
    srows = sd.view(N, K // 32)[rows].cpu().numpy().view(np.uint16)
    assert np.array_equal(oracle.dequant(qrows, srows), w[rows].cpu().numpy())
    for M, xdt in ((1, "f16"), (2, "f16"), (8, "f16"), (8, "bf16"), (20, "f16")):
        x = _x(M, K, xdt, cfg=51)
        y = _run(backend, qw, x)
        xd = x.double()
        num = den = 0.0
        for r0 in range(0, N, 16032):
            ref = xd @ w[r0:r0 + 16032].double().T
            num += ((y[:, r0:r0 + 16032].double() - ref) ** 2).sum().item()
            den += (ref ** 2).sum().item()
        assert (num / den) ** 0.5 < TIGHT, (M, xdt)
        ref = oracle.matmul_f64(qrows, srows, x.float().cpu().numpy())
        assert oracle.rel_l2(y[:, rows].cpu().numpy(), ref) < TIGHT, (M, xdt)


# ------------------------------------------------------- fused epilogues
# The reference's definitions of the ops around a linear are not in its tree (parity
# unpinned); the checks below pin the library's stated formulas: y = r + x W^T, and
# y = silu(x Wg^T) * (x Wu^T) with silu(t) = t / (1 + exp(-t)), against float64.

def _silu_mul(g, u):
    return g / (1.0 + np.exp(-g)) * u


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,xdt", [(1, "f16"), (2, "bf16"), (3, "f32"), (4, "f16"), (16, "bf16"), (40, "bf16"), (300, "f16")])
def test_epilogue_residual_add(backend, oracle, prefill_mode, bits, M, xdt):
    N, K = 272, 1024
    q, s = _quant(oracle, bits, N, K)
    qw = backend.upload_quantized(q, s, bits)
    x = _x(M, K, xdt)
    r = torch.from_numpy(synth.activations(33, M, N)).cuda()
    ref = oracle.matmul_f64(q, s, x.float().cpu().numpy()) + r.double().cpu().numpy()
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    backend.matmul_ex(qw, x, y, "add", r)
    torch.cuda.synchronize()
    bar = TIGHT if (M <= 16 or xdt == "f32") else _bar(prefill_mode)
    assert oracle.rel_l2(y.cpu().numpy(), ref) < bar
    # in place (residual aliases y) and with a 16-bit residual stream: added in fp32, rounded once
    y2 = r.clone()
    backend.matmul_ex(qw, x, y2, "add", y2)
    torch.cuda.synchronize()
    assert torch.equal(y2, y)
    rb = r.to(torch.bfloat16)
    yb = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    backend.matmul_ex(qw, x, yb, "add", rb)
    y32 = torch.empty((M, N), dtype=torch.float32, device="cuda")
    backend.matmul(qw, x, y32)
    torch.cuda.synchronize()
    assert torch.equal(yb, (y32 + rb.float()).to(torch.bfloat16))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,xdt", [(1, "f16"), (2, "bf16"), (3, "f32"), (4, "f16"), (9, "f16"), (16, "bf16"), (40, "bf16"), (300, "f16")])
def test_epilogue_swiglu(backend, oracle, prefill_mode, bits, M, xdt):
    N, K = 336, 1024                      # 21 strips per projection
    qg, sg = _quant(oracle, bits, N, K, cfg=41)
    qu, su = _quant(oracle, bits, N, K, cfg=42)
    wg = backend.upload_quantized(qg, sg, bits)
    wu = backend.upload_quantized(qu, su, bits)
    wf = backend.fuse_pairs(wg, wu)
    assert (wf.N, wf.K) == (2 * N, K)
    x = _x(M, K, xdt)
    xf = x.float().cpu().numpy()
    g, u = oracle.matmul_f64(qg, sg, xf), oracle.matmul_f64(qu, su, xf)
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    backend.matmul_ex(wf, x, y, "swiglu")
    torch.cuda.synchronize()
    assert not torch.isnan(y).any()
    bar = TIGHT if (M <= 16 or xdt == "f32") else 2 * _bar(prefill_mode)
    assert oracle.rel_l2(y.cpu().numpy(), _silu_mul(g, u)) < bar
    # the fused weight as a plain matmul: gate and up columns interleaved in blocks of 16
    if True:
        yi = _run(backend, wf, x)
        yg, yu = _run(backend, wg, x), _run(backend, wu, x)
        inter = torch.stack([yg.view(M, N // 16, 16), yu.view(M, N // 16, 16)], dim=2).reshape(M, 2 * N)
        if M <= 16:
            assert torch.equal(yi, inter)
            # and the epilogue is exactly silu * mul of those sums, in fp32
            want = (yg / (1.0 + torch.exp(-yg)) * yu)
            assert (y - want).abs().max().item() <= 2e-6 * want.abs().max().item()
        else:
            assert ((yi - inter).double().norm() / inter.double().norm()).item() < 1e-6


def test_epilogue_swiglu_full_size_and_split_k(backend, oracle):
    # Llama-3-8B FFN width at decode (M = 1, 8) and prefill (M = 128: 14 column tiles per row block,
    # so K is split over workgroups and the activation runs in the slab-adding kernel)
    K, N = 4096, 14336
    qg, sg = _quant(oracle, 4, N, K, cfg=43)
    qu, su = _quant(oracle, 4, N, K, cfg=44)
    wg, wu = backend.upload_quantized(qg, sg, 4), backend.upload_quantized(qu, su, 4)
    wf = backend.fuse_pairs(wg, wu)
    dg = torch.from_numpy(oracle.dequant(qg, sg)).cuda().double()
    du = torch.from_numpy(oracle.dequant(qu, su)).cuda().double()
    for M, xdt, bar in ((1, "f16", TIGHT), (8, "f16", TIGHT), (128, "bf16", 2 * FAST), (512, "bf16", 2 * FAST)):
        x = _x(M, K, xdt)
        g, u = x.double() @ dg.T, x.double() @ du.T
        ref = g / (1.0 + torch.exp(-g)) * u
        y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
        backend.matmul_ex(wf, x, y, "swiglu")
        torch.cuda.synchronize()
        err = ((y.double() - ref).norm() / ref.norm()).item()
        assert err < bar, (M, err)


def _norm_ref(oracle, q, s, x, gamma, eps, op_dt):
    """float64 restatement of the stated formula: x * gamma rounded once to the operand type,
    exact matmul, rows scaled by rstd of the unrounded input."""
    xf = x.float()
    xg = xf * gamma.float()[None, :]
    if op_dt == "f32":                                # two f16 halves keep ~22 bits: compare against unrounded
        xr = xg.double().cpu().numpy()
    else:
        xr = xg.to(TDT[op_dt]).double().cpu().numpy()
    rstd = 1.0 / np.sqrt((xf.double().cpu().numpy() ** 2).mean(axis=1) + eps)
    return oracle.matmul_f64(q, s, xr) * rstd[:, None]


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,xdt,gdt", [(1, "f16", "f16"), (2, "bf16", "f32"), (3, "f32", "f32"), (4, "f16", "bf16"), (9, "bf16", "bf16"),
                                       (16, "f16", "f32"), (16, "f32", "f16"), (40, "bf16", "f32"), (300, "f16", "f16"),
                                       (70, "f32", "f32")])
def test_folded_rmsnorm(backend, oracle, prefill_mode, bits, M, xdt, gdt):
    N, K = 272, 1184                                   # K = 9 tiles + 1 group: a padded last tile
    eps = 1e-5
    q, s = _quant(oracle, bits, N, K)
    qw = backend.upload_quantized(q, s, bits)
    x = _x(M, K, xdt)
    x[0] *= 7.0                                        # rows of different scale: rstd must be per row
    gamma = (1.0 + 0.25 * torch.from_numpy(synth.activations(51, 1, K)[0])).cuda().to(TDT[gdt])
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    backend.matmul_norm(qw, x, gamma, eps, y)
    torch.cuda.synchronize()
    assert not torch.isnan(y).any()
    fast_prefill = M > (16 if xdt == "f32" else 32) and prefill_mode == "fast"
    op_dt = "f16" if (fast_prefill and xdt != "f16") else xdt       # FAST multiplies in f16
    ref = _norm_ref(oracle, q, s, x, gamma, eps, op_dt)
    bar = FAST if fast_prefill else TIGHT
    assert oracle.rel_l2(y.cpu().numpy(), ref) < bar
    # reproducible, and composes with the epilogues
    y2 = torch.empty_like(y)
    backend.matmul_norm(qw, x, gamma, eps, y2)
    r = torch.from_numpy(synth.activations(52, M, N)).cuda()
    y3 = torch.empty_like(y)
    backend.matmul_norm(qw, x, gamma, eps, y3, "add", r)
    torch.cuda.synchronize()
    assert torch.equal(y2, y)
    assert torch.equal(y3, y + r)


@pytest.mark.parametrize("M,xdt", [(1, "f16"), (8, "f16"), (64, "bf16")])
def test_folded_rmsnorm_with_swiglu_and_long_k(backend, oracle, M, xdt):
    # FFN entry as the decode loop has it: norm -> gate/up -> SwiGLU; K long enough for several x slabs
    N, K = 192, 14336
    eps = 1e-6
    qg, sg = _quant(oracle, 4, N, K, cfg=45)
    qu, su = _quant(oracle, 4, N, K, cfg=46)
    wf = backend.fuse_pairs(backend.upload_quantized(qg, sg, 4), backend.upload_quantized(qu, su, 4))
    x = _x(M, K, xdt)
    gamma = (1.0 + 0.25 * torch.from_numpy(synth.activations(53, 1, K)[0])).cuda().to(torch.float32)
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    backend.matmul_norm(wf, x, gamma, eps, y, "swiglu")
    torch.cuda.synchronize()
    op_dt = "f16" if M > 16 else xdt
    g = _norm_ref(oracle, qg, sg, x, gamma, eps, op_dt)
    u = _norm_ref(oracle, qu, su, x, gamma, eps, op_dt)
    assert oracle.rel_l2(y.cpu().numpy(), _silu_mul(g, u)) < (2 * FAST if M > 16 else TIGHT)


@pytest.mark.parametrize("M,xdt,gdt", [(1, "f16", "f16"), (3, "f16", "f32"), (8, "bf16", "bf16"), (16, "f16", "f16"), (16, "bf16", "f32")])
def test_folded_rmsnorm_very_long_k(backend, oracle, M, xdt, gdt):
    # K far past anything a workgroup could keep of gamma in LDS at once
    N, K = 48, 32768
    q, s = _quant(oracle, 4, N, K, cfg=47)
    qw = backend.upload_quantized(q, s, 4)
    x = _x(M, K, xdt)
    gamma = (1.0 + 0.25 * torch.from_numpy(synth.activations(54, 1, K)[0])).cuda().to(TDT[gdt])
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    backend.matmul_norm(qw, x, gamma, 1e-6, y)
    torch.cuda.synchronize()
    assert oracle.rel_l2(y.cpu().numpy(), _norm_ref(oracle, q, s, x, gamma, 1e-6, xdt)) < TIGHT


@pytest.mark.parametrize("bits,N,K,M,ydt", [(4, 100, 16416, 257, "f32"), (4, 112, 16384, 300, "bf16"), (8, 130, 17000 // 32 * 32, 513, "f16"),
                                            (8, 224, 18432, 256, "f32"), (4, 2050, 6176, 200, "f32")])
def test_role_split_kernel_over_ranges_of_k(backend, oracle, bits, N, K, M, ydt):
    # K ranges of 16 tiles and more, a shorter last one, a padded last tile, row and column tiles that are not full, tiles of seven and
    # eight column blocks; with a residual, and the same twice over
    q, s = _quant(oracle, bits, N, K, cfg=49)
    qw = backend.upload_quantized(q, s, bits)
    x = _x(M, K, "bf16")
    r = torch.from_numpy(synth.activations(56, M, N)).cuda().to(TDT[ydt])
    y = torch.full((M, N), float("nan"), dtype=TDT[ydt], device="cuda")
    y2 = torch.empty_like(y)
    backend.set_gemm_tuning(2)          # (the tiled kernels alone: small outputs are other kernels' otherwise)
    try:
        backend.matmul_ex(qw, x, y, "add", r)
        backend.matmul_ex(qw, x, y2, "add", r)
        torch.cuda.synchronize()
    finally:
        backend.set_gemm_tuning(0)
    ref = oracle.matmul_f64(q, s, x.double().cpu().numpy()) + r.double().cpu().numpy()
    rounding = {"f32": 0.0, "f16": 5e-4, "bf16": 4e-3}[ydt]      # of the result
    assert oracle.rel_l2(y.double().cpu().numpy(), ref) < FAST + rounding
    assert torch.equal(y, y2)


# (the calls above are many ranges of small outputs, the last of them short ranges, which are gemm_kernel's.)  Two, three, four ranges and
# more, one to five row tiles, seven and eight column blocks, a last range that is shorter
@pytest.mark.parametrize("bits,N,K,M,nf,splits", [(4, 2050, 16416, 200, 8, 8), (4, 4000, 6176, 700, 8, 2), (8, 3584, 6176, 700, 7, 2), (4, 3100, 6176, 520, 8, 3),
                                                  (4, 3600, 8224, 300, 8, 4), (8, 1568, 12320, 513, 7, 6), (4, 1000, 12320, 1030, 7, 5)])
def test_ranges_of_k_have_the_same_bits_in_both_tiled_kernels(backend, oracle, bits, N, K, M, nf, splits):
    """With roles or with waves that do everything (tuning 2 and 7) a K range is walked and left in its slab alike: plain, with a
    residual, with a folded norm of bf16 and of f16 rows, as a pair."""
    qw, wd = _random_weight(backend, bits, N, K, seed=71)
    r = torch.from_numpy(synth.activations(72, M, N)).cuda()
    gamma = (1.0 + 0.1 * torch.from_numpy(synth.activations(73, 1, K))[0]).cuda()
    half = N // 32 * 16
    qh, hd = _random_weight(backend, bits, half, K, seed=74)
    pair = backend.fuse_pairs(qh, qh)
    codes = {"f32": 0, "f16": 1, "bf16": 2}

    def both(w, n, xdt, ydt, call, norm=False, epilogue="none"):
        out = []
        for tuning, kernel in ((2, "roles"), (7, "tiles")):
            backend.set_gemm_tuning(tuning)
            plan = backend.debug_prefill_plan(w, codes[xdt], M, norm, epilogue)
            assert plan["kernel"] == kernel and plan["splits"] >= 2, plan
            if w is qw:
                assert (plan["nf"], plan["splits"]) == (nf, splits), plan
            y = torch.full((M, n), float("nan"), dtype=TDT[ydt], device="cuda")
            call(y)
            out.append(y)
        torch.cuda.synchronize()
        assert torch.equal(*out), (xdt, ydt, norm, epilogue)
        return out[0].double()

    def rel(y, ref):
        return ((y - ref).norm() / ref.norm()).item()

    try:
        x = _x(M, K, "bf16", cfg=75)
        ref = x.double() @ wd.T
        assert rel(both(qw, N, "bf16", "f32", lambda y: backend.matmul(qw, x, y)), ref) < FAST
        rb = r.bfloat16()
        assert rel(both(qw, N, "bf16", "bf16", lambda y: backend.matmul_ex(qw, x, y, "add", rb), epilogue="add"), ref + rb.double()) < 4e-3
        for xdt in ("bf16", "f16"):
            x = _x(M, K, xdt, cfg=75)
            xd = x.double()
            ref = (xd * torch.rsqrt((xd * xd).mean(dim=1, keepdim=True) + 1e-5) * gamma.double()) @ wd.T + r.double()
            y = both(qw, N, xdt, "f32", lambda y: backend.matmul_norm(qw, x, gamma, 1e-5, y, "add", r), norm=True, epilogue="add")
            assert rel(y, ref) < 2 * FAST, xdt
        z = xd @ hd.T
        y = both(pair, half, "f16", "f16", lambda y: backend.matmul_ex(pair, x, y, "swiglu"), epilogue="swiglu")
        assert rel(y, torch.nn.functional.silu(z) * z) < 4e-3
    finally:
        backend.set_gemm_tuning(0)
    for w in (qw, qh, pair):
        w.free()


@pytest.mark.parametrize("xdt,gdt", [("bf16", "f16"), ("bf16", "f32"), ("f32", "bf16")])
@pytest.mark.parametrize("K", [32, 512, 544, 2048, 2080, 4128, 8224, 16416])
def test_row_scaling_pass_at_the_edges_of_its_pieces(backend, oracle, K, xdt, gdt):
    # pieces of 512 k, shared out to a row's waves: fewer pieces than waves, a last piece of one group, one more than all
    # waves hold in a round, rows that do not stay in registers; with a folded norm and without (other rows per workgroup)
    M, N, eps = 37, 48, 1e-5
    q, s = _quant(oracle, 4, N, K, cfg=48)
    qw = backend.upload_quantized(q, s, 4)
    x = _x(M, K, xdt)
    x[1] *= 1e-6                                       # another power of two, another rstd
    gamma = (1.0 + 0.25 * torch.from_numpy(synth.activations(55, 1, K)[0])).cuda().to(TDT[gdt])
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    backend.matmul_norm(qw, x, gamma, eps, y)
    plain = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    backend.matmul(qw, x, plain)
    torch.cuda.synchronize()
    assert oracle.rel_l2(y.cpu().numpy(), _norm_ref(oracle, q, s, x, gamma, eps, "f32")) < 2 * FAST     # x * gamma and scale * q rounded
    ref = oracle.matmul_f64(q, s, x.double().cpu().numpy())
    got = plain.cpu().numpy()
    assert oracle.rel_l2(got, ref) < FAST and oracle.rel_l2(got[1:2], ref[1:2]) < FAST


# (plain bf16 rows of the calls above go to other kernels, and many of the fp32 ones have one way of sharing out.)  A workgroup's sixteen waves share out its
# rows' pieces of 512 k: sixteen, eight, four to a row with one, two, four rows to the workgroup.  One piece and fewer than waves, a last piece of one group, as many
# as stay in registers, one more; rows that are no multiple of the workgroup's
@pytest.mark.parametrize("xdt,rows,M,K", [
    ("bf16", 1, 37, 8224), ("bf16", 1, 37, 16384), ("bf16", 1, 37, 16416), ("bf16", 1, 33, 32768), ("bf16", 1, 33, 32800),
    ("bf16", 2, 37, 32), ("bf16", 2, 37, 512), ("bf16", 2, 37, 544), ("bf16", 2, 37, 4096), ("bf16", 2, 37, 4128), ("bf16", 2, 37, 8192),
    ("bf16", 2, 133, 8224), ("bf16", 2, 133, 16384), ("bf16", 2, 133, 16416),
    ("bf16", 4, 53, 32), ("bf16", 4, 53, 2080), ("bf16", 4, 53, 4096), ("bf16", 4, 53, 4128), ("bf16", 4, 53, 8192),
    ("bf16", 4, 389, 8224), ("bf16", 4, 389, 16384), ("bf16", 4, 389, 16416),
    ("f32", 1, 33, 16416), ("f32", 1, 33, 32800), ("f32", 2, 37, 4128), ("f32", 2, 133, 16416), ("f32", 4, 53, 2048), ("f32", 4, 53, 2080),
    ("f32", 4, 53, 4128), ("f32", 4, 517, 8224)])
def test_row_scaling_pass_with_one_two_and_four_rows_to_a_workgroup(backend, oracle, xdt, rows, M, K):
    N = 48
    q, s = _quant(oracle, 4, N, K, cfg=76)
    qw = backend.upload_quantized(q, s, 4)
    x = _x(M, K, xdt, cfg=77)
    x[1] *= 1e-6                                       # another power of two
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    backend.set_gemm_tuning(2)                         # the tiled kernels, and no decode passes in their place
    backend.set_gemv_tuning(0, 2, 0)
    try:
        plan = backend.debug_prefill_plan(qw, {"f32": 0, "bf16": 2}[xdt], M)
        assert plan["stage_rows"] == rows and plan["kernel"] in ("tiles", "roles"), plan
        backend.matmul(qw, x, y)
        torch.cuda.synchronize()
    finally:
        backend.set_gemm_tuning(0)
        backend.set_gemv_tuning(0, 0, 0)
    ref = x.double() @ torch.from_numpy(oracle.dequant(q, s)).cuda().double().T
    errs = ((y.double() - ref).norm(dim=1) / ref.norm(dim=1)).cpu()
    assert errs.max().item() < 2 * FAST, int(errs.argmax())     # (a row's 48 outputs; FAST is for all of a call's)


# (residuals asked for ahead of the sums, and not: Q8, eight rows and fewer, seven strips and more)
@pytest.mark.parametrize("bits,N,K,M,xdt", [(4, 28672, 4128, 9, "f16"), (4, 28672, 4128, 16, "bf16"), (4, 28670, 4128, 5, "f16"), (8, 6144, 4128, 9, "f16"),
                                            (8, 6150, 4128, 16, "bf16"), (4, 9212, 4128, 13, "f16"), (4, 9212, 4128, 7, "bf16"), (4, 6142, 4128, 12, "bf16"),
                                            (4, 6142, 4128, 3, "f16"), (4, 4096, 4128, 11, "f16"), (4, 6142, 1056, 16, "f32"), (4, 6142, 1056, 6, "f32")])
def test_folded_rmsnorm_with_a_residual_on_several_strips(backend, bits, N, K, M, xdt):
    qw, wd = _random_weight(backend, bits, N, K, seed=78)
    x = _x(M, K, xdt, cfg=79)
    gamma = (1.0 + 0.25 * torch.from_numpy(synth.activations(80, 1, K)[0])).cuda().to(TDT[xdt])
    r = torch.from_numpy(synth.activations(81, M, N)).cuda()
    xd = x.double()
    # x * gamma is an operand of 16 bits where the rows are
    v = (xd * gamma.double()).to(TDT[xdt]).double() if xdt != "f32" else xd * gamma.double()
    ref = (v * torch.rsqrt((xd * xd).mean(dim=1, keepdim=True) + 1e-5)) @ wd.T
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    for epilogue, res, want in (("none", None, ref), ("add", r, ref + r.double())):
        backend.matmul_norm(qw, x, gamma, 1e-5, y, epilogue, res)
        torch.cuda.synchronize()
        assert ((y.double() - want).norm() / want.norm()).item() < TIGHT, epilogue
    y.copy_(r)                                          # the output over the residual
    backend.matmul_norm(qw, x, gamma, 1e-5, y, "add", y)
    torch.cuda.synchronize()
    assert ((y.double() - want).norm() / want.norm()).item() < TIGHT
    qw.free()


# (more than four rows per CU: the row-scaling pass loads gamma twice and two of its workgroups share a CU)
@pytest.mark.parametrize("M", [1024, 1030])
@pytest.mark.parametrize("K,gdt", [(4128, "f32"), (6144, "f16"), (8192, "bf16")])
def test_folded_rmsnorm_of_many_rows(backend, oracle, M, K, gdt):
    N, eps = 48, 1e-5
    q, s = _quant(oracle, 4, N, K, cfg=82)
    qw = backend.upload_quantized(q, s, 4)
    x = _x(M, K, "bf16", cfg=83)
    x[1] *= 1e-6
    gamma = (1.0 + 0.25 * torch.from_numpy(synth.activations(84, 1, K)[0])).cuda().to(TDT[gdt])
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    assert backend.debug_prefill_plan(qw, 2, M, norm=True)["stage_rows"] == 4
    backend.matmul_norm(qw, x, gamma, eps, y)
    torch.cuda.synchronize()
    xd = x.double()
    ref = (xd * torch.rsqrt((xd * xd).mean(dim=1, keepdim=True) + eps) * gamma.double()) @ torch.from_numpy(oracle.dequant(q, s)).cuda().double().T
    errs = ((y.double() - ref).norm(dim=1) / ref.norm(dim=1)).cpu()
    assert ((y.double() - ref).norm() / ref.norm()).item() < 2 * FAST and errs.max().item() < 4 * FAST, int(errs.argmax())


# (fewer than eight waves finish a workgroup's outputs)
@pytest.mark.parametrize("bits,N,K,M,xdt", [(4, 24922, 384, 11, "f16"), (4, 9000, 256, 3, "f16"), (8, 8533, 320, 5, "f16"), (4, 5790, 1120, 32, "bf16"), (4, 4099, 1920, 16, "f16"),
                                            (4, 12290, 896, 16, "f32"), (8, 12290, 1056, 23, "bf16"), (4, 28672, 640, 8, "bf16")])
def test_batched_rows_of_a_short_k_with_a_residual(backend, bits, N, K, M, xdt):
    qw, wd = _random_weight(backend, bits, N, K, seed=85)
    x = _x(M, K, xdt, cfg=86)
    r = torch.from_numpy(synth.activations(87, M, N)).cuda()
    ref = x.double() @ wd.T
    assert ((_run(backend, qw, x).double() - ref).norm() / ref.norm()).item() < TIGHT
    y = r.clone()                                       # the output over the residual
    backend.matmul_ex(qw, x, y, "add", y)
    torch.cuda.synchronize()
    want = ref + r.double()
    assert ((y.double() - want).norm() / want.norm()).item() < TIGHT
    qw.free()


@pytest.mark.parametrize("M", [1, 2, 4, 16])
def test_folded_rmsnorm_counts_subnormal_inputs(backend, oracle, M):
    # a row of f16 subnormals (|x| < 6.1e-5) with an eps far below its mean square: its squares must
    # not be flushed on the way into the sum
    N, K = 64, 1024
    eps = 1e-14
    q, s = _quant(oracle, 4, N, K, cfg=48)
    qw = backend.upload_quantized(q, s, 4)
    x = _x(M, K, "f16")
    x[M - 1] = (x[M - 1].float() * 1e-5).to(torch.float16)
    assert x[M - 1].float().abs().max().item() < 6.1e-5
    gamma = torch.ones(K, dtype=torch.float16, device="cuda")
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    backend.matmul_norm(qw, x, gamma, eps, y)
    torch.cuda.synchronize()
    ref = _norm_ref(oracle, q, s, x, gamma, eps, "f16")
    assert oracle.rel_l2(y[M - 1:].cpu().numpy(), ref[M - 1:]) < TIGHT
    assert oracle.rel_l2(y.cpu().numpy(), ref) < TIGHT


def _random_cases(seed, count):
    """Seeded draws over everything a call can vary in: block type, interchange layout, ragged N / K,
    batch rows on both sides of every kernel boundary, the three activation types, output type,
    epilogue, folded norm, prefill mode.  CYBQ_FUZZ_SEED / CYBQ_FUZZ_COUNT widen the sweep by hand."""
    rng = np.random.default_rng(seed)
    rows = [1, 2, 3, 4, 5, 8, 13, 16, 17, 24, 31, 32, 33, 48, 100, 129, 257, 300]
    cases = []
    for i in range(count):
        epi = ["none", "add", "swiglu"][int(rng.integers(0, 3))]
        N = int(rng.integers(1, 30)) * 16 if epi == "swiglu" else int(rng.integers(1, 500))
        K = 32 * int(rng.integers(1, 150)) if rng.random() < 0.8 else 32 * int(rng.integers(150, 600))
        cases.append(dict(i=i, bits=int(rng.choice([4, 8])), layout=int(rng.choice([formats.PLANAR, formats.BLOCK_AOS])),
                          N=N, K=K, M=int(rng.choice(rows)), xdt=str(rng.choice(["f16", "bf16", "f32"])),
                          ydt=str(rng.choice(["f32", "f32", "f16", "bf16"])), epi=epi, norm=bool(rng.random() < 0.4),
                          gdt=str(rng.choice(["f32", "f16", "bf16"])), mode=str(rng.choice(["fast", "exact"]))))
    return cases


@pytest.mark.parametrize("case", _random_cases(int(__import__("os").environ.get("CYBQ_FUZZ_SEED", "20240607")), int(__import__("os").environ.get("CYBQ_FUZZ_COUNT", "72"))), ids=lambda c: "-".join(str(v) for v in c.values()))
def test_random_calls_match_float64(backend, oracle, case):
    _check_random_case(backend, oracle, case)


def _random_wide_cases(seed, count):
    """The same draws over outputs wide enough for workgroups of two, four, seven or eight strips, several
    rounds of workgroups, one round of narrow prefill tiles: the variants the model shapes run, on a short K."""
    rng = np.random.default_rng(seed)
    rows = [1, 2, 3, 4, 7, 8, 12, 16, 17, 24, 32, 33, 48, 64, 100, 128, 200, 256, 300, 512]
    cases = []
    for i in range(count):
        epi = ["none", "add", "swiglu"][int(rng.integers(0, 3))]
        N = int(rng.choice([4096, 7168, 14336])) if epi == "swiglu" else int(rng.choice([6144, 8192, 9008, 12288, 14336, 16400, 28672]))
        cases.append(dict(i=1000 + i, bits=int(rng.choice([4, 4, 8])), layout=int(rng.choice([formats.PLANAR, formats.BLOCK_AOS])),
                          N=N, K=32 * int(rng.integers(1, 25)), M=int(rng.choice(rows)), xdt=str(rng.choice(["f16", "bf16", "f32"])),
                          ydt=str(rng.choice(["f32", "f32", "f16", "bf16"])), epi=epi, norm=bool(rng.random() < 0.3),
                          gdt=str(rng.choice(["f32", "f16", "bf16"])), mode=str(rng.choice(["fast", "fast", "exact"]))))
    return cases


@pytest.mark.parametrize("case", _random_wide_cases(20240608, int(__import__("os").environ.get("CYBQ_FUZZ_WIDE_COUNT", "48"))), ids=lambda c: "-".join(str(v) for v in c.values()))
def test_random_wide_calls_match_float64(backend, oracle, case):
    _check_random_case(backend, oracle, case)


def _random_mid_k_cases(seed, count):
    """Draws over K of 16 .. 34 tiles with few rows on a wide output or up to 512 rows on a narrow one: the calls
    whose 64-row pieces fill one round of workgroups (the prefill kernel whose waves split K), their neighbours
    that do not, and the modes and epilogues around them."""
    rng = np.random.default_rng(seed)
    cases = []
    for i in range(count):
        wide = bool(rng.random() < 0.4)
        N = int(rng.choice([8192, 8200, 12288, 14336])) if wide else int(rng.choice([1024, 1040, 2048, 3072, 4096, 6144]))
        M = int(rng.choice([17, 24, 33, 48, 64])) if wide else int(rng.choice([17, 40, 65, 100, 128, 129, 200, 256, 300, 384, 512]))
        cases.append(dict(i=2000 + i, bits=int(rng.choice([4, 4, 8])), layout=int(rng.choice([formats.PLANAR, formats.BLOCK_AOS])),
                          N=N, K=128 * int(rng.integers(16, 35)), M=M, xdt=str(rng.choice(["f16", "bf16", "f32"])),
                          ydt=str(rng.choice(["f32", "f32", "f16", "bf16"])), epi=str(rng.choice(["none", "add"])),
                          norm=bool(rng.random() < 0.3), gdt=str(rng.choice(["f32", "f16", "bf16"])),
                          mode=str(rng.choice(["fast", "fast", "fast", "exact"]))))
    return cases


@pytest.mark.parametrize("case", _random_mid_k_cases(20240609, int(__import__("os").environ.get("CYBQ_FUZZ_MID_COUNT", "24"))), ids=lambda c: "-".join(str(v) for v in c.values()))
def test_random_mid_k_calls_match_float64(backend, oracle, case):
    _check_random_case(backend, oracle, case)


def _check_random_case(backend, oracle, c):
    bits, N, K, M = c["bits"], c["N"], c["K"], c["M"]
    backend.set_prefill_mode(c["mode"])
    try:
        x = _x(M, K, c["xdt"], cfg=60 + c["i"])
        if M > 1:
            x[M // 2] *= 5.0
        gamma = (1.0 + 0.25 * torch.from_numpy(synth.activations(61, 1, K)[0])).cuda().to(TDT[c["gdt"]])
        eps = 1e-5
        prefill = (M > 32 and c["xdt"] != "f32") or (M > 16 and c["xdt"] == "f32" and c["mode"] == "fast")
        fast = prefill and c["mode"] == "fast"
        op_dt = "f16" if (fast and c["xdt"] != "f16") else c["xdt"]

        def product(q, s):
            if c["norm"]:
                return _norm_ref(oracle, q, s, x, gamma, eps, op_dt)
            return oracle.matmul_f64(q, s, x.float().cpu().numpy())

        if c["epi"] == "swiglu":
            qg, sg = _quant(oracle, bits, N, K, cfg=70 + c["i"])
            qu, su = _quant(oracle, bits, N, K, cfg=170 + c["i"])
            w = backend.fuse_pairs(backend.upload_quantized(qg, sg, bits, c["layout"]),
                                   backend.upload_quantized(qu, su, bits, c["layout"]))
            ref = _silu_mul(product(qg, sg), product(qu, su))
        else:
            q, s = _quant(oracle, bits, N, K, cfg=70 + c["i"])
            w = backend.upload_quantized(q, s, bits, c["layout"])
            ref = product(q, s)
        r = None
        if c["epi"] == "add":
            r = torch.from_numpy(synth.activations(62, M, N)).cuda().to(TDT[c["ydt"]])
            ref = ref + r.double().cpu().numpy()
        y = torch.full((M, N), float("nan"), dtype=TDT[c["ydt"]], device="cuda")
        if c["norm"]:
            backend.matmul_norm(w, x, gamma, eps, y, c["epi"], r)
        else:
            backend.matmul_ex(w, x, y, c["epi"], r)
        torch.cuda.synchronize()
        assert not torch.isnan(y).any(), c
        bar = FAST if fast else TIGHT
        if c["epi"] == "swiglu":
            bar *= 2
        if c["ydt"] == "f16":
            bar = max(bar, 6e-4)                          # one rounding to 11 bits
        if c["ydt"] == "bf16":
            bar = max(bar, 4e-3)                          # one rounding to 8 bits
        err = oracle.rel_l2(y.float().cpu().numpy(), ref)
        assert err < bar, (c, err)
        w.free()
    finally:
        backend.set_prefill_mode("fast")


def test_epilogue_errors(backend, oracle):
    q, s = _quant(oracle, 4, 64, 256)
    qw = backend.upload_quantized(q, s, 4)
    x = _x(2, 256, "f16")
    y = torch.empty((2, 64), dtype=torch.float32, device="cuda")
    with pytest.raises(CybqError):
        backend.matmul_ex(qw, x, y, "swiglu")                 # not a fused pair
    with pytest.raises(CybqError):
        backend.matmul_ex(qw, x, y, "add", None)              # no residual
    q2, s2 = _quant(oracle, 4, 40, 256)
    with pytest.raises(CybqError):
        backend.fuse_pairs(backend.upload_quantized(q2, s2, 4), backend.upload_quantized(q2, s2, 4))   # N % 16
    with pytest.raises(CybqError):
        backend.fuse_pairs(qw, backend.upload_quantized(q2, s2, 4))                                    # shapes differ


# ------------------------------------------------------------------ quantise

@pytest.mark.parametrize("bits", [4, 8])
def test_device_quantizer_bit_exact(backend, oracle, bits):
    N, K = 300, 1024
    w = synth.weights(31, N, K)
    w[0, :32] = 0
    w[1, 32:64] *= 1e-6
    w[2, 5] = 0.35
    src = torch.from_numpy(w).cuda()
    qd = torch.empty(N * K * bits // 8, dtype=torch.uint8, device="cuda")
    sd = torch.empty(N * K // 32, dtype=torch.int16, device="cuda")
    backend.quantize(bits, src, N, K, qd, sd)
    torch.cuda.synchronize()
    q, s = oracle.quantize(w, bits)
    assert np.array_equal(sd.cpu().numpy().view(np.uint16).reshape(N, -1), s)
    assert np.array_equal(qd.cpu().numpy(), oracle.pack_planar(q, bits))
    # device buffers -> weight handle -> the op, without touching the host
    qw = backend.weight_from_device(bits, N, K, qd, sd)
    out = torch.empty((N, K), dtype=torch.float32, device="cuda")
    backend.dequant(qw, out)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy().view(np.uint32), oracle.dequant(q, s).view(np.uint32))


# quotients at and next to the half-integers (the ties the quantiser rounds away from zero, and the values whose correctly
# rounded quotient is a tie although they are not), scales from subnormal f16 to the largest; a last workgroup of one group
@pytest.mark.parametrize("bits", [4, 8])
def test_device_quantizer_at_the_ties(backend, oracle, bits):
    qmax = 7 if bits == 4 else 127
    K, rows = 32 * 65, []
    for d in np.array([1, 3, 1023, 1024, 5000, 15360, 15361, 20001, 31743], dtype=np.uint16).view(np.float16).astype(np.float32):
        half = (np.arange(qmax, dtype=np.float32) + np.float32(0.5)) * d
        below, above = np.nextafter(half, np.float32(0)), np.nextafter(half, np.float32(np.inf))
        v = np.concatenate([half, below, above, np.nextafter(below, np.float32(0)), half * np.float32(1 + 2e-6), half * np.float32(1 - 2e-6)])
        v = np.resize(np.concatenate([v, -v]), (K // 32, 31))
        rows.append(np.concatenate([np.full((K // 32, 1), np.float32(qmax) * d, dtype=np.float32), v], axis=1).reshape(-1))
    w = np.stack(rows).astype(np.float32)
    N = w.shape[0]
    qd = torch.empty(N * K * bits // 8, dtype=torch.uint8, device="cuda")
    sd = torch.empty(N * K // 32, dtype=torch.int16, device="cuda")
    backend.quantize(bits, torch.from_numpy(w).cuda(), N, K, qd, sd)
    torch.cuda.synchronize()
    q, s = oracle.quantize(w, bits)
    assert np.array_equal(sd.cpu().numpy().view(np.uint16).reshape(N, -1), s)
    assert np.array_equal(qd.cpu().numpy(), oracle.pack_planar(q, bits))


# ------------------------------------------------------------ interface / errors

def test_graph_node_execution(backend, oracle):
    N, K = 64, 128
    q, s = _quant(oracle, 4, N, K)
    backend.upload_quantized(q, s, 4, name="model.layers.0.self_attn.q_proj.weight")
    node = QMatMul(w="model.layers.0.self_attn.q_proj.weight", x="h0", y="q0", quant=4, M=2, N=N, K=K)
    edges = {"h0": _x(2, K, "f16"), "q0": torch.empty((2, N), dtype=torch.float32, device="cuda")}
    backend.run(node, edges)
    torch.cuda.synchronize()
    assert oracle.rel_l2(edges["q0"].cpu().numpy(),
                         oracle.matmul_f64(q, s, edges["h0"].float().cpu().numpy())) < TIGHT
    with pytest.raises(CybqError):
        backend.run(QMatMul(w="missing", x="h0", y="q0"), edges)
    with pytest.raises(CybqError):
        backend.run(QMatMul(w=node.w, x="h0", y="q0", quant=4, N=N + 16, K=K), edges)


def test_error_codes(backend, oracle):
    q, s = _quant(oracle, 4, 16, 64)
    with pytest.raises(CybqError) as e:
        backend.upload(4, formats.PLANAR, 16, 48, formats.pack_planar(q, 4), s)       # K % 32
    assert e.value.status == -2
    with pytest.raises(CybqError) as e:
        backend.upload(4, formats.PLANAR, 16, 64, formats.pack_planar(q, 4), None)    # no scales
    assert e.value.status == -1
    with pytest.raises(CybqError) as e:
        backend.upload(5, formats.PLANAR, 16, 64, formats.pack_planar(q, 4), s)       # bad quant
    assert e.value.status == -1
    with pytest.raises(CybqError) as e:
        backend.upload(4, formats.PLANAR, 32, 64, formats.pack_planar(q, 4), s)       # buffers of a 16-row tensor
    assert e.value.status == -2
    qw = backend.upload_quantized(q, s, 4)
    x = _x(2, 64, "f16")
    y = torch.empty((2, 16), dtype=torch.float32, device="cuda")
    with pytest.raises(CybqError) as e:
        backend.matmul(qw, x, y, M=0)
    assert e.value.status == -2
    # the host wrapper refuses tensors the library could only see as raw pointers of the wrong size
    for bad_x, bad_y in ((x[:1], y), (x, y[:1]), (x.t().contiguous().t(), y), (x.cpu(), y)):
        with pytest.raises(CybqError) as e:
            backend.matmul(qw, bad_x, bad_y, M=2)
        assert e.value.status in (-1, -2)
    buf = torch.empty(2 * 64 + 8, dtype=torch.float16, device="cuda")
    with pytest.raises(CybqError) as e:
        backend.matmul(qw, buf.data_ptr() + 2, y, M=2, xdt=1)                         # misaligned x
    assert e.value.status == -3
    # the context stays usable after errors
    backend.matmul(qw, x, y)
    torch.cuda.synchronize()
    assert oracle.rel_l2(y.cpu().numpy(), oracle.matmul_f64(q, s, x.float().cpu().numpy())) < TIGHT


# ------------------------------------------------------------ decode-step stack

def test_decode_stack_small(backend, oracle):
    """Config 5 in miniature: 2 layers x 7 linears of a scaled-down LlamaStyle model,
    weights generated and quantised on the device, every linear checked on its own."""
    from cyb_amd import stack
    shapes = {"q_proj": (512, 512), "k_proj": (512, 128), "v_proj": (512, 128), "o_proj": (512, 512),
              "gate_proj": (512, 1792), "up_proj": (512, 1792), "down_proj": (1792, 512)}
    st = stack.build(backend, layers=2, seed=5, keep_planar=2, shapes=shapes)
    assert len(st.nodes) == 14
    for M in (1, 8):
        edges = stack.edges_for(st, M, shapes=shapes)
        pl = stack.plan(st, edges)
        # run linear by linear so that every output can be read before it is overwritten
        for i, node in enumerate(st.nodes):
            node.M = M
            backend.run(node, edges)
            torch.cuda.synchronize()
            qd, sd = st.planar[node.w]
            q = formats.unpack_planar(qd.cpu().numpy(), 4, node.N, node.K)
            s = sd.cpu().numpy().view(np.uint16).reshape(node.N, node.K // 32)
            ref = oracle.matmul_f64(q, s, edges[node.x].float().cpu().numpy())
            assert oracle.rel_l2(edges[node.y].cpu().numpy(), ref) < TIGHT, node.w
        # and the whole step through the native node walk gives the last layer's outputs
        backend.matmul_many(pl, M)
        torch.cuda.synchronize()
        last = st.nodes[-1]
        qd, sd = st.planar[last.w]
        q = formats.unpack_planar(qd.cpu().numpy(), 4, last.N, last.K)
        s = sd.cpu().numpy().view(np.uint16).reshape(last.N, last.K // 32)
        ref = oracle.matmul_f64(q, s, edges[last.x].float().cpu().numpy())
        assert oracle.rel_l2(edges[last.y].cpu().numpy(), ref) < TIGHT
    assert st.step_bytes(1) == sum(formats.matmul_bytes(4, n.N, n.K, 1, 2, 4) for n in st.nodes)
    for w in st.weights:
        w.free()


def test_decode_stack_with_epilogues(backend, oracle):
    """The fused node list (qkv, o + residual, gate/up with SwiGLU, down + residual) through
    cybq_matmul_many_ex; every node's output recomputed from the weights the stack kept."""
    from cyb_amd import stack
    base = {"q_proj": (512, 512), "k_proj": (512, 128), "v_proj": (512, 128), "o_proj": (512, 512),
            "gate_proj": (512, 1792), "up_proj": (512, 1792), "down_proj": (1792, 512)}
    shapes = stack.fused_shapes(base)
    st = stack.build(backend, layers=2, seed=6, keep_planar=2, shapes=shapes, order=list(shapes), epilogues=True)
    assert st.epilogues == ["none", "add", "swiglu", "add"] * 2
    for M in (1, 8, 40):
        edges = stack.edges_for(st, M, shapes=shapes, xdtype=torch.bfloat16 if M > 16 else None)
        pl = stack.plan(st, edges)
        backend.matmul_many(pl, M)
        torch.cuda.synchronize()
        bar = TIGHT if M <= 16 else 2 * FAST
        for node, epi in list(zip(st.nodes, st.epilogues))[-4:]:          # the last layer's outputs are still in place
            qd, sd = st.planar[node.w]
            q = formats.unpack_planar(qd.cpu().numpy(), 4, node.N, node.K)
            s = sd.cpu().numpy().view(np.uint16).reshape(node.N, node.K // 32)
            ref = oracle.matmul_f64(q, s, edges[node.x].float().cpu().numpy())
            if epi == "add":
                ref = ref + edges[f"res.{node.N}"].double().cpu().numpy()
            elif epi == "swiglu":
                h = node.N // 2
                ref = _silu_mul(ref[:, :h], ref[:, h:])
            got = edges[node.y].cpu().numpy()
            assert got.shape == ref.shape
            assert oracle.rel_l2(got, ref) < bar, (M, node.w, epi)
    for w in st.weights:
        w.free()


def test_decode_stack_with_norms(backend, oracle):
    """A whole layer's linear path in one native walk (cybq_matmul_many_norm): RMSNorm folded in front
    of qkv and gate/up, SwiGLU and the two residual adds in the epilogues.  Every node of the last
    layer against the float64 restatement, and against the one-node entry point bit for bit."""
    from cyb_amd import stack
    base = {"q_proj": (512, 512), "k_proj": (512, 128), "v_proj": (512, 128), "o_proj": (512, 512),
            "gate_proj": (512, 1792), "up_proj": (512, 1792), "down_proj": (1792, 512)}
    shapes = stack.fused_shapes(base)
    st = stack.build(backend, layers=2, seed=8, keep_planar=2, shapes=shapes, order=list(shapes), epilogues=True, norms=True)
    assert [g is not None for g in st.gammas] == [True, False, True, False] * 2
    assert st.gammas[0] is not st.gammas[2] and st.gammas[0] is not st.gammas[4]
    for M in (1, 2, 8, 40):
        xdt = "bf16" if M > 16 else "f16"
        edges = stack.edges_for(st, M, shapes=shapes, xdtype=torch.bfloat16 if M > 16 else None)
        pl = stack.plan(st, edges)
        backend.matmul_many(pl, M)
        torch.cuda.synchronize()
        bar = TIGHT if M <= 16 else 2 * FAST
        for i in range(len(st.nodes) - 4, len(st.nodes)):                 # the last layer's outputs are still in place
            node, epi, gamma = st.nodes[i], st.epilogues[i], st.gammas[i]
            if gamma is None:
                ref = _node_reference(oracle, st, node, epi, edges)
            else:
                qd, sd = st.planar[node.w]
                q = formats.unpack_planar(qd.cpu().numpy(), 4, node.N, node.K)
                s = sd.cpu().numpy().view(np.uint16).reshape(node.N, node.K // 32)
                ref = _norm_ref(oracle, q, s, edges[node.x], gamma, st.eps, "f16" if M > 16 else xdt)
                if epi == "swiglu":
                    ref = _silu_mul(ref[:, :node.N // 2], ref[:, node.N // 2:])
            got = edges[node.y]
            assert oracle.rel_l2(got.cpu().numpy(), ref) < bar, (M, node.w, epi)
            one = torch.empty_like(got)
            res = edges[f"res.{node.N}"] if epi == "add" else None
            if gamma is None:
                backend.matmul_ex(st.weights[i], edges[node.x], one, epi, res)
            else:
                backend.matmul_norm(st.weights[i], edges[node.x], gamma, st.eps, one, epi, res)
            torch.cuda.synchronize()
            assert torch.equal(one, got), (M, node.w)
    for w in st.weights:
        w.free()


def test_many_norm_without_gammas_is_many_ex_and_rejects_bad_arguments(backend, oracle):
    """cybq_matmul_many_norm with no gamma anywhere is cybq_matmul_many_ex bit for bit; a node whose gamma is
    NULL runs without a norm; errors come back as values."""
    N, K, M = 96, 512, 5
    q, s = _quant(oracle, 4, N, K, cfg=95)
    w = backend.upload_quantized(q, s, 4)
    x = _x(M, K, "f16", cfg=96)
    gamma = (1.0 + 0.25 * torch.from_numpy(synth.activations(97, 1, K)[0])).cuda().to(torch.float16)
    y_plain = torch.empty((M, N), dtype=torch.float32, device="cuda")
    y_norm = torch.empty_like(y_plain)
    backend.matmul(w, x, y_plain)
    backend.matmul_norm(w, x, gamma, 1e-5, y_norm)
    ya, yb = torch.zeros_like(y_plain), torch.zeros_like(y_plain)
    backend.matmul_many(backend.plan_many([w, w], [x, x], [ya, yb], gammas=[None, gamma], eps=1e-5), M)
    torch.cuda.synchronize()
    assert torch.equal(ya, y_plain) and torch.equal(yb, y_norm)
    lib, ctx = backend._lib, backend._ctx
    import ctypes
    arr = lambda vals: (ctypes.c_void_p * len(vals))(*vals)
    ws, xs, ys = arr([w.handle]), arr([x.data_ptr()]), arr([ya.data_ptr()])
    ya.zero_()
    rc = lib.cybq_matmul_many_norm(ctx, 1, ws, xs, None, 1, ctypes.c_float(1e-5), ys, None, None, 1, M, 0, None)
    torch.cuda.synchronize()
    assert rc == 0 and torch.equal(ya, y_plain)                         # no gamma array at all
    gs = arr([gamma.data_ptr()])
    assert lib.cybq_matmul_many_norm(ctx, 1, ws, xs, gs, 77, ctypes.c_float(1e-5), ys, None, None, 1, M, 0, None) != 0     # unknown gamma type
    assert lib.cybq_matmul_many_norm(ctx, 1, ws, xs, gs, 1, ctypes.c_float(-1.0), ys, None, None, 1, M, 0, None) != 0    # negative eps
    assert lib.cybq_matmul_many_norm(ctx, 1, None, xs, gs, 1, ctypes.c_float(1e-5), ys, None, None, 1, M, 0, None) != 0   # no weights
    assert lib.cybq_matmul_many_norm(ctx, 0, ws, xs, gs, 1, ctypes.c_float(1e-5), ys, None, None, 1, M, 0, None) == 0     # nothing to do


@pytest.mark.parametrize("M", [33, 40, 64])
@pytest.mark.parametrize("xdt", ["f16", "bf16"])
def test_rows_33_to_64_on_a_small_weight_are_two_decode_passes(backend, oracle, M, xdt):
    """33..64 rows of 16-bit activations on a small weight: rows 0..31 carry the bits of a 32-row call,
    the rest those of a call with the remaining rows (a row's bits do not depend on the batch it is in),
    in both prefill modes (prefill EXACT asks the decode kernels for their exact operands), and the
    float64 result within the decode kernels' bar."""
    N, K = 272, 1184
    q, s = _quant(oracle, 4, N, K, cfg=98)
    w = backend.upload_quantized(q, s, 4)
    x = _x(M, K, xdt, cfg=99)
    r = torch.from_numpy(synth.activations(100, M, N)).cuda()
    for mode in ("fast", "exact"):
        backend.set_prefill_mode(mode)
        try:
            y = torch.empty((M, N), dtype=torch.float32, device="cuda")
            backend.matmul_ex(w, x, y, "add", r)
            y_a = torch.empty((32, N), dtype=torch.float32, device="cuda")
            y_b = torch.empty((M - 32, N), dtype=torch.float32, device="cuda")
            backend.set_decode_mode("exact" if mode == "exact" else "stream")
            backend.matmul_ex(w, x[:32].contiguous(), y_a, "add", r[:32].contiguous())
            backend.matmul_ex(w, x[32:].contiguous(), y_b, "add", r[32:].contiguous())
            torch.cuda.synchronize()
            assert torch.equal(y[:32], y_a) and torch.equal(y[32:], y_b)
            ref = oracle.matmul_f64(q, s, x.float().cpu().numpy()) + r.double().cpu().numpy()
            assert oracle.rel_l2(y.cpu().numpy(), ref) < TIGHT
        finally:
            backend.set_prefill_mode("fast")
            backend.set_decode_mode("stream")
    if xdt == "f16":
        # prefill EXACT at these row counts: a tensor of zeros gives exact zeros (the exact integer operands)
        wz = backend.upload_quantized(np.zeros_like(q), s, 4)
        backend.set_prefill_mode("exact")
        try:
            assert not _run(backend, wz, x).any()
        finally:
            backend.set_prefill_mode("fast")
        wz.free()


def _two_passes(backend, w, x):
    return torch.cat([_run(backend, w, x[:32].contiguous()), _run(backend, w, x[32:].contiguous())])


def test_rows_33_to_64_with_a_k_that_the_scratch_does_not_hold(backend):
    """256 staged rows of a K over 251 904 pass the scratch: 33..64 bf16 rows of Q4 stay two decode passes there; just below they are one
    prefill call with exact operands."""
    N, M = 48, 45
    g = torch.Generator(device="cuda").manual_seed(17)
    for K, fits in ((262144 + 32, False), (131072, True)):
        qd = torch.randint(0, 256, (N * K // 2,), dtype=torch.uint8, device="cuda", generator=g)
        sd = (0.01 * torch.rand(N * (K // 32), device="cuda", generator=g)).half().view(torch.int16)
        w = backend.weight_from_device(4, N, K, qd, sd)
        wd = torch.empty((N, K), device="cuda")
        backend.dequant(w, wd)
        x = torch.empty((M, K), device="cuda").normal_(generator=g).bfloat16()
        y = _run(backend, w, x)
        ref = x.double() @ wd.double().t()
        assert ((y.double() - ref).norm() / ref.norm()).item() < TIGHT
        assert torch.equal(y, _two_passes(backend, w, x)) == (not fits)


def test_rows_33_to_64_in_exact_mode_may_be_captured_first(backend):
    """EXACT mode, 33..64 bf16 rows of Q4 on a small weight with a long K: the first call on a weight made from device memory sits in a
    capture, so nothing in it may wait for the scan of the weight's scales."""
    N, K, M = 528, 4640, 45
    g = torch.Generator(device="cuda").manual_seed(18)
    qd = torch.randint(0, 256, (N * K // 2,), dtype=torch.uint8, device="cuda", generator=g)
    sd = (0.01 * torch.rand(N * (K // 32), device="cuda", generator=g)).half().view(torch.int16)
    x = torch.empty((M, K), device="cuda").normal_(generator=g).bfloat16()
    y = torch.zeros((M, N), device="cuda")
    w = backend.weight_from_device(4, N, K, qd, sd)
    torch.cuda.synchronize()
    backend.set_prefill_mode("exact")
    try:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
            backend.matmul(w, x, y, stream=torch.cuda.current_stream().cuda_stream)
        for _ in range(2):
            y.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, _run(backend, w, x))
        wd = torch.empty((N, K), device="cuda")
        backend.dequant(w, wd)
        ref = x.double() @ wd.double().t()
        assert ((y.double() - ref).norm() / ref.norm()).item() < TIGHT
    finally:
        backend.set_prefill_mode("fast")


def _node_reference(oracle, st, node, epi, edges, rows=None):
    """float64 oracle output of one stack node from the PLANAR buffers the stack kept."""
    qd, sd = st.planar[node.w]
    q = formats.unpack_planar(qd.cpu().numpy(), 4, node.N, node.K)
    s = sd.cpu().numpy().view(np.uint16).reshape(node.N, node.K // 32)
    x = edges[node.x] if rows is None else edges[node.x][rows]
    ref = oracle.matmul_f64(q, s, x.float().cpu().numpy())
    if epi == "add":
        r = edges[f"res.{node.N}"] if rows is None else edges[f"res.{node.N}"][rows]
        ref = ref + r.double().cpu().numpy()
    elif epi == "swiglu":
        h = node.N // 2
        ref = _silu_mul(ref[:, :h], ref[:, h:])
    return ref


@pytest.mark.timeout(900)
@pytest.mark.parametrize("form", ["per_linear", "fused", "fused_epilogues"])
def test_config5_full_size_stack(backend, oracle, form):
    """The 32-layer Llama-3-8B-shaped decode step through cybq_matmul_many at full size, batch 1 and 8:
    every node of the first, a middle and the last layer against the oracle; for the fused forms also
    one 512-token bf16 prefill chunk through the same node list."""
    from cyb_amd import stack
    shapes = None if form == "per_linear" else stack.fused_shapes()
    checked = (0, 15, 31)
    st = stack.build(backend, layers=32, seed=5, keep_planar=checked, shapes=shapes,
                     order=list(shapes) if shapes else None, epilogues=form == "fused_epilogues")
    per_layer = len(st.nodes) // 32
    assert per_layer == (7 if shapes is None else 4)
    epis = st.epilogues or ["none"] * len(st.nodes)
    mine = [i for i in range(len(st.nodes)) if i // per_layer in checked]
    for M in (1, 8, 512) if shapes is not None else (1, 8):
        edges = stack.edges_for(st, M, shapes=shapes, xdtype=torch.bfloat16 if M > 16 else None)
        xs, ys = [edges[n.x] for n in st.nodes], [edges[n.y] for n in st.nodes]
        for i in mine:                                  # the checked nodes write buffers of their own
            ys[i] = torch.full_like(ys[i], float("nan"))
        res = None
        if st.epilogues:
            res = [edges[f"res.{n.N}"] if e == "add" else None for n, e in zip(st.nodes, st.epilogues)]
        pl = backend.plan_many(st.weights, xs, ys, st.epilogues or None, res)
        backend.matmul_many(pl, M)
        torch.cuda.synchronize()
        for i in mine:
            node, epi = st.nodes[i], epis[i]
            if M <= 16:
                ref = _node_reference(oracle, st, node, epi, edges)
                assert oracle.rel_l2(ys[i].cpu().numpy(), ref) < TIGHT, (M, node.w, epi)
            else:
                rows = [0, M // 2, M - 1]
                ref = _node_reference(oracle, st, node, epi, edges, rows)
                assert oracle.rel_l2(ys[i][rows].cpu().numpy(), ref) < 2 * FAST, (M, node.w, epi)
                assert torch.isfinite(ys[i]).all()
        if M > 16:
            # every row of the widest and of the longest-K node of the last layer: float64 matmul on the
            # oracle's dequantised weights
            for i in mine[-per_layer:]:
                node, epi = st.nodes[i], epis[i]
                if epi == "swiglu" or node.N * node.K < 4096 * 14336:
                    continue
                qd, sd = st.planar[node.w]
                q = formats.unpack_planar(qd.cpu().numpy(), 4, node.N, node.K)
                s = sd.cpu().numpy().view(np.uint16).reshape(node.N, node.K // 32)
                wd = torch.from_numpy(oracle.dequant(q, s)).cuda().double()
                full = edges[node.x].double() @ wd.T
                if epi == "add":
                    full = full + edges[f"res.{node.N}"].double()
                err = ((ys[i].double() - full).norm() / full.norm()).item()
                assert err < 2 * FAST, (M, node.w, err)
                del wd, full
    assert st.weight_bytes == 32 * 122_683_392
    for w in st.weights:
        w.free()


def test_driver_events_and_rates(backend):
    """The caller loop in the reference's units: event order, token counts, positive rates."""
    from cyb_amd import driver, stack
    shapes = stack.fused_shapes({"q_proj": (512, 512), "k_proj": (512, 128), "v_proj": (512, 128), "o_proj": (512, 512),
                                 "gate_proj": (512, 1792), "up_proj": (512, 1792), "down_proj": (1792, 512)})
    st = stack.build(backend, layers=2, seed=7, shapes=shapes, order=list(shapes))
    evs = list(driver.ask(backend, st, prompt_tokens=300, new_tokens=5, chunk=128, shapes=shapes))
    pre = [e["Prefill"] for e in evs if "Prefill" in e]
    assert [p["done"] for p in pre] == [0, 128, 256, 300] and all(p["total"] == 300 for p in pre)
    assert [e["Delta"] for e in evs if "Delta" in e] == [0, 1, 2, 3, 4]
    ans = evs[-1]["Answer"]
    assert ans.tokens == 5 and ans.tok_in_s > 0 and ans.tok_out_s > 0 and ans.tok_per_s > 0
    # decode only, batch of 4
    evs = list(driver.ask(backend, st, prompt_tokens=0, new_tokens=3, batch=4, shapes=shapes))
    assert evs[-1]["Answer"].tokens == 12 and evs[-1]["Answer"].tok_in_s == 0.0
    with pytest.raises(ValueError):
        list(driver.ask(backend, st, 1, 1, batch=17, shapes=shapes))
    for w in st.weights:
        w.free()


@pytest.mark.parametrize("M,xdt", [(1, "f16"), (8, "f16"), (300, "bf16")])
def test_calls_can_be_captured_in_a_graph(backend, oracle, M, xdt):
    """Every call is a short run of plain kernel launches on the caller's stream (no allocation, no
    memset, no host synchronisation), so a caller may record a step into a HIP graph.  The graph is
    replayed several times with eager work and synchronisations in between, every replay checked
    bit for bit against the eager result (decode kernels; staging pass + multiply + slab adding for
    the prefill shape, whose 4096 columns split K over workgroups)."""
    K1, N1, K2, N2 = 512, 1024, 2048, 4096
    q1, s1 = _quant(oracle, 4, N1, K1, cfg=81)
    q2, s2 = _quant(oracle, 8, N2, K2, cfg=82)
    w1, w2 = backend.upload_quantized(q1, s1, 4), backend.upload_quantized(q2, s2, 8)
    x1, x2 = _x(M, K1, xdt, cfg=83), _x(M, K2, xdt, cfg=84)
    r = torch.from_numpy(synth.activations(85, M, N2)).cuda()
    h = torch.empty((M, N1), dtype=torch.float32, device="cuda")
    y = torch.empty((M, N2), dtype=torch.float32, device="cuda")

    def step(stream):
        backend.matmul(w1, x1, h, stream=stream)
        backend.matmul_ex(w2, x2, y, "add", r, stream=stream)

    step(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    h0, y0 = h.clone(), y.clone()
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        step(torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        h.zero_()
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(h, h0) and torch.equal(y, y0)
        assert (x1.float() @ x1.float().T).sum().isfinite()          # eager work between replays


def test_first_call_of_a_kernel_may_sit_inside_a_capture(oracle):
    """No launch path changes a function attribute (cybq_init raised every kernel's dynamic LDS limit): a
    fresh context may record calls whose kernels it has never launched - kernels that need more than the
    default 64 KB of LDS among them - and the replay matches an eager run made afterwards."""
    from cyb_amd import Backend
    be = Backend(0)
    try:
        be.set_prefill_mode("exact")                       # EXACT prefill tiles stage 112 - 128 KB of operands in LDS
        N, K, M = 208, 2176, 77                            # shapes no other test uses
        q, s = _quant(oracle, 8, N, K, cfg=91)
        qw = be.upload_quantized(q, s, 8, formats.BLOCK_AOS)
        x = _x(M, K, "bf16", cfg=92)
        x32 = _x(12, K, "f32", cfg=93)                     # LDS decode kernel, fp32 rows: its largest LDS request
        y = torch.zeros((M, N), dtype=torch.float32, device="cuda")
        y32 = torch.zeros((12, N), dtype=torch.float32, device="cuda")
        side = torch.cuda.Stream()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            st = torch.cuda.current_stream().cuda_stream
            be.matmul(qw, x, y, stream=st)
            be.matmul(qw, x32, y32, stream=st)
        for _ in range(2):
            y.zero_()
            y32.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert oracle.rel_l2(y.cpu().numpy(), oracle.matmul_f64(q, s, x.float().cpu().numpy())) < TIGHT
            assert oracle.rel_l2(y32.cpu().numpy(), oracle.matmul_f64(q, s, x32.cpu().numpy())) < TIGHT
        ye = torch.zeros_like(y)
        be.matmul(qw, x, ye)
        torch.cuda.synchronize()
        assert torch.equal(ye, y)
        qw.free()
        # FAST mode, 50 rows on a wide output: the kernel whose waves split K (80 KB of LDS for its one exchange)
        be.set_prefill_mode("fast")
        N, K, M = 8192 + 64, 4096 + 128, 50
        q, s = _quant(oracle, 4, N, K, cfg=94)
        qw = be.upload_quantized(q, s, 4)
        x = _x(M, K, "bf16", cfg=95)
        y = torch.zeros((M, N), dtype=torch.float32, device="cuda")
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            be.matmul(qw, x, y, stream=torch.cuda.current_stream().cuda_stream)
        for _ in range(2):
            y.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert oracle.rel_l2(y.cpu().numpy(), oracle.matmul_f64(q, s, x.float().cpu().numpy())) < FAST
        ye = torch.zeros_like(y)
        be.matmul(qw, x, ye)
        torch.cuda.synchronize()
        assert torch.equal(ye, y)
        qw.free()
    finally:
        be.close()


def test_trim_gives_the_memory_of_freed_weights_back(backend):
    """A program that unloads a model and wants the memory for something else gets it: what the library keeps for the
    next tensors is bounded, and cybq_trim hands it to the device."""
    N, K = 16384, 8192                                           # 75.5 MB packed
    qd = torch.zeros(N * K // 2, dtype=torch.uint8, device="cuda")
    sd = torch.zeros(N * (K // 32), dtype=torch.int16, device="cuda")
    torch.cuda.synchronize()
    backend.trim()
    free0 = torch.cuda.mem_get_info()[0]
    ws = [backend.weight_from_device(4, N, K, qd, sd) for _ in range(9)]
    # (the device hands memory out in pages of 2 MiB and more, and part of a tensor may lie in one that was mapped before: eight of
    # the nine are past what the library keeps in any case)
    assert torch.cuda.mem_get_info()[0] <= free0 - 8 * ws[0].device_bytes
    assert 8 * ws[0].device_bytes > 512 << 20
    for w in ws:
        w.free()
    assert torch.cuda.mem_get_info()[0] >= free0 - (512 << 20) - (16 << 20)
    backend.trim()
    assert torch.cuda.mem_get_info()[0] >= free0 - (16 << 20)    # (the runtime's own bookkeeping may move)
    w = backend.weight_from_device(4, N, K, qd, sd)              # and the next tensor is made as ever
    out = torch.full((N, K), 1.0, device="cuda")
    backend.dequant(w, out)
    torch.cuda.synchronize()
    assert not out.any()
    w.free()


@pytest.mark.parametrize("first", ["default", "side"])
@pytest.mark.parametrize("then", ["default", "side", "host"])
def test_a_freed_weight_s_memory_waits_for_the_work_that_reads_it(backend, first, then):
    """A weight is freed while milliseconds of calls that read it are queued, and the next one (made on the same stream, on
    another, or from host memory) gets its memory: the queued calls still see the old tensor, later ones the new one."""
    N, K, calls = 28672, 4096, 300
    packed = []
    for seed in (1, 2):
        g = torch.Generator(device="cuda").manual_seed(seed)
        w = torch.empty((N, K), device="cuda").normal_(0.0, 0.02, generator=g)
        qd = torch.empty(N * K // 2, dtype=torch.uint8, device="cuda")
        sd = torch.empty(N * (K // 32), dtype=torch.int16, device="cuda")
        backend.quantize(4, w, N, K, qd, sd)
        packed.append((qd, sd))
    host = [t.cpu().numpy() for t in packed[1]]
    x = torch.empty((1, K), device="cuda").normal_().to(torch.float16)
    want = []
    for qd, sd in packed:                                        # each tensor alone, nothing shared
        w = backend.weight_from_device(4, N, K, qd, sd)
        want.append(torch.empty((1, N), device="cuda"))
        backend.matmul(w, x, want[-1])
        torch.cuda.synchronize()
        w.free()
        backend.trim()
    y = torch.zeros((calls, N), device="cuda")
    late = torch.zeros((1, N), device="cuda")
    rows = [y[i:i + 1] for i in range(calls)]
    side = [torch.cuda.Stream(), torch.cuda.Stream()]
    st = [0 if s == "default" else side[i].cuda_stream for i, s in enumerate((first, then))]
    torch.cuda.synchronize()
    old = backend.weight_from_device(4, N, K, *packed[0], stream=st[0])
    free1 = torch.cuda.mem_get_info()[0]
    for r in rows:
        backend.matmul(old, x, r, stream=st[0])
    old.free()
    if then == "host":
        new = backend.upload(4, formats.PLANAR, N, K, host[0], host[1].view(np.uint16))
    else:
        new = backend.weight_from_device(4, N, K, *packed[1], stream=st[1])
    backend.matmul(new, x, late, stream=0 if then == "host" else st[1])
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] >= free1 - (32 << 20)    # (no second tensor's worth was allocated)
    assert torch.equal(y, want[0].expand(calls, N))
    assert torch.equal(late, want[1])
    new.free()


def test_upload_of_a_list_that_fails_half_way_leaves_nothing(backend):
    """The second tensor of the list asks for more memory than any device has (its source is never read): the first one's memory
    comes back, no handle is left, and the library goes on."""
    import ctypes
    N, K = 1024, 4096
    blocks = np.zeros(N * (K // 32) * 18, np.uint8)
    backend.trim()
    free0 = torch.cuda.mem_get_info()[0]
    two = lambda t, *v: (t * 2)(*v)
    out = two(ctypes.c_void_p, 1, 1)
    rc = backend._lib.cybq_weight_upload_many(backend._ctx, 2, two(ctypes.c_int, 4, 4), two(ctypes.c_int, 1, 1), two(ctypes.c_int64, N, 1 << 20),
                                              two(ctypes.c_int64, K, 1 << 20), two(ctypes.c_void_p, blocks.ctypes.data, blocks.ctypes.data), None, out)
    assert rc == -6 and not out[0] and not out[1]
    backend.trim()
    assert torch.cuda.mem_get_info()[0] >= free0 - (1 << 20)
    w = backend.upload(4, formats.BLOCK_AOS, N, K, blocks)
    y = torch.ones((N, K), device="cuda")
    backend.dequant(w, y)
    torch.cuda.synchronize()
    assert not y.any()
    w.free()


def test_a_weight_is_not_made_on_a_capturing_stream(backend):
    """Also where nothing has to be allocated for it (the memory and the scan word of a weight freed before): the recorded repack
    would not have run when the call returns.  The capture goes on, and the first prefill call of a weight made outside of it may
    sit inside."""
    N, K, M = 1024, 2048, 100
    w = torch.empty((N, K), device="cuda").normal_(0.0, 0.02)
    qd = torch.empty(N * K // 2, dtype=torch.uint8, device="cuda")
    sd = torch.empty(N * (K // 32), dtype=torch.int16, device="cuda")
    backend.quantize(4, w, N, K, qd, sd)
    qw = backend.weight_from_device(4, N, K, qd, sd)
    backend.weight_from_device(4, N, K, qd, sd).free()
    x = torch.empty((M, K), device="cuda").normal_().to(torch.bfloat16)
    y, want = torch.zeros((M, N), device="cuda"), torch.zeros((M, N), device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        st = torch.cuda.current_stream().cuda_stream
        with pytest.raises(CybqError) as err:
            backend.weight_from_device(4, N, K, qd, sd, stream=st)
        assert err.value.status == -7
        backend.matmul(qw, x, y, stream=st)
    backend.matmul(qw, x, want)
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
    again = backend.weight_from_device(4, N, K, qd, sd)          # (and nothing was left behind by the refusal)
    backend.matmul(again, x, y)
    torch.cuda.synchronize()
    assert torch.equal(y, want)
    again.free()
    qw.free()


def test_read_pattern_probes_run(backend, oracle):
    """The pure-read probes the benchmark records as ceilings: every pattern runs on the headline tensor's
    K and on a ragged tensor (flat patterns), and the strip patterns refuse shapes they do not cover."""
    q, s = _quant(oracle, 4, 272, 4096, cfg=61)
    w = backend.upload_quantized(q, s, 4)
    q2, s2 = _quant(oracle, 8, 40, 416, cfg=62)
    w2 = backend.upload_quantized(q2, s2, 8)
    xd = torch.zeros(8, dtype=torch.float16, device="cuda")            # (a plan wants edges; the probes read none)
    yd = torch.zeros(8, dtype=torch.float32, device="cuda")
    plan = backend.plan_many([w, w], [xd, xd], [yd, yd])
    plan2 = backend.plan_many([w2], [xd], [yd])
    for pattern in range(1, 7):
        backend.debug_read_pattern(plan, pattern)
    for pattern in (3, 4, 5, 6):
        backend.debug_read_pattern(plan2, pattern)
    torch.cuda.synchronize()
    for pattern in (1, 2, 0, 7):
        with pytest.raises(CybqError) as e:
            backend.debug_read_pattern(plan2, pattern)
        assert e.value.status == -7
    w.free()
    w2.free()


def test_container_to_backend(backend, oracle, tmp_path):
    from cyb_amd import container
    q, s = _quant(oracle, 4, 64, 256)
    path = str(tmp_path / "one.model")
    container.write_container(path, "one", "", [container.tensor_entry("lm_head.weight", q, s, 4, formats.BLOCK_AOS)])
    recs = container.load_into(backend, path)
    assert [r.name for r in recs] == ["lm_head.weight"]
    x = _x(3, 256, "f16")
    y = torch.empty((3, 64), dtype=torch.float32, device="cuda")
    backend.run(QMatMul(w="lm_head.weight", x="x", y="y", quant=4, M=3, N=64, K=256), {"x": x, "y": y})
    torch.cuda.synchronize()
    assert oracle.rel_l2(y.cpu().numpy(), oracle.matmul_f64(q, s, x.float().cpu().numpy())) < TIGHT
