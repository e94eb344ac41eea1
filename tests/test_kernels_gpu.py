"""Each kernel alone against a plain float32 PyTorch reference of the same operation, at sizes
other than the engine's tiny models use (sizes that are no power of two, several head sizes)."""
import math

import numpy as np
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DT = [torch.float32, torch.bfloat16]


def rnd(*shape, dtype=torch.float32, scale=1.0, seed=0):
    g = torch.Generator(device="cpu").manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


def i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


def close(got, want, dtype, what="", f32=1e-5, bf16=1.2e-2):
    got, want = got.float().cpu(), want.float().cpu()
    tol = f32 if dtype == torch.float32 else bf16
    scale = want.abs().max().item() + 1e-30
    err = (got - want).abs().max().item()
    assert err <= tol * scale, f"{what}: error {err:.3e} > {tol} x {scale:.3e}"


@pytest.mark.parametrize("table_dtype", DT)
def test_embed(table_dtype):
    from gibbs_amd import ops
    table = rnd(331, 72, dtype=table_dtype)
    ids = i32([0, 330, 5, 5, 17])
    out = ops.embed(table, ids, 5)
    assert out.dtype == torch.float32
    assert torch.equal(out, table.float()[ids.long()])


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("hidden", [48, 70, 200, 2048, 5000, 20000])   # 70 and 20000: the element-wise kernel
def test_add_rmsnorm(dtype, hidden):
    from gibbs_amd import ops
    x = rnd(7, hidden, scale=3.0)
    delta = rnd(7, hidden, dtype=dtype, seed=1)
    gain = rnd(hidden, seed=2) + 1.0
    x0 = x.clone()
    out = ops.add_rmsnorm(x, delta, gain, 1e-6, dtype)
    v = x0 + delta.float()
    assert torch.equal(x, v), "the residual stream must hold x + delta exactly"
    want = F.rms_norm(v.double(), (hidden,), gain.double(), eps=1e-6)
    close(out, want, dtype, "add_rmsnorm")
    # without delta; and on chosen rows only (x untouched)
    out2 = ops.add_rmsnorm(x, None, gain, 1e-6, dtype)
    close(out2, want, dtype, "rmsnorm")
    rows = i32([6, 0, 3])
    x1 = x.clone()
    out3 = ops.add_rmsnorm(x, delta, gain, 1e-6, dtype, rows)
    assert torch.equal(x, x1)
    want3 = F.rms_norm((x1 + delta.float())[rows.long()].double(), (hidden,), gain.double(), eps=1e-6)
    close(out3, want3, dtype, "rmsnorm rows")


@pytest.mark.parametrize("shape", [(1, 64, 32), (5, 331, 112), (130, 200, 72), (257, 129, 1000)])
def test_gemm_f32(shape):
    from gibbs_amd import ops
    n, o, i = shape
    a, w = rnd(n, i), rnd(o, i, seed=1)
    close(ops.gemm_f32(a, w), a.double() @ w.double().t(), torch.float32, f"gemm_f32 {shape}")
    # a row's result does not depend on the other rows of the call
    assert torch.equal(ops.gemm_f32(a[:1].contiguous(), w), ops.gemm_f32(a, w)[:1])


@pytest.mark.parametrize("shape", [(1, 1, 4), (17, 33, 516), (33, 65, 1000), (31, 50, 28), (129, 255, 4608), (200, 96, 520),
                                   (65, 130, 2052), (300, 1024, 1024), (1100, 2112, 512)])
def test_gemm_f32_tiles_and_stretches(shape):
    """Every tile of the 32-bit product at remainders of rows, features and k: the error of a sum of k products in 32 bits is at most
    k 2^-24 of the sum of their magnitudes, and a row's result is the same to the bit in whatever tile it is computed."""
    from gibbs_amd import ops
    n, o, i = shape
    a, w = rnd(n, i), rnd(o, i, seed=1)
    want, scale = a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()
    out = ops.gemm_f32(a, w)
    assert ((out.double() - want).abs() <= i * 2.0 ** -24 * scale).all(), shape
    for m in (1, 16, 17, 33, 97):
        if m < n:
            assert torch.equal(ops.gemm_f32(a[:m].contiguous(), w), out[:m]), (shape, m)


@pytest.mark.parametrize("shape", [(5, 96, 512), (40, 1000, 516), (200, 2112, 100), (700, 2112, 512)])
def test_gemm_f32_values_without_three_bfloat16_parts(shape):
    """Infinities, NaN, values that round up to infinity and values whose low parts bfloat16 does not hold come out as in plain float32: which
    results are infinite or NaN is the inputs' affair, and the others keep the error of a sum in 32 bits (of results that float32 holds
    with fewer digits: 2^-149 a product)."""
    from gibbs_amd import ops
    n, o, i = shape
    w = rnd(o, i, seed=1)
    for size in (1e-36, 1e-30, 1e-20, 1.0, 1e15):
        a = rnd(n, i) * size
        want, scale = a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()
        assert ((ops.gemm_f32(a, w).double() - want).abs() <= i * (2.0 ** -24 * scale + 2.0 ** -149)).all(), (shape, size)
    a = rnd(n, i)
    a[0, 7], a[2, 9], a[3, i - 1], a[n - 1, 0] = float("inf"), float("nan"), 3.4e38, -float("inf")
    w[o // 2, 5] = float("inf")
    w[o - 1, i - 1] = 0.0            # (0 times an infinity or times what rounds up to one)
    got, want = ops.gemm_f32(a, w), a.double() @ w.double().t()
    assert torch.equal(got.isnan(), want.isnan())
    big = want.abs() > 3.5e38
    assert torch.equal(got[big], want[big].float())
    assert got[~big & ~want.isnan() & (want.abs() < 3.3e38)].isfinite().all()


@pytest.mark.parametrize("shape", [(5, 96, 512), (40, 1000, 516), (200, 2112, 100), (70, 48, 4), (700, 2112, 512)])
def test_gemm_f32_keeps_the_digits_of_small_operands(shape):
    """Operands with bits under 2^-133, which three bfloat16 do not hold, against operands large enough that the results are ordinary, from either side, in
    single rows and in single columns.  An error of I additions, each of at most 2^-24 of a partial sum that is no larger than the whole in the root mean
    square, is 2^-24 sqrt(I) of the whole, row by row (three products instead of six are at 4e-6, parts without these digits up to 2e-2), and 2^-149
    a product where float32 ends.  A row's bits are its own, in whatever company and kernel."""
    from gibbs_amd import ops
    n, o, i = shape
    a0, w0 = rnd(n, i), rnd(o, i, seed=1)
    def check(a, w, what):
        got = ops.gemm_f32(a, w)
        want = a.double() @ w.double().t()
        bound = 2.0 ** -24 * (1 + i ** 0.5) * want.norm(dim=1) + i * 2.0 ** -149 * o ** 0.5
        err = (got.double() - want).norm(dim=1)
        assert (err <= bound).all(), (shape, what, float((err / want.norm(dim=1)).max()))
        for m in (1, 17, 70):
            if m < n:
                assert torch.equal(ops.gemm_f32(a[:m].contiguous(), w), got[:m]), (shape, what, m)
        return got
    for small, large in ((-107, 20), (-112, 0), (-120, 27), (-124, 30), (-124, 124), (-130, 40), (-140, 60), (-70, -66)):
        check(a0 * 2.0 ** small, w0 * 2.0 ** large, (small, large))
        check(a0 * 2.0 ** large, w0 * 2.0 ** small, (large, small))
    plain = ops.gemm_f32(a0, w0)
    a = a0.clone()
    a[n // 2] *= 2.0 ** -125
    got = check(a, w0, "a small row")
    keep = torch.arange(n, device="cuda") != n // 2
    assert torch.equal(got[keep], plain[keep])
    w = w0.clone()
    w[o // 3] *= 2.0 ** -125
    got = check(a0, w, "a small feature")
    keep = torch.arange(o, device="cuda") != o // 3
    assert torch.equal(got[:, keep], plain[:, keep])
    a, w = a0 * 2.0 ** -10, w0.clone()
    a[:, i // 2], w[:, i // 2] = a0[:, i // 2] * 2.0 ** -123, w0[:, i // 2] * 2.0 ** 124
    check(a, w, "small values that count")


@pytest.mark.parametrize("shape", [(333, 1000, 2052), (270, 1024, 4608), (450, 640, 3000), (700, 500, 2080)])
def test_gemm_f32_stretches_shared_between_workgroups(shape):
    """Few tiles of a long inner size share the chip through a workspace: the bits of the product without one, for ordinary values and for
    rows whose results are taken again (infinities, NaN, digits that three bfloat16 do not hold, in a stretch of any of a tile's workgroups)."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import library
    n, o, i = shape
    assert library().gibbs_gemm_f32_workspace(n, o, i) > 0
    a, w = rnd(n, i, seed=1), rnd(o, i, seed=2)
    want = ops.gemm_f32(a, w, workspace=False)
    assert torch.equal(ops.gemm_f32(a, w), want)
    a[0, 7], a[n // 2, i - 1], a[n - 1, i // 2], w[o // 3, 5] = float("inf"), float("nan"), 3.4e38, -float("inf")
    a[1, i - 2], a[70, 3], w[o - 1, i // 3] = 2.0 ** -124, 2.0 ** -130, 2.0 ** -120
    a[5] *= 2.0 ** -118
    bits = [ops.gemm_f32(a, w, workspace=k).view(torch.int32) for k in (False, True)]
    assert torch.equal(*bits)
    assert not torch.equal(bits[0].view(torch.float32), want)


# (stretches of a workgroup: 3 to 7, which no tile's 8 are a multiple of)
@pytest.mark.parametrize("shape,run", [((700, 1000, 4608), 3), ((1000, 1040, 2052), 5), ((1194, 1000, 2052), 5), ((1500, 1000, 2080), 6), ((1590, 1000, 4608), 7)])
def test_gemm_f32_workgroups_that_go_on_to_the_next_tile(shape, run):
    """A workgroup's run of stretches that ends one tile and begins the next: the bits of a workgroup a tile, for ordinary values and with
    infinities, NaN and lost digits in rows of every tile, in stretches on both sides of wherever a tile is cut."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import library
    n, o, i = shape
    assert library().gibbs_gemm_f32_workspace(n, o, i) > 0
    rows, cols = -(-n // 64), -(-o // 128)
    assert run == max(2, -(-rows * cols * 8 // 256)) and 8 % run
    a, w = rnd(n, i, seed=1), rnd(o, i, seed=2)
    want = ops.gemm_f32(a, w, workspace=False)
    assert torch.equal(ops.gemm_f32(a, w), want)
    segment = -(-(-(-i // 8)) // 32) * 32
    for t in range(rows):      # (tile t of rows: its special values in other stretches than its neighbours')
        def put(row, stretch, v):
            a[min(64 * t + row, n - 1), min(stretch % 8 * segment + 5 + row, i - 1)] = v
        put(3, t, 2.0 ** -124)
        put(17, t + 7, float("inf"))
        put(40, t + 4, float("nan"))
        put(63, 3 * t + 1, 2.0 ** -130)
    for t in range(cols):
        w[min(128 * t + 9, o - 1), t % 8 * segment + 3] = 2.0 ** -121
        w[min(128 * t + 100, o - 1), (t + 5) % 8 * segment + 1] = -float("inf")
    bits = [ops.gemm_f32(a, w, workspace=k).view(torch.int32) for k in (False, True)]
    assert torch.equal(*bits)
    assert not torch.equal(bits[0].view(torch.float32), want)


def test_gemm_f32_as_many_rows_as_the_plain_kernel_takes():
    """4,194,240 rows, which is where the plain kernel's grid ends, of few features: the tiles that cut k over their waves have no grid for them."""
    from gibbs_amd import ops
    n, o, i = 65535 * 64, 5, 4
    a, w = rnd(n, i), rnd(o, i, seed=1)
    out, want, scale = ops.gemm_f32(a, w), a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()
    assert ((out.double() - want).abs() <= i * 2.0 ** -24 * scale).all()


@pytest.mark.parametrize("out_dtype", DT)
@pytest.mark.parametrize("shape", [(1, 64, 32), (5, 331, 112), (130, 200, 72), (257, 129, 1000), (300, 512, 2048),
                                   (2048, 6144, 192), (1024, 12288, 64), (768, 16384, 320)])   # the 256 x 256 kernel: both tile orders
def test_gemm_bf16(shape, out_dtype):
    from gibbs_amd import ops
    n, o, i = shape
    a, w = rnd(n, i, dtype=torch.bfloat16), rnd(o, i, dtype=torch.bfloat16, seed=1)
    want = a.double() @ w.double().t()
    got = ops.gemm_bf16(a, w, out_dtype)
    assert got.dtype == out_dtype
    # float32 output: only the accumulation order differs from the exact product
    close(got, want, out_dtype, f"gemm_bf16 {shape}", f32=2e-5, bf16=4e-3)
    # a view with a row stride (the q part of a fused projection)
    big = rnd(n, i + 64, dtype=torch.bfloat16, seed=3)
    close(ops.gemm_bf16(big[:, :i], w, out_dtype), big[:, :i].double() @ w.double().t(), out_dtype, "strided", f32=2e-5, bf16=4e-3)


@pytest.mark.parametrize("shape", [(65, 64, 32), (130, 200, 72), (257, 129, 1000), (512, 6144, 2048), (2048, 2048, 512)])
def test_gemm_library(shape):
    """The library's product called directly (descriptors and algorithm kept per shape), also on a
    view with a row stride and into a strided output, and twice (the second call takes the kept plan)."""
    from gibbs_amd import ops
    n, o, i = shape
    a, w = rnd(n, i, dtype=torch.bfloat16), rnd(o, i, dtype=torch.bfloat16, seed=1)
    want = a.double() @ w.double().t()
    for _ in range(2):
        close(ops.gemm_library(a, w), want, torch.bfloat16, f"gemm_library {shape}", bf16=4e-3)
    big = rnd(n, i + 64, dtype=torch.bfloat16, seed=3)
    close(ops.gemm_library(big[:, :i], w), big[:, :i].double() @ w.double().t(), torch.bfloat16, "strided input", bf16=4e-3)
    wide = torch.zeros(n, o + 16, dtype=torch.bfloat16, device=DEV)
    ops.gemm_library(a, w, out=wide[:, :o])
    close(wide[:, :o], want, torch.bfloat16, "strided output", bf16=4e-3)
    assert float(wide[:, o:].abs().max()) == 0.0


@pytest.mark.parametrize("out_dtype", DT)
@pytest.mark.parametrize("n,o,i,splits", [(1, 64, 128, 1), (8, 331, 1000, 1), (16, 2048, 2048, 2), (17, 200, 8192, 8),
                                          (33, 48, 72, 1), (64, 515, 1024, 1), (5, 2048, 8192, 4), (64, 96, 4096, 3),
                                          (64, 2048, 2048, 8), (40, 8200, 512, 1), (50, 1000, 4096, 16)])   # 4 tiles a workgroup
def test_gemm_skinny(n, o, i, splits, out_dtype):
    from gibbs_amd import ops
    x, w = rnd(n, i, dtype=torch.bfloat16), rnd(o, i, dtype=torch.bfloat16, seed=1)
    want = x.double() @ w.double().t()
    if splits > 1 and out_dtype == torch.float32:          # partial sums are float32
        parts = ops.gemm_skinny(x, w, torch.float32, splits)
        assert parts.shape == (splits, n, o)
        close(parts.sum(0), want, torch.float32, "skinny partial sums", f32=2e-5)
    got = ops.gemm_skinny(x, w, out_dtype)
    assert got.dtype == out_dtype and got.shape == (n, o)
    close(got, want, out_dtype, f"gemm_skinny {(n, o, i)}", f32=2e-5, bf16=4e-3)
    # a strided view of x (rows of a wider buffer)
    big = rnd(n, i + 64, dtype=torch.bfloat16, seed=3)
    close(ops.gemm_skinny(big[:, :i], w, out_dtype), big[:, :i].double() @ w.double().t(), out_dtype, "strided",
          f32=2e-5, bf16=4e-3)


def test_packed_weight_layout():
    """Many rows: [group][16-row tile][32-k tile][lane = g * 16 + r][8]; few rows (workgroups of 8 features):
    [group][8-row tile][pair of k tiles][g][half][r8][8]; zeros beyond the matrix."""
    from gibbs_amd import ops
    rows = 4104                                             # 257 tiles of 16
    assert not ops.pair_layout(rows) and not ops.pair_layout(4081) and ops.pair_layout(4080) and ops.pair_layout(40)
    w = rnd(2 * rows, 72, dtype=torch.bfloat16)
    p = ops.PackedWeight(w, groups=2)
    assert p.shape == (2 * rows, 72) and p.stride(0) == 0 and tuple(p.data.shape) == (2, 257, 3, 4, 16, 8) and not p.pairs
    for q, ot, kt, g, r in [(0, 0, 0, 0, 0), (1, 2, 1, 3, 7), (0, 256, 2, 0, 15), (1, 256, 2, 1, 3), (1, 256, 0, 2, 8)]:
        row, k = ot * 16 + r, kt * 32 + g * 8
        want = torch.zeros(8, dtype=torch.bfloat16, device=DEV)
        if row < rows and k < 72:
            want[:min(8, 72 - k)] = w[q * rows + row, k:k + 8]
        assert torch.equal(p.data[q, ot, kt, g, r], want), (q, ot, kt, g, r)
    w = rnd(2 * 40, 72, dtype=torch.bfloat16)
    p = ops.PackedWeight(w, groups=2)
    assert p.shape == (80, 72) and p.stride(0) == 0 and tuple(p.data.shape) == (2, 6, 2, 4, 2, 8, 8) and p.pairs
    for q, o8, pair, g, half, r8 in [(0, 0, 0, 0, 0, 0), (1, 4, 1, 0, 0, 7), (0, 2, 1, 1, 1, 5), (1, 5, 0, 3, 1, 3), (0, 4, 0, 2, 1, 7)]:
        row, k = o8 * 8 + r8, pair * 64 + half * 32 + g * 8
        want = torch.zeros(8, dtype=torch.bfloat16, device=DEV)
        if row < 40 and k < 72:
            want[:min(8, 72 - k)] = w[q * 40 + row, k:k + 8]
        assert torch.equal(p.data[q, o8, pair, g, half, r8], want), (q, o8, pair, g, half, r8)
    x = rnd(5, 72, dtype=torch.bfloat16, seed=2)
    for splits in (1, 2):
        w1 = rnd(50, 256, dtype=torch.bfloat16, seed=3)
        x1 = rnd(5, 256, dtype=torch.bfloat16, seed=4)
        assert torch.equal(ops.gemm_skinny(x1, ops.PackedWeight(w1), torch.float32, splits), ops.gemm_skinny(x1, w1, torch.float32, splits))
        w2 = rnd(4200, 256, dtype=torch.bfloat16, seed=5)                    # 16-row tiles
        assert torch.equal(ops.gemm_skinny(x1, ops.PackedWeight(w2), torch.float32, splits), ops.gemm_skinny(x1, w2, torch.float32, splits))


def test_skinny_splits_cover_k():
    from gibbs_amd import ops
    for o, i in [(2048, 2048), (2048, 8192), (6144, 2048), (65536, 2048), (96, 96), (200, 1000), (64, 12800)]:
        s = ops.skinny_splits(o, i)
        per = -(-(-(-i // s)) // 128) * 128
        assert s >= 1 and -(-i // per) == s, (o, i, s)
        x, w = rnd(3, i, dtype=torch.bfloat16), rnd(min(o, 64), i, dtype=torch.bfloat16, seed=1)
        parts = ops.gemm_skinny(x, w, torch.float32, s)
        got = parts.sum(0) if s > 1 else parts
        close(got, x.double() @ w.double().t(), torch.float32, f"splits {s}", f32=2e-5)


@pytest.mark.parametrize("dtype", DT)
def test_add_partials_rmsnorm(dtype):
    from gibbs_amd import ops
    hidden, n, s = 200, 5, 3
    x = rnd(n, hidden, scale=2.0)
    parts = rnd(s, n, hidden, seed=4)
    gain = rnd(hidden, seed=2) + 1.0
    x0 = x.clone()
    out = ops.add_rmsnorm(x, parts, gain, 1e-6, dtype)
    v = x0 + (parts[0] + parts[1]) + parts[2]
    close(x, v, torch.float32, "x + partials", f32=1e-6)
    close(out, F.rms_norm(v.double(), (hidden,), gain.double(), eps=1e-6), dtype, "partials rmsnorm")
    rows = i32([4, 1])
    x1 = x.clone()
    out2 = ops.add_rmsnorm(x, parts, gain, 1e-6, dtype, rows)
    assert torch.equal(x, x1)
    close(out2, F.rms_norm((x1 + parts.sum(0))[rows.long()].double(), (hidden,), gain.double(), eps=1e-6), dtype, "rows")


def test_gemm_bf16_refuses_unaligned():
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import KernelError
    with pytest.raises(KernelError, match="multiples of 8"):
        ops.gemm_bf16(rnd(3, 20, dtype=torch.bfloat16), rnd(4, 20, dtype=torch.bfloat16))


@pytest.mark.parametrize("dtype", DT)
def test_glu(dtype):
    from gibbs_amd import ops
    gu = rnd(9, 2 * 200, dtype=dtype, scale=2.0)
    want = F.silu(gu.double()[:, :200]) * gu.double()[:, 200:]
    close(ops.glu(gu), want, dtype, "glu")
    one = torch.tensor([[0.0, 2.0, 1.0, 3.0]], device=DEV)              # silu(0)*1 = 0, silu(2)*3
    out = ops.glu(one)
    assert out[0, 0].item() == 0.0 and abs(out[0, 1].item() - 2 / (1 + math.exp(-2)) * 3) < 1e-6


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("K,C,bias", [(3, 40, False), (4, 300, True), (2, 72, True), (7, 16, False)])
def test_shortconv_ragged_with_state(dtype, K, C, bias):
    """Three requests in one call: a fresh one, one with history shorter than K-1 before this chunk,
    one decoding a single token; against conv1d over each whole sequence."""
    from gibbs_amd import ops
    taps = rnd(C, K, seed=4)
    b = rnd(C, seed=5) if bias else None
    lens_before, lens_now = [0, 1, 9], [6, 2, 1]
    slots = [2, 0, 3]
    seqs = [rnd(lb + ln, 3 * C, dtype=dtype, seed=10 + i) for i, (lb, ln) in enumerate(zip(lens_before, lens_now))]
    state = torch.full((4, K - 1, C), 7.0, device=DEV)                   # stale content of a reused slot
    def reference(seq):
        s = seq.double()
        bx = s[:, :C] * s[:, 2 * C:]
        cv = F.conv1d(bx.t()[None], taps.double()[:, None, :], None if b is None else b.double(), groups=C,
                      padding=K - 1)[0, :, :seq.shape[0]].t()
        return s[:, C:2 * C] * cv, bx
    # first call: the histories (requests 1 and 2 only)
    cu = i32([0, lens_before[1], lens_before[1] + lens_before[2]])
    hist = torch.cat([seqs[1][:lens_before[1]], seqs[2][:lens_before[2]]])
    ops.shortconv(hist, taps, b, state, cu, i32([0, 0]), i32(slots[1:]), hist.shape[0], 2)
    # second call: all three together
    now = torch.cat([s[lb:] for s, lb in zip(seqs, lens_before)])
    cu = i32(np.concatenate([[0], np.cumsum(lens_now)]))
    y = ops.shortconv(now, taps, b, state, cu, i32(lens_before), i32(slots), now.shape[0], 3)
    at = 0
    for seq, lb, ln, slot in zip(seqs, lens_before, lens_now, slots):
        want, bx = reference(seq)
        close(y[at:at + ln], want[lb:], dtype, f"shortconv rows K={K}")
        at += ln
        full = torch.cat([torch.zeros(K - 1, C, device=DEV, dtype=torch.float64), bx])
        close(state[slot], full[-(K - 1):], torch.float32, "state", f32=1e-6)
    assert torch.all(state[1] == 7.0), "a slot of no request was written"

@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("C,over", [(64, 1), (1024, 1), (1024, 5)])
def test_shortconv_tiles_of_few_and_of_many_rows(dtype, C, over):
    """Where rows stop being few (4 MB of values): the rows of a request are to the bit those of the same request a few rows longer, and its state that of
    the same rows brought by two calls."""
    from gibbs_amd import ops
    line = (1 << (20 if dtype == torch.float32 else 21)) // C
    taps, x = rnd(C, 3, seed=4), rnd(line + over, 3 * C, dtype=dtype, seed=5)
    def run(*cuts):
        state, rows, at = torch.full((1, 2, C), 7.0, device=DEV), [], 0
        for cut in cuts:
            rows.append(ops.shortconv(x[at:cut].contiguous(), taps, None, state, i32([0, cut - at]), i32([at]), i32([0]), cut - at, 1))
            at = cut
        return torch.cat(rows), state
    few, few_state = run(line)
    many, many_state = run(line + over)
    rest, rest_state = run(line, line + over)
    assert torch.equal(few, many[:line]) and torch.equal(rest, many) and torch.equal(rest_state, many_state)
    assert torch.equal(few_state[0], (x[line - 2:line, :C].float() * x[line - 2:line, 2 * C:].float()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C", [24, 520])
@pytest.mark.parametrize("lens_now", [[1, 1, 1, 1, 1], [1, 1, 1, 40, 2], [1, 1, 70, 1, 1]])
def test_shortconv_decoded_rows_at_the_head(dtype, C, lens_now):
    """Requests that bring one row each at the head of the batch (decoded tokens) are found by their tile's number,
    the others by a walk over the requests behind them: the same result whatever the caller says about the head
    (nothing, its true length, less), and against conv1d over each whole sequence."""
    from gibbs_amd import ops
    K = 3
    taps, b = rnd(C, K, seed=4), rnd(C, seed=5)
    lens_before = [9, 1, 3, 0, 5]
    slots = [4, 0, 3, 1, 5]
    seqs = [rnd(lb + ln, 3 * C, dtype=dtype, seed=20 + i) for i, (lb, ln) in enumerate(zip(lens_before, lens_now))]
    lead = next((i for i, n in enumerate(lens_now) if n != 1), len(lens_now))
    results = []
    for say in (None, lead, max(lead - 1, 0), 0):
        state = torch.full((6, K - 1, C), 7.0, device=DEV)
        with_history = [i for i, lb in enumerate(lens_before) if lb]
        hist = torch.cat([seqs[i][:lens_before[i]] for i in with_history])
        cu = i32(np.concatenate([[0], np.cumsum([lens_before[i] for i in with_history])]))
        ops.shortconv(hist, taps, b, state, cu, i32([0] * len(with_history)), i32([slots[i] for i in with_history]),
                      hist.shape[0], len(with_history))
        now = torch.cat([s[lb:] for s, lb in zip(seqs, lens_before)])
        cu = i32(np.concatenate([[0], np.cumsum(lens_now)]))
        y = ops.shortconv(now, taps, b, state, cu, i32(lens_before), i32(slots), now.shape[0], len(lens_now), lead_single=say)
        results.append((y, state))
    for y, state in results[1:]:
        assert torch.equal(y, results[0][0]) and torch.equal(state, results[0][1])
    y, state = results[0]
    at = 0
    for seq, lb, ln, slot in zip(seqs, lens_before, lens_now, slots):
        s = seq.double()
        bx = s[:, :C] * s[:, 2 * C:]
        cv = F.conv1d(bx.t()[None], taps.double()[:, None, :], b.double(), groups=C, padding=K - 1)[0, :, :seq.shape[0]].t()
        close(y[at:at + ln], (s[:, C:2 * C] * cv)[lb:], dtype, "shortconv rows")
        at += ln
        full = torch.cat([torch.zeros(K - 1, C, device=DEV, dtype=torch.float64), bx])
        close(state[slot], full[-(K - 1):], torch.float32, "state", f32=1e-6)
    assert torch.all(state[2] == 7.0), "a slot of no request was written"
    with pytest.raises(ops.KernelError, match="leading single rows"):
        ops.shortconv(now, taps, b, state, cu, i32(lens_before), i32(slots), now.shape[0], len(lens_now), lead_single=6)


def paged_setup(dtype, nkv, hd, page_size, seq_lens, num_pages, seed=0):
    """Random keys and values of several requests scattered over shuffled pages (the rest of the
    pool holds large garbage)."""
    rng = np.random.default_rng(seed)
    kp = torch.full((num_pages, nkv, page_size, hd), 50.0, dtype=dtype, device=DEV)
    vp = torch.full((num_pages, nkv, page_size, hd), -50.0, dtype=dtype, device=DEV)
    free = rng.permutation(num_pages).tolist()
    width = max(-(-l // page_size) for l in seq_lens)
    table = np.full((len(seq_lens), width), -1, dtype=np.int32)
    ks, vs = [], []
    for r, l in enumerate(seq_lens):
        k, v = rnd(l, nkv, hd, dtype=dtype, seed=seed + 2 * r), rnd(l, nkv, hd, dtype=dtype, seed=seed + 2 * r + 1)
        ks.append(k); vs.append(v)
        for j in range(-(-l // page_size)):
            p = free.pop()
            table[r, j] = p
            n = min(page_size, l - j * page_size)
            kp[p, :, :n] = k[j * page_size:j * page_size + n].transpose(0, 1)
            vp[p, :, :n] = v[j * page_size:j * page_size + n].transpose(0, 1)
    return kp, vp, i32(table), ks, vs


def attention_reference(q, k, v, positions, scale, window):
    """q: [n, nh, hd] rows at `positions` of one request with keys k, v: [L, nkv, hd]."""
    nh, nkv = q.shape[1], k.shape[1]
    kk, vv = k.double().repeat_interleave(nh // nkv, 1), v.double().repeat_interleave(nh // nkv, 1)
    out = torch.zeros(q.shape, dtype=torch.float64, device=q.device)
    for i, p in enumerate(positions):
        lo = 0 if not window else max(0, p - window + 1)
        s = torch.einsum("hd,lhd->hl", q[i].double(), kk[lo:p + 1]) * scale
        out[i] = torch.einsum("hl,lhd->hd", s.softmax(-1), vv[lo:p + 1])
    return out


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("nh,nkv,hd,page,window", [(4, 2, 16, 16, None), (6, 1, 48, 8, None), (5, 5, 80, 32, 37),
                                                   (8, 2, 128, 16, None), (2, 2, 256, 64, 100)])
def test_attention_plain_paged(dtype, nh, nkv, hd, page, window):
    from gibbs_amd import ops
    seq_lens = [150, 3, 77]
    kp, vp, table, ks, vs = paged_setup(dtype, nkv, hd, page, seq_lens, 40)
    # request 0: a portion of 20 rows ending at its last key; request 1: all 3 rows; request 2: one decoded row
    rows = [(0, list(range(130, 150))), (1, [0, 1, 2]), (2, [76])]
    pos = i32([p for _, ps in rows for p in ps])
    row_req = i32([r for r, ps in rows for _ in ps])
    n = pos.numel()
    q = rnd(n, nh * hd, dtype=dtype, seed=9)
    scale = 1 / math.sqrt(hd)
    out = ops.attention_plain(q, n, nh, nkv, hd, kp, vp, table, 3, pos, row_req, scale, window)
    at = 0
    for r, ps in rows:
        want = attention_reference(q[at:at + len(ps)].view(-1, nh, hd), ks[r], vs[r], ps, scale, window)
        close(out[at:at + len(ps)].view(-1, nh, hd), want, dtype, f"attention request {r}", f32=2e-5, bf16=1e-2)
        at += len(ps)


@pytest.mark.parametrize("kind", ["valu", "mfma", "valu-merge-pass", "mfma-merge-pass"])
@pytest.mark.parametrize("n_splits,waves", [(1, 4), (1, 8), (3, 8), (16, 4), (None, None)])
@pytest.mark.parametrize("nh,nkv,hd,page,window", [(4, 2, 16, 16, None), (6, 1, 48, 8, None), (5, 5, 80, 32, 37),
                                                   (32, 8, 64, 16, None), (16, 2, 128, 16, None), (2, 2, 256, 64, 100),
                                                   (24, 2, 32, 16, None), (3, 1, 24, 16, None)])
def test_attention_decode_split_keys(nh, nkv, hd, page, window, n_splits, waves, kind):
    """The key-splitting kernel against the float64 reference and against the plain kernel, for
    rows of different lengths (one key, a page edge, hundreds of keys) in one call."""
    from gibbs_amd import ops
    dtype = torch.bfloat16
    seq_lens = [700, 1, 33, 16]
    kp, vp, table, ks, vs = paged_setup(dtype, nkv, hd, page, seq_lens, 120, seed=7)
    positions = [l - 1 for l in seq_lens]
    pos, row_req = i32(positions), i32([0, 1, 2, 3])
    q = rnd(4, nh * hd, dtype=dtype, seed=9)
    scale = 1 / math.sqrt(hd)
    if kind.startswith("mfma") and (hd % 16 or hd > 128):
        with pytest.raises(ops.KernelError, match="matrix-core"):
            ops.attention_decode(q, 4, nh, nkv, hd, kp, vp, table, 4, pos, row_req, scale, window, max_seq=700,
                                 n_splits=n_splits, waves=waves, kind=kind)
        return
    out = ops.attention_decode(q, 4, nh, nkv, hd, kp, vp, table, 4, pos, row_req, scale, window, max_seq=700,
                               n_splits=n_splits, waves=waves, kind=kind)
    plain = ops.attention_plain(q, 4, nh, nkv, hd, kp, vp, table, 4, pos, row_req, scale, window)
    for r in range(4):
        want = attention_reference(q[r:r + 1].view(1, nh, hd), ks[r], vs[r], [positions[r]], scale, window)
        close(out[r].view(1, nh, hd), want, dtype, f"decode attention row {r}", bf16=1e-2)
    close(out, plain, dtype, "decode vs plain kernel", bf16=1e-2)


@pytest.mark.parametrize("kind", ["valu", "mfma"])
@pytest.mark.parametrize("n_splits", [1, 4])
@pytest.mark.parametrize("bound", [0, 64, 700])
def test_attention_decode_rows_as_requests_and_rows_beyond_the_bound(bound, n_splits, kind):
    """Without a row-to-request map row n is request n; and the caller's bound on the keys only steers the
    kernel (it asks for a row's page ids before it knows the row's position when the whole table fits its
    staging area): rows beyond the bound take the ids of their slice afterwards and are as right."""
    from gibbs_amd import ops
    dtype, nh, nkv, hd, page = torch.bfloat16, 8, 2, 64, 8
    seq_lens = [700, 1, 33, 16, 300]
    kp, vp, table, ks, vs = paged_setup(dtype, nkv, hd, page, seq_lens, 180, seed=11)
    positions = [l - 1 for l in seq_lens]
    pos = i32(positions)
    q = rnd(5, nh * hd, dtype=dtype, seed=12)
    scale = 1 / math.sqrt(hd)
    out = ops.attention_decode(q, 5, nh, nkv, hd, kp, vp, table, 5, pos, None, scale, None, max_seq=bound,
                               n_splits=n_splits, waves=4, kind=kind)
    mapped = ops.attention_decode(q, 5, nh, nkv, hd, kp, vp, table, 5, pos, i32([0, 1, 2, 3, 4]), scale, None, max_seq=bound,
                                  n_splits=n_splits, waves=4, kind=kind)
    assert torch.equal(out, mapped)
    for r in range(5):
        want = attention_reference(q[r:r + 1].view(1, nh, hd), ks[r], vs[r], [positions[r]], scale, None)
        close(out[r].view(1, nh, hd), want, dtype, f"decode attention row {r}", bf16=1e-2)


@pytest.mark.parametrize("n_splits", [1, 3, 7])
@pytest.mark.parametrize("nh,nkv,hd,page,window", [(4, 2, 16, 16, None), (6, 1, 48, 8, None), (5, 5, 80, 32, 37),
                                                   (32, 8, 64, 16, None), (4, 2, 128, 16, None), (2, 2, 96, 64, 100),
                                                   (3, 1, 32, 16, 5), (8, 2, 48, 16, None), (12, 2, 32, 8, 90),
                                                   (4, 1, 64, 4, None), (4, 2, 64, 5, 60), (2, 1, 64, 24, None), (4, 2, 128, 2, None),
                                                   (2, 1, 128, 24, 70), (4, 2, 32, 12, None), (2, 2, 64, 1, None)])
def test_attention_prefill_matrix_cores(nh, nkv, hd, page, window, n_splits):
    """Prompt portions on the matrix cores: a long portion after a cached context that ends off a
    tile edge, a whole short prompt, a 2-token portion, a single decoded row and a 65-row portion
    that starts at position 0, all in one call; with the key tiles whole or cut into slices (more
    slices than the short requests have tiles: slices without keys)."""
    from gibbs_amd import ops
    dtype = torch.bfloat16
    seq_lens = [333, 9, 130, 77, 65]
    q_lens = [150, 9, 2, 1, 65]
    kp, vp, table, ks, vs = paged_setup(dtype, nkv, hd, page, seq_lens, max(120, sum(-(-s // page) for s in seq_lens) + 3), seed=11)
    ctx = [s - q for s, q in zip(seq_lens, q_lens)]
    cu = np.concatenate([[0], np.cumsum(q_lens)])
    n = int(cu[-1])
    q = rnd(n, nh * hd, dtype=dtype, seed=9)
    scale = 1 / math.sqrt(hd)
    out = ops.attention_prefill(q, n, nh, nkv, hd, kp, vp, table, 5, i32(cu), i32(ctx), scale, window, n_splits=n_splits)
    pos = i32([c + t for c, ql in zip(ctx, q_lens) for t in range(ql)])
    row_req = i32([r for r, ql in enumerate(q_lens) for _ in range(ql)])
    plain = ops.attention_plain(q, n, nh, nkv, hd, kp, vp, table, 5, pos, row_req, scale, window)
    for r in range(5):
        rows = slice(int(cu[r]), int(cu[r + 1]))
        want = attention_reference(q[rows].view(-1, nh, hd), ks[r], vs[r], list(range(ctx[r], seq_lens[r])), scale, window)
        close(out[rows].view(-1, nh, hd), want, dtype, f"prefill attention request {r}", bf16=1e-2)
    close(out, plain, dtype, "prefill vs plain kernel", bf16=1e-2)
    # only the requests from the third on: the rows before them stay as they were
    first_req, first_row = 2, int(cu[2])
    part = torch.full_like(out, 7.0)
    ops.attention_prefill(q, n, nh, nkv, hd, kp, vp, table, 5, i32(cu), i32(ctx), scale, window, out=part,
                          n_splits=n_splits, first_req=first_req, first_row=first_row)
    assert torch.equal(part[first_row:], out[first_row:]) and (part[:first_row] == 7.0).all()
    # several query heads of a kv head's group in one workgroup (one K and V tile for all of them): every row of
    # every head goes through the same operations in the same order, so the result is the same to the bit
    for heads in (2, 4):
        if (nh // nkv) % heads == 0 and hd <= 64:
            many = ops.attention_prefill(q, n, nh, nkv, hd, kp, vp, table, 5, i32(cu), i32(ctx), scale, window,
                                         n_splits=n_splits, heads_per_wg=heads)
            assert torch.equal(many, out), f"{heads} heads a workgroup"
    with pytest.raises(ops.KernelError, match="heads a workgroup"):
        ops.attention_prefill(q, n, nh, nkv, hd, kp, vp, table, 5, i32(cu), i32(ctx), scale, window, heads_per_wg=3)


@pytest.mark.parametrize("nh,nkv,hd,page,extra", [
    (4, 2, 64, 16, {}), (2, 1, 16, 8, {"window": 50}), (3, 1, 48, 7, {"chunk": 40}), (4, 4, 96, 32, {"softcap": 2.0, "sink": True}),
    (2, 2, 128, 5, {"slopes": True, "bias": True}), (1, 1, 80, 16, {"window": 1})])
def test_attention_float32_portions(nh, nkv, hd, page, extra):
    """The matrix-core kernel against the one with a wave a row, which has an oracle of its own: portions that start and end on
    and off the tiles of 64 rows and keys, every form of mask and bias.  Both are sums of at most 333 32-bit products of weights
    that add up to 1, so they differ by less than 333 * 2^-24 of the largest value, and scores of size S move weights by S * hd *
    2^-24: 1e-4 bounds both here.  A value that is not finite reaches the rows that see it and no other."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import call, ptr, stream
    seq_lens, q_lens = [333, 9, 130, 77, 64, 128], [150, 9, 2, 1, 64, 63]
    kp, vp, table, _, _ = paged_setup(torch.float32, nkv, hd, page, seq_lens, 400, seed=11)
    ctx = [s - q for s, q in zip(seq_lens, q_lens)]
    cu = np.concatenate([[0], np.cumsum(q_lens)])
    n, R = int(cu[-1]), len(q_lens)
    q = rnd(n, nh * hd + 4, dtype=torch.float32, seed=9)
    pos = i32([c + t for c, ql in zip(ctx, q_lens) for t in range(ql)])
    row_req = i32([r for r, ql in enumerate(q_lens) for _ in range(ql)])
    opt = dict(extra)
    for name, shape in (("sink", (nh,)), ("slopes", (nh,)), ("bias", (19, nh))):
        if name in opt:
            opt[name] = rnd(*shape, dtype=torch.float32, seed=3)
    bias = opt.get("bias")
    def both():
        want = ops.attention_plain(q, n, nh, nkv, hd, kp, vp, table, R, pos, row_req, hd ** -0.5, **opt)
        got = torch.full((n, nh * hd + 1), 7.0, device="cuda")
        cud, ctxd = i32(cu), i32(ctx)
        for first in (0, 2):      # the requests from some request on: the rows before keep what they hold
            got.fill_(7.0)
            call("gibbs_attention_f32", ptr(q), ptr(kp), ptr(vp), ptr(got), ptr(cud[first:]), ptr(ctxd[first:]), ptr(table[first:]), R - first,
                 table.shape[1], page, kp.shape[0], n - int(cu[first]), nh, nkv, hd, q.stride(0), nh * hd + 1, float(hd ** -0.5),
                 int(opt.get("window", 0)), ptr(opt.get("slopes")), ptr(bias), 0 if bias is None else bias.shape[0], ptr(opt.get("sink")),
                 int(opt.get("chunk", 0)), float(opt.get("softcap", 0.0)), stream())
            assert (got[:, -1] == 7.0).all() and (got[:int(cu[first])] == 7.0).all()
            yield want[int(cu[first]):], got[int(cu[first]):, :-1]
    for want, got in both():
        assert (want - got).abs().max() <= 1e-4 * max(1.0, float(want.abs().max()))
    key = seq_lens[0] - 3        # a key that the first request's last three rows see
    vp[int(table[0, key // page]), :, key % page] = float("inf")
    for want, got in both():
        assert torch.equal(want.isfinite(), got.isfinite())
        assert (want - got)[want.isfinite()].abs().max() <= 1e-4 * max(1.0, float(want[want.isfinite()].abs().max()))


@pytest.mark.parametrize("nh,nkv,hd,page,extra", [
    (4, 2, 64, 16, {}), (2, 1, 16, 8, {"window": 50}), (3, 1, 48, 7, {"chunk": 40}), (4, 4, 32, 32, {"softcap": 2.0, "sink": True}),
    (2, 2, 64, 5, {"slopes": True, "bias": True}), (1, 1, 64, 16, {"window": 1})])
def test_attention_float32_values_twice_as_wide_as_keys(nh, nkv, hd, page, extra):
    """The portions, masks and bounds of the test above with values of 2 hd; a request's rows alone and among the others, the same bits."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import call, ptr, stream
    vd = 2 * hd
    seq_lens, q_lens = [333, 9, 130, 77, 64, 128], [150, 9, 2, 1, 64, 63]
    kp, _, table, _, _ = paged_setup(torch.float32, nkv, hd, page, seq_lens, 400, seed=11)
    vp = rnd(kp.shape[0], nkv, page, vd, dtype=torch.float32, seed=12)
    ctx = [s - q for s, q in zip(seq_lens, q_lens)]
    cu = np.concatenate([[0], np.cumsum(q_lens)])
    n, R = int(cu[-1]), len(q_lens)
    q = rnd(n, nh * hd + 4, dtype=torch.float32, seed=9)
    pos = i32([c + t for c, ql in zip(ctx, q_lens) for t in range(ql)])
    row_req = i32([r for r, ql in enumerate(q_lens) for _ in range(ql)])
    opt = dict(extra)
    for name, shape in (("sink", (nh,)), ("slopes", (nh,)), ("bias", (19, nh))):
        if name in opt:
            opt[name] = rnd(*shape, dtype=torch.float32, seed=3)
    bias = opt.get("bias")
    cud, ctxd = i32(cu), i32(ctx)
    def run(first, count):
        got = torch.full((n, nh * vd + 1), 7.0, device="cuda")
        call("gibbs_attention_f32_values", ptr(q), ptr(kp), ptr(vp), ptr(got), ptr(cud[first:]), ptr(ctxd[first:]), ptr(table[first:]), count, table.shape[1], page,
             kp.shape[0], int(cu[first + count] - cu[first]), nh, nkv, hd, vd, q.stride(0), nh * vd + 1, float(hd ** -0.5), int(opt.get("window", 0)),
             ptr(opt.get("slopes")), ptr(bias), 0 if bias is None else bias.shape[0], ptr(opt.get("sink")), int(opt.get("chunk", 0)),
             float(opt.get("softcap", 0.0)), stream())
        assert (got[:, -1] == 7.0).all() and (got[:int(cu[first])] == 7.0).all() and (got[int(cu[first + count]):] == 7.0).all()
        return got[:, :-1]
    for poisoned in (False, True):
        if poisoned:
            key = seq_lens[0] - 3        # a key that the first request's last three rows see
            vp[int(table[0, key // page]), :, key % page] = float("inf")
        want, got = ops.attention_plain(q, n, nh, nkv, hd, kp, vp, table, R, pos, row_req, hd ** -0.5, **opt), run(0, R)
        finite = want.isfinite()
        assert torch.equal(finite, got.isfinite())
        assert (want - got)[finite].abs().max() <= 1e-4 * max(1.0, float(want[finite].abs().max()))
        for r in range(R):
            a, b = int(cu[r]), int(cu[r + 1])
            assert torch.equal(torch.nan_to_num(run(r, 1)[a:b], nan=5.0), torch.nan_to_num(got[a:b], nan=5.0))


def test_attention_float32_many_requests():
    """150 requests of 1 to 130 rows in one call: each one's rows are those of a call of its own, to the bit (the workgroups find their request among
    64 at a time)."""
    from gibbs_amd.ops.lib import call, ptr, stream
    nh, nkv, hd, page, R = 2, 1, 16, 16, 150
    q_lens = [1 + (i * 37) % 130 if i % 3 else 1 for i in range(R)]
    ctx = [(i * 53) % 90 for i in range(R)]
    kp, vp, table, _, _ = paged_setup(torch.float32, nkv, hd, page, [c + ql for c, ql in zip(ctx, q_lens)], 2200, seed=5)
    cu = np.concatenate([[0], np.cumsum(q_lens)])
    n = int(cu[-1])
    q = rnd(n, nh * hd, dtype=torch.float32, seed=6)
    cud, ctxd = i32(cu), i32(ctx)
    def run(first, count):
        out = torch.zeros((n, nh * hd), device="cuda")
        call("gibbs_attention_f32", ptr(q), ptr(kp), ptr(vp), ptr(out), ptr(cud[first:]), ptr(ctxd[first:]), ptr(table[first:]), count, table.shape[1], page, kp.shape[0],
             int(cu[first + count] - cu[first]), nh, nkv, hd, nh * hd, nh * hd, 0.25, 0, None, None, 0, None, 0, 0.0, stream())
        return out
    whole = run(0, R)
    for r in range(R):
        assert torch.equal(run(r, 1)[cu[r]:cu[r + 1]], whole[cu[r]:cu[r + 1]]), r
    assert whole.isfinite().all() and (whole.abs().sum(1) > 0).all()


@pytest.mark.parametrize("nh,nkv,hd,page,how", [
    (8, 2, 64, 16, {}), (4, 2, 64, 8, {"window": 70}), (3, 1, 64, 64, {"chunk": 100}), (4, 1, 128, 16, {"softcap": 3.0}),
    (2, 1, 128, 8, {"window": 1}), (3, 3, 128, 32, {"sink": True}), (2, 1, 64, 128, {"splits": 3})])
def test_attention_prompt_edges(nh, nkv, hd, page, how):
    """Rows around the edges of a wave's 32 and keys around those of a tile's 64, one tile and more than 64 of them (page ids are
    taken anew), unused keys of the last page that are no numbers, against the kernel with a wave a row."""
    from gibbs_amd import ops
    q_lens = [1, 31, 32, 33, 64, 65, 129, 3, 40]
    seq_lens = [1, 63, 64, 65, 128, 193, 129, 2050, 4330]
    kp, vp, table, _, _ = paged_setup(torch.bfloat16, nkv, hd, page, seq_lens, sum(-(-s // page) for s in seq_lens) + 3, seed=17)
    for r, s in enumerate(seq_lens):
        if s % page:
            kp[table[r, s // page].item(), :, s % page:] = math.nan
            vp[table[r, s // page].item(), :, s % page:] = math.nan
    ctx = [s - n for s, n in zip(seq_lens, q_lens)]
    cu = np.concatenate([[0], np.cumsum(q_lens)])
    n = int(cu[-1])
    q = rnd(n, nh * hd, dtype=torch.bfloat16, seed=4)
    scale, window, chunk, softcap = 1 / math.sqrt(hd), how.get("window"), how.get("chunk", 0), how.get("softcap", 0.0)
    sink = rnd(nh, seed=6) if how.get("sink") else None
    out = ops.attention_prefill(q, n, nh, nkv, hd, kp, vp, table, len(q_lens), i32(cu), i32(ctx), scale, window, sink=sink, chunk=chunk,
                                softcap=softcap, n_splits=how.get("splits", 1), heads_per_wg=0)
    pos = i32([c + t for c, m in zip(ctx, q_lens) for t in range(m)])
    row_req = i32([r for r, m in enumerate(q_lens) for _ in range(m)])
    plain = ops.attention_plain(q, n, nh, nkv, hd, kp, vp, table, len(q_lens), pos, row_req, scale, window, sink=sink, chunk=chunk,
                                softcap=softcap)
    assert out.isfinite().all()
    close(out, plain, torch.bfloat16, "prompt attention", bf16=1e-2)


@pytest.mark.parametrize("heads", [0, 1])
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("softcap", [0.0, 6.0])
@pytest.mark.parametrize("nh,nkv,hd,page", [(4, 1, 64, 16), (2, 1, 64, 8), (3, 3, 64, 64), (4, 1, 128, 16), (2, 1, 128, 32), (2, 2, 128, 8)])
def test_attention_prompt_bias_by_distance(nh, nkv, hd, page, softcap, splits, heads):
    """A bias on the scores by distance, with heads that look at one distance each: a table that lies one key or one row off gives other
    rows altogether.  One, two and four heads a workgroup, capped scores too, slices that begin at any tile, more than 64 tiles; both kernels against
    the one with a wave a row."""
    from gibbs_amd import ops
    q_lens, seq_lens = [1, 33, 64, 129, 70, 200], [1, 65, 64, 193, 4300, 333]
    kp, vp, table, _, _ = paged_setup(torch.bfloat16, nkv, hd, page, seq_lens, sum(-(-s // page) for s in seq_lens) + 3, seed=17)
    ctx = [s - n for s, n in zip(seq_lens, q_lens)]
    cu, n, scale = np.concatenate([[0], np.cumsum(q_lens)]), sum(q_lens), 1 / math.sqrt(hd)
    q, bias = rnd(n, nh * hd, dtype=torch.bfloat16, seed=4), rnd(300, nh, seed=5)
    for h in range(nh):
        bias[[63, 64, 1, 130][h], h] += 12.0
    pos = i32([c + t for c, m in zip(ctx, q_lens) for t in range(m)])
    row_req = i32([r for r, m in enumerate(q_lens) for _ in range(m)])
    out = ops.attention_prefill(q, n, nh, nkv, hd, kp, vp, table, len(q_lens), i32(cu), i32(ctx), scale, n_splits=splits, heads_per_wg=heads,
                                softcap=softcap, bias=bias)
    plain = ops.attention_plain(q, n, nh, nkv, hd, kp, vp, table, len(q_lens), pos, row_req, scale, bias=bias, softcap=softcap)
    close(out, plain, torch.bfloat16, "biased prompt attention", bf16=1e-2)


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("nh,nkv,hd,page,how", [
    (4, 1, 64, 16, {}), (4, 2, 64, 8, {"window": 40}), (3, 3, 64, 16, {}), (2, 2, 64, 32, {"chunk": 90}), (4, 1, 128, 16, {"window": 70}),
    (3, 3, 128, 8, {"softcap": 4.0}), (2, 1, 128, 16, {})])
def test_attention_prompt_values_that_are_not_finite(nh, nkv, hd, page, how, splits):
    """A value that is not finite reaches the rows that see its key and no other, whatever rows a wave and a workgroup have: in one tile and
    in several, on and beside the diagonal, behind rows that no longer see it.  The rest is what it is without those values."""
    from gibbs_amd import ops
    q_lens, ctx = [64, 150, 300], [0, 70, 3]
    seq_lens = [a + b for a, b in zip(q_lens, ctx)]
    cu = np.concatenate([[0], np.cumsum(q_lens)])
    n, scale, window, chunk = int(cu[-1]), 1 / math.sqrt(hd), how.get("window"), how.get("chunk", 0)
    kp, vp, table, _, _ = paged_setup(torch.bfloat16, nkv, hd, page, seq_lens, sum(-(-s // page) for s in seq_lens), seed=3)
    q = rnd(n, nh * hd, dtype=torch.bfloat16, seed=4)
    pos = i32([c + t for c, m in zip(ctx, q_lens) for t in range(m)])
    row_req = i32([r for r, m in enumerate(q_lens) for _ in range(m)])

    def run():
        return ops.attention_prefill(q, n, nh, nkv, hd, kp, vp, table, 3, i32(cu), i32(ctx), scale, window, chunk=chunk, n_splits=splits,
                                     softcap=how.get("softcap", 0.0), heads_per_wg=0).view(n, nh, hd)
    clean = run()
    seen = torch.zeros(n, nh, hd, dtype=torch.bool, device=DEV)
    for r, key, kvh, d, bad in ((0, 63, 0, 5, math.nan), (1, 100, nkv - 1, hd - 1, math.inf), (1, 219, 0, 33, math.nan), (2, 17, 0, 8, -math.inf),
                                (2, 130, nkv - 1, 0, math.nan), (2, 302, 0, 31, math.inf)):
        vp[table[r, key // page].item(), kvh, key % page, d] = bad
        sees = (row_req == r) & (pos >= key)
        if window:
            sees &= pos - key < window
        if chunk:
            sees &= pos // chunk == key // chunk
        heads = slice(kvh * (nh // nkv), (kvh + 1) * (nh // nkv))
        seen[:, heads, d] |= sees[:, None]
    got = run()
    assert torch.equal(~got.isfinite(), seen)
    # (rows that are taken again: other roundings of float32 sums, and a weight's bfloat16 may round the other way)
    close(got[~seen], clean[~seen], torch.bfloat16, "beside values that are not finite", bf16=4e-3)


def test_prefill_splits_choice():
    from gibbs_amd.ops import prefill_splits
    assert prefill_splits(32, 32, 2048) == 1                 # a whole 2,048-token prompt fills the chip
    assert prefill_splits(8, 32, 8192) == 8                  # a portion of 512 late in a long prompt does not
    assert prefill_splits(1, 4, 300) == 1 and prefill_splits(1, 4, 100000) == 16
    assert prefill_splits(8, 32, 8192, window=128) == 1      # a window bounds the keys


@pytest.mark.parametrize("dtype", DT)
def test_attention_far_key_stands_out(dtype):
    """One key far back among hundreds gets a large score: its value must dominate the output."""
    from gibbs_amd import ops
    nh = nkv = 1; hd = 32; L = 700
    kp, vp, table, ks, vs = paged_setup(dtype, nkv, hd, 16, [L], 64, seed=3)
    q = rnd(1, hd, dtype=dtype, seed=1)
    far = 5
    page, off = table[0, far // 16].item(), far % 16
    kp[page, 0, off] = (q[0].float() * 8).to(dtype)
    ks[0][far, 0] = kp[page, 0, off]
    out = ops.attention_plain(q, 1, nh, nkv, hd, kp, vp, table, 1, i32([L - 1]), i32([0]), 1 / math.sqrt(hd))
    want = attention_reference(q.view(1, 1, hd), ks[0], vs[0], [L - 1], 1 / math.sqrt(hd), None)
    close(out.view(1, 1, hd), want, dtype, "far key", f32=2e-5, bf16=1e-2)
    assert (out.float() - vs[0][far, 0].float()).abs().max() < 0.05 * vs[0][far, 0].float().abs().max() + 0.05
    if dtype == torch.bfloat16:
        # the same through the fast kernels: split keys (the far key lies in the first slice), and
        # the matrix-core kernel with the row as the last of a 2-row portion
        split = ops.attention_decode(q, 1, nh, nkv, hd, kp, vp, table, 1, i32([L - 1]), i32([0]), 1 / math.sqrt(hd), n_splits=8)
        close(split.view(1, 1, hd), want, dtype, "far key, split keys", bf16=1e-2)
        q2 = torch.cat([rnd(1, hd, dtype=dtype, seed=2), q])
        pre = ops.attention_prefill(q2, 2, nh, nkv, hd, kp, vp, table, 1, i32([0, 2]), i32([L - 2]), 1 / math.sqrt(hd))
        close(pre[1].view(1, 1, hd), want, dtype, "far key, matrix cores", bf16=1e-2)


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("variant", ["half_split", "interleaved"])
@pytest.mark.parametrize("table_len", [0, 6, 64])       # no table; positions 9 and 17 beyond it; all from it
@pytest.mark.parametrize("nh,nkv,hd,rot", [(4, 2, 16, 16), (3, 1, 48, 32), (2, 2, 128, 128), (2, 1, 24, 12)])
def test_qk_rope_kv(dtype, variant, nh, nkv, hd, rot, table_len):
    from gibbs_amd import ops
    from gibbs_amd.parts.rope import rope_inv_freq
    n, page, num_pages = 6, 8, 10
    qkv = rnd(n, (nh + 2 * nkv) * hd, dtype=dtype)
    qkv0 = qkv.clone()
    qg, kg = rnd(hd, seed=1) + 1, rnd(hd, seed=2) + 1
    inv = torch.from_numpy(rope_inv_freq(rot, 10000.0, "f32")).to(DEV)
    positions = [3, 4, 5, 0, 17, 9]
    row_req = [0, 0, 0, 1, 1, 2]
    table = i32([[4, 7, -1], [2, 9, 0], [5, 1, -1]])
    kp = torch.zeros(num_pages, nkv, page, hd, dtype=dtype, device=DEV)
    vp = torch.zeros_like(kp)
    cos_sin = ops.rope_table(inv, table_len) if table_len else None
    ops.qk_rope_kv(qkv, n, nh, nkv, hd, q_gain=qg, k_gain=kg, eps=1e-6, inv_freq=inv, rotary_dim=rot, variant=variant,
                   pos=i32(positions), row_req=i32(row_req), kpages=kp, vpages=vp, table=table, n_req=3, cos_sin=cos_sin)
    if table_len:   # a table changes nothing, to the bit: it holds what the kernel computes
        qkv1, kp1, vp1 = qkv0.clone(), torch.zeros_like(kp), torch.zeros_like(vp)
        ops.qk_rope_kv(qkv1, n, nh, nkv, hd, q_gain=qg, k_gain=kg, eps=1e-6, inv_freq=inv, rotary_dim=rot,
                       variant=variant, pos=i32(positions), row_req=i32(row_req), kpages=kp1, vpages=vp1, table=table,
                       n_req=3)
        assert torch.equal(qkv1, qkv) and torch.equal(kp1, kp) and torch.equal(vp1, vp)

    def ref(x, gain):                                     # x: [n, heads, hd] float64
        x = F.rms_norm(x, (hd,), gain.double(), eps=1e-6)
        ang = torch.tensor(positions, dtype=torch.float32, device=DEV)[:, None] * inv[None, :]
        c, s = ang.double().cos()[:, None, :], ang.double().sin()[:, None, :]
        out = x.clone()
        half = rot // 2
        i0 = torch.arange(half) if variant == "half_split" else torch.arange(half) * 2
        i1 = i0 + half if variant == "half_split" else i0 + 1
        out[..., i0] = x[..., i0] * c - x[..., i1] * s
        out[..., i1] = x[..., i0] * s + x[..., i1] * c
        return out
    q0 = qkv0[:, :nh * hd].double().view(n, nh, hd)
    k0 = qkv0[:, nh * hd:(nh + nkv) * hd].double().view(n, nkv, hd)
    v0 = qkv0[:, (nh + nkv) * hd:].view(n, nkv, hd)
    close(qkv[:, :nh * hd].view(n, nh, hd), ref(q0, qg), dtype, "q", bf16=8e-3)
    kr = ref(k0, kg)
    for i, (p, r) in enumerate(zip(positions, row_req)):
        pg = table[r, p // page].item()
        close(kp[pg, :, p % page], kr[i], dtype, "k page", bf16=8e-3)
        assert torch.equal(vp[pg, :, p % page], v0[i])
    assert kp.float().abs().sum(dim=(1, 3)).count_nonzero().item() == n, "exactly one page slot per row was written"

@pytest.mark.parametrize("nh,nkv,hd", [(16, 8, 64), (3, 1, 48), (6, 1, 256), (5, 2, 16)])
def test_qk_rope_kv_one_head_or_four_a_lane_group(nh, nkv, hd):
    """Where rows stop being few (393,216 lanes of 8 values): rows and cache pages are to the bit those of a call with some more rows."""
    from gibbs_amd import ops
    from gibbs_amd.parts.rope import rope_inv_freq
    line = (3 << 17) // ((nh + 2 * nkv) * (hd // 8))
    rows, page = line + 3, 64
    pages = rows // page + 1
    x, qg, kg = rnd(rows, (nh + 2 * nkv) * hd, dtype=torch.bfloat16), rnd(hd, seed=1) + 1, rnd(hd, seed=2) + 1
    inv = torch.from_numpy(rope_inv_freq(hd, 10000.0, "f32")).to(DEV)
    table = i32([np.random.default_rng(3).permutation(pages).tolist()])
    def run(n):
        qkv = x[:n].clone()
        kp, vp = (torch.zeros(pages, nkv, page, hd, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        ops.qk_rope_kv(qkv, n, nh, nkv, hd, q_gain=qg, k_gain=kg, eps=1e-6, inv_freq=inv, rotary_dim=hd, variant="half_split",
                       pos=i32(list(range(n))), row_req=i32([0] * n), kpages=kp, vpages=vp, table=table, n_req=1, cos_sin=ops.rope_table(inv, 128))
        for r in range(n, rows):
            assert not kp[table[0, r // page].item(), :, r % page].any()
        return qkv[:, :nh * hd], kp, vp
    few, many = run(line), run(rows)
    for r in range(line, rows):
        many[1][table[0, r // page].item(), :, r % page] = 0
        many[2][table[0, r // page].item(), :, r % page] = 0
    assert torch.equal(few[0], many[0][:line]) and torch.equal(few[1], many[1]) and torch.equal(few[2], many[2])


def plain_qk(x, gain, positions, inv, eps):
    """Per-head RMSNorm then the half-split rotation of x [n, heads, hd], by the plain implementation
    (float32 angle = float32(pos) * inv_freq, src/graph/cpu.rs:673)."""
    from tests.plain import lfm2_plain as P
    return torch.tensor(P.rope_half_split(P.rms_norm(x.double().cpu().numpy(), gain.double().cpu().numpy(), eps), positions, inv))


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("table_len", [0, 4096])
def test_qk_rope_kv_at_far_positions(dtype, table_len):
    """theta 1e6, heads of 64, rows at positions 32,767 and 99,999 (and beside them, and near the start):
    there the float32 product float32(pos) * inv_freq has lost its low bits, and an angle computed any
    other way (in float64, from a recurrence, as pos * a rounded inverse) is off by up to 4e-3 rad.  Against
    the plain implementation's rotation, which takes the reference's float32 steps."""
    from gibbs_amd import ops
    from tests.plain import lfm2_plain as P
    nh, nkv, hd, page = 4, 2, 64, 16
    positions = [99999, 32767, 99998, 5, 65536, 32768]
    n = len(positions)
    inv_np = P.rope_inv_freq(hd, 1e6)
    inv = torch.from_numpy(inv_np).to(DEV)
    qkv = rnd(n, (nh + 2 * nkv) * hd, dtype=dtype, seed=3)
    qkv0 = qkv.clone()
    qg, kg = rnd(hd, seed=1) * 0.1 + 1, rnd(hd, seed=2) * 0.1 + 1
    width = 100000 // page
    table = np.full((n, width), -1, dtype=np.int32)
    for r, p in enumerate(positions):                       # one request per row, one real page each
        table[r, p // page] = n - 1 - r
    kp = torch.zeros(n, nkv, page, hd, dtype=dtype, device=DEV)
    vp = torch.zeros_like(kp)
    ops.qk_rope_kv(qkv, n, nh, nkv, hd, q_gain=qg, k_gain=kg, eps=1e-5, inv_freq=inv, rotary_dim=hd, variant="half_split",
                   pos=i32(positions), row_req=i32(list(range(n))), kpages=kp, vpages=vp, table=i32(table), n_req=n,
                   cos_sin=ops.rope_table(inv, table_len) if table_len else None)
    q0 = qkv0[:, :nh * hd].view(n, nh, hd)
    k0 = qkv0[:, nh * hd:(nh + nkv) * hd].view(n, nkv, hd)
    close(qkv[:, :nh * hd].view(n, nh, hd), plain_qk(q0, qg, positions, inv_np, 1e-5), dtype, "q at far positions", f32=2e-6, bf16=8e-3)
    kr = plain_qk(k0, kg, positions, inv_np, 1e-5)
    for r, p in enumerate(positions):
        close(kp[n - 1 - r, :, p % page], kr[r], dtype, f"k at position {p}", f32=2e-6, bf16=8e-3)
    # the same angles in float64 would fail this bound: the test can tell the difference
    ang32 = (np.float32(99999) * inv_np).astype(np.float64)
    ang64 = 99999.0 * inv_np.astype(np.float64)
    assert np.abs(np.cos(ang32) - np.cos(ang64)).max() > 1e-4


@pytest.mark.parametrize("kind", ["valu", "mfma"])
@pytest.mark.parametrize("window", [None, 48])
def test_attention_decode_fused_at_far_positions(kind, window):
    """Decoded tokens at positions 99,999 and 32,767 (theta 1e6, pages of 16: 6,250 page ids, so the
    matrix-core walk must cut the cache into slices whatever the batch) beside a short request: q/k norm and
    rotation against the plain implementation's, attention against float64 over all 100,000 keys.  The
    query gain is large, so that the softmax stands on a few hundred keys spread over the whole cache (a
    slice or a page lost shows), and with a window of 48 keys every score depends on the rotation."""
    from gibbs_amd import ops
    from tests.plain import lfm2_plain as P
    dtype, nh, nkv, hd, page = torch.bfloat16, 8, 2, 64, 16
    seq_lens = [100000, 32768, 40]
    kp, vp, table, ks, vs = paged_setup(dtype, nkv, hd, page, seq_lens, sum(-(-l // page) for l in seq_lens) + 3, seed=11)
    n = len(seq_lens)
    positions = [l - 1 for l in seq_lens]
    pos, row_req = i32(positions), i32(list(range(n)))
    qkv = rnd(n, (nh + 2 * nkv) * hd, dtype=dtype, seed=9)
    qg, kg = rnd(hd, seed=1) * 0.1 + 3.0, rnd(hd, seed=2) * 0.1 + 1
    inv_np = P.rope_inv_freq(hd, 1e6)
    inv = torch.from_numpy(inv_np).to(DEV)
    scale = 1 / math.sqrt(hd)
    got = ops.attention_decode_fused(qkv, n, nh, nkv, hd, kp, vp, table, n, pos, row_req, scale, q_gain=qg, k_gain=kg,
                                     eps=1e-5, inv_freq=inv, rotary_dim=hd, variant="half_split", window=window,
                                     max_seq=max(seq_lens), kind=kind, cos_sin=ops.rope_table(inv, 4096))
    # (the kernel rounds the prepared q and the new key to bfloat16, as the separate kernels store them; with
    # scores this large that rounding alone moves the output by 1 %, so the reference takes the same values)
    q = plain_qk(qkv[:, :nh * hd].view(n, nh, hd), qg, positions, inv_np, 1e-5).to(DEV).to(dtype).double()
    k_new = plain_qk(qkv[:, nh * hd:(nh + nkv) * hd].view(n, nkv, hd), kg, positions, inv_np, 1e-5).to(DEV).to(dtype).double()
    v_new = qkv[:, (nh + nkv) * hd:].view(n, nkv, hd)
    for r, p in enumerate(positions):
        pg = table[r, p // page].item()
        close(kp[pg, :, p % page], k_new[r], dtype, f"new key at position {p}", bf16=8e-3)
        assert torch.equal(vp[pg, :, p % page], v_new[r])
        k_all = torch.cat([ks[r][:p].double(), k_new[r:r + 1]])
        v_all = torch.cat([vs[r][:p].double(), v_new[r:r + 1].double()])
        want = attention_reference(q[r:r + 1], k_all, v_all, [p], scale, window)
        close(got[r].view(1, nh, hd), want, dtype, f"row at position {p}", bf16=1e-2)


def test_rope_table():
    from gibbs_amd import ops
    from gibbs_amd.parts.rope import rope_inv_freq
    inv = torch.from_numpy(rope_inv_freq(48, 1e6, "f32")).to(DEV)
    t = ops.rope_table(inv, 5000)
    ang = (torch.arange(5000, dtype=torch.float32, device=DEV)[:, None] * inv[None, :]).double()   # float32 products
    assert t.shape == (5000, 24, 2)
    assert (t[..., 0].double() - ang.cos()).abs().max().item() < 2e-7
    assert (t[..., 1].double() - ang.sin()).abs().max().item() < 2e-7


def test_argmax_rules():
    from gibbs_amd import ops
    nan, inf = float("nan"), float("inf")
    rows = torch.tensor([[1.0, 3.0, 3.0, 2.0, 0.0], [nan, 1.0, nan, 1.0, 0.0], [-inf] * 5, [nan] * 5,
                         [0.0, -1.0, -2.0, -3.0, 5.0]], device=DEV)
    assert ops.argmax(rows).tolist() == [1, 1, 0, 0, 4]
    big = rnd(3, 65536 + 37)
    big[1, 40000] = big[1, 70] = 99.0
    assert ops.argmax(big).tolist() == [big[0].argmax().item(), 70, big[2].argmax().item()]


def test_sample_against_plain():
    from gibbs_amd import ops
    from tests.plain import lfm2_plain as P
    V, M = 1000, 12
    logits = rnd(M, V, scale=3.0, seed=5)
    rng = np.random.default_rng(0)
    temp = np.array([0.8, 1.0, 0.3, 1.5] * 3, dtype=np.float32)
    top_p = np.array([0.9, 0.5, 1.0, 0.95] * 3, dtype=np.float32)
    top_k = np.array([50, 64, 5, 1] * 3, dtype=np.int32)
    u = rng.random(M).astype(np.float32)
    got = ops.sample(logits, torch.tensor(temp, device=DEV), torch.tensor(top_p, device=DEV), i32(top_k),
                     torch.tensor(u, device=DEV)).tolist()
    for m in range(M):
        cand, probs = P.nucleus(logits[m].cpu().numpy(), float(temp[m]), int(top_k[m]), float(top_p[m]))
        assert got[m] == P.draw(cand, probs, float(u[m])), f"row {m}"
    # temperature <= 1e-4 is greedy
    g = ops.sample(logits, torch.zeros(M, device=DEV), torch.tensor(top_p, device=DEV), i32(top_k), torch.tensor(u, device=DEV))
    assert g.tolist() == logits.argmax(-1).tolist()


@pytest.mark.parametrize("V,R", [(700, 64), (65536 + 37, 64), (97, 5)])
def test_repetition_penalty(V, R):
    """The kernel against the plain rule, row by row: greedy and sampled rows, tokens seen once and
    several times, positive and negative logits, ids outside the vocabulary and empty places in the
    list, rows without a penalty (left alone bit for bit)."""
    from gibbs_amd import ops
    from tests.plain import lfm2_plain as P
    rng = np.random.default_rng(V + R)
    M = 7
    logits = rnd(M, V, scale=3.0, seed=V)
    recent = rng.integers(0, min(V, 12), size=(M, R)).astype(np.int32)       # few distinct ids: many repeats
    recent[1, R // 2:] = -1                                                      # a short history
    recent[2, 0] = V + 5                                                         # an id outside the vocabulary
    recent[3] = rng.integers(0, V, size=R)
    recent[6] = -1                                                               # nothing recent
    penalty = np.array([1.3, 2.0, 1.1, 1.5, 1.0, 0.7, 1.8], dtype=np.float32)  # 1.0 and below: none
    temp = np.array([0.0, 0.8, 1e-4, 1.2, 0.0, 0.9, 0.7], dtype=np.float32)
    before = logits.clone()
    got = ops.repetition_penalty(logits, i32(recent), torch.tensor(penalty, device=DEV), torch.tensor(temp, device=DEV))
    assert got.data_ptr() == logits.data_ptr()
    got = got.cpu().numpy()
    for m in range(M):
        want = P.repetition_penalty(before[m].cpu().numpy(), [t for t in recent[m] if t >= 0], float(penalty[m]),
                                    greedy=bool(temp[m] <= 1e-4))
        assert np.array_equal(got[m], want), f"row {m}: {np.abs(got[m] - want).max()}"
    assert np.array_equal(got[4], before[4].cpu().numpy()) and np.array_equal(got[6], before[6].cpu().numpy())
    assert not np.array_equal(got[0], before[0].cpu().numpy())


@pytest.mark.parametrize("V", [65536, 50001, 700])
def test_sample_large_vocabulary_ties_and_specials(V):
    """Top-k by two walks over the row: vocabularies beyond one element per thread, a thousand values tied
    at the top (the smaller ids win), a row of equal logits (more ties than the candidate list holds),
    NaN (never a candidate) and -inf among the values, and -0 beside +0 at the top (equal values)."""
    from gibbs_amd import ops
    from tests.plain import lfm2_plain as P
    rng = np.random.default_rng(V)
    rows = [rng.standard_normal(V).astype(np.float32) * 3 for _ in range(6)]
    top = rows[1].max() + 1
    rows[1][rng.choice(V, size=min(1000, V // 2), replace=False)] = top          # many ties at the top
    rows[2][:] = 0.25                                                          # everything ties
    rows[3][rng.choice(V, size=V // 3, replace=False)] = np.nan
    rows[3][rng.choice(V, size=V // 4, replace=False)] = -np.inf
    rows[4] = -np.abs(rows[4]) - 1
    zeros = rng.choice(V, size=40, replace=False)
    rows[4][zeros[:20]] = 0.0
    rows[4][zeros[20:]] = -0.0
    rows[5][:] = -np.inf                                                       # nothing above -inf: still candidates
    rows[5][V // 2] = 1.0
    logits = torch.tensor(np.stack(rows), device=DEV)
    M = len(rows)
    for temp, p, k in [(0.8, 0.9, 50), (1.3, 1.0, 64), (0.5, 0.97, 7)]:
        u = rng.random(M).astype(np.float32)
        got = ops.sample(logits, torch.full((M,), temp, device=DEV), torch.full((M,), p, device=DEV),
                         i32([k] * M), torch.tensor(u, device=DEV)).tolist()
        for m in range(M):
            cand, probs = P.nucleus(rows[m], temp, k, p)
            assert got[m] == P.draw(cand, probs, float(u[m])), f"row {m}, k {k}"
    greedy = ops.sample(logits, torch.zeros(M, device=DEV), torch.ones(M, device=DEV), i32([50] * M), torch.zeros(M, device=DEV))
    assert greedy.tolist() == [P.argmax_first(r) for r in rows] == ops.argmax(logits).tolist()


# --------------------------------------------------------------------------- fused decode kernels
def rms_scale(x, eps):
    return 1.0 / torch.sqrt((x.double() ** 2).mean(-1, keepdim=True) + eps)


@pytest.mark.parametrize("n,o,i", [(1, 64, 128), (8, 3072, 2048), (16, 331 * 8, 1000), (17, 200, 512), (64, 96, 4096), (5, 40, 72),
                                   (48, 8200, 512), (64, 3072, 2048),      # two tiles a workgroup; many rows, one tile
                                   (3, 20, 104), (8, 1001, 1000), (7, 4100, 104), (8, 4099, 2048), (9, 4100, 72),
                                   (12, 36, 200),                           # paired operands with ragged ends, both layouts
                                   (13, 2100, 264), (10, 40, 520)])         # 9 to 16 rows: two tiles of 8 rows in pairs; few features: staged
def test_skinny_store_with_rms_prologue(n, o, i):
    from gibbs_amd import ops
    x, w = rnd(n, i, dtype=torch.bfloat16, scale=3.0), rnd(o, i, dtype=torch.bfloat16, seed=1)
    plain = x.double() @ w.double().t()
    close(ops.skinny_store(x, w), plain, torch.bfloat16, "skinny_store", bf16=4e-3)
    got = ops.skinny_store(x, w, rms_eps=1e-5)
    close(got, plain * rms_scale(x, 1e-5), torch.bfloat16, "skinny_store rms", bf16=4e-3)
    assert torch.equal(ops.skinny_store(x, ops.PackedWeight(w), rms_eps=1e-5), got), "tile-ordered weights: same sums"


@pytest.mark.parametrize("n,o,i", [(1, 2048, 2048), (8, 2048, 8192), (33, 200, 512), (64, 72, 96), (64, 2048, 2048),
                                   (40, 1000, 4096),                        # many rows: partial sums over k, then the add
                                   (7, 36, 200), (8, 4100, 136), (2, 12, 8),
                                   (12, 2056, 200), (15, 4100, 136), (10, 36, 200)])   # 9 to 16 rows: pairs (8 and 16 features), staged
def test_skinny_residual(n, o, i):
    from gibbs_amd import ops
    y, w = rnd(n, i, dtype=torch.bfloat16), rnd(o, i, dtype=torch.bfloat16, seed=1)
    x = rnd(n, o, scale=2.0, seed=2)
    want = x.double() + y.double() @ w.double().t()
    mirror = torch.zeros(n, o, dtype=torch.bfloat16, device=DEV)
    x0 = x.clone()
    ops.skinny_residual(y, w, x, mirror)
    close(x, want, torch.float32, "skinny_residual", f32=2e-5)
    assert torch.equal(mirror, x.to(torch.bfloat16))
    ops.skinny_residual(y, ops.PackedWeight(w), x0, mirror)
    assert torch.equal(x0, x), "tile-ordered weights: same sums"


@pytest.mark.parametrize("n", [1, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("o,i", [(72, 1088), (72, 64), (4104, 520)])
def test_few_row_products_add_waves_in_order_and_a_waves_halves_one_after_the_other(n, o, i):
    """The order in which the eight waves' shares of k are added is part of the bits.  Workgroups of 8 features hold a share as two
    sums, of the even and of the odd 32 of k: first + second of wave 0, + first of wave 1, + its second, and so on; workgroups of 16 one sum a wave.  A
    share by itself is the product with X zero everywhere else (zeros add nothing).  Products of two and three row groups add like those of one."""
    from gibbs_amd import ops
    x, w = rnd(n, i, dtype=torch.bfloat16, seed=1), rnd(3 * o, i, dtype=torch.bfloat16, seed=2)
    def product(rows, matrix):
        total, mirror = torch.zeros(n, o, device=DEV), torch.empty(n, o, dtype=torch.bfloat16, device=DEV)
        ops.skinny_residual(rows, ops.PackedWeight(matrix), total, mirror)
        return total
    pairs = ops.pair_layout(o) and n <= 32
    unit = 64 if pairs else 32
    share = -(-(-(-i // unit)) // 8) * unit
    k = torch.arange(i, device=DEV)
    want = torch.zeros(n, o, device=DEV)
    for wave in range(8):
        for half in range(2 if pairs else 1):
            mine = (k // share == wave) & ((k // 32 % 2 == half) if pairs else True)
            want += product(torch.where(mine, x, torch.zeros_like(x)), w[:o])
    assert torch.equal(product(x, w[:o]), want)
    if n > 8:      # (rows that pass through LDS: a wave starts elsewhere in its share with every number of row groups)
        return
    b, c, d = (product(x, w[g * o:(g + 1) * o].contiguous()) for g in range(3))
    assert torch.equal(ops.skinny_glu(x, ops.PackedWeight(w[:2 * o].contiguous(), groups=2), activation="relu"), (b.relu() * c).to(torch.bfloat16))
    taps = torch.zeros(o, 3, device=DEV)
    taps[:, 2] = 1.0
    state = torch.zeros(n, 2, o, device=DEV)
    y = ops.skinny_conv(x, ops.PackedWeight(w, groups=3), taps, None, state, i32(list(range(n))), i32([0] * n))
    assert torch.equal(state[:, 1], b * d) and torch.equal(y, (c * (b * d)).to(torch.bfloat16))


@pytest.mark.parametrize("f", [8, 520, 2056])
@pytest.mark.parametrize("clamped", [False, True])
def test_gates_of_every_size(f, clamped):
    """Gates around 80, beyond which the exponential is taken in full for a wave's elements, signed zeros, infinities and NaN among them, against
    float64, and each row the same beside any other."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import call, dtype_code, ptr, stream
    bf = torch.bfloat16
    gu = rnd(9, 2 * f, dtype=bf, scale=4.0, seed=f)
    odd = torch.tensor([80.0, -80.0, 80.5, -80.5, -100.0, -0.0, 0.0, 1e37], dtype=bf, device=DEV)      # (1e37 times an up value is still a bfloat16)
    gu[1, :8], gu[2, f - 8:f], gu[3, :2], gu[4, f - 1] = odd, odd, torch.tensor([math.inf, -math.inf], dtype=bf, device=DEV), math.nan
    def run(t):
        if not clamped:
            return ops.glu(t)
        o = torch.empty((t.shape[0], f), dtype=bf, device=DEV)
        call("gibbs_glu_clamped", ptr(t), ptr(o), dtype_code(bf), t.shape[0], f, 1.702, 7.0, stream())
        return o
    out, x, u = run(gu), gu[:, :f].double(), gu[:, f:].double()
    if clamped:
        g = torch.fmin(x, torch.full_like(x, 7.0))      # (a gate that is no number counts as the cap)
        want = g * torch.sigmoid(1.702 * g) * (1 + u.clamp(-7.0, 7.0))
    else:
        want = x * torch.sigmoid(x) * u
    rows = [0, 1, 2, 5, 8]
    # (half a unit of bfloat16, and some 1e-7 of float32 arithmetic in front of it)
    assert ((out[rows].double() - want[rows]).abs() <= 2.0 ** -8 * 1.001 * want[rows].abs() + 1e-33).all()
    assert torch.equal(out[3:5].isnan(), want[3:5].to(bf).isnan())
    for r in rows:
        assert torch.equal(run(gu[r:r + 1].contiguous())[0], out[r])


@pytest.mark.parametrize("limit", [-100.0, -60.0, -3.0, 7.0, 60.0, 100.0, math.inf])
@pytest.mark.parametrize("f", [520, 521])
def test_clamped_gates_whatever_the_limit(f, limit):
    """The cap is part of the gate that the exponential is taken of: caps on both sides of where it is taken in full, for rows of whole 16 bytes and
    for others, against float64."""
    from gibbs_amd.ops.lib import call, dtype_code, ptr, stream
    bf = torch.bfloat16
    gu = rnd(3, 2 * f, dtype=bf, scale=30.0, seed=5)
    gu[1, 3], gu[1, 70], gu[2, 9] = math.nan, math.inf, -math.inf
    out = torch.empty((3, f), dtype=bf, device=DEV)
    call("gibbs_glu_clamped", ptr(gu), ptr(out), dtype_code(bf), 3, f, 1.702, limit, stream())
    cap = torch.full((), limit, dtype=torch.float64, device=DEV)
    g = torch.fmin(gu[:, :f].double(), cap)
    want = g * torch.sigmoid(1.702 * g) * (1 + torch.minimum(torch.maximum(gu[:, f:].double(), -cap), cap))
    ok = want.isfinite()
    # (half a unit of bfloat16, some 1e-7 of float32 arithmetic in front of it, and products under the smallest float32)
    assert ((out[ok].double() - want[ok]).abs() <= 2.0 ** -8 * 1.001 * want[ok].abs() + 1e-33).all()
    assert not out[~ok].isfinite().any()


@pytest.mark.parametrize("hidden", [512, 1020, 1024, 1028, 2044, 2048, 2052, 3072, 4096, 4100])
@pytest.mark.parametrize("parts", [0, 1, 3])
@pytest.mark.parametrize("n", [5, 520])
def test_add_rmsnorm_whether_or_not_everything_is_asked_for_at_once(n, hidden, parts):
    """Around the widths that are whole threads of four elements, and the rows up to which two chunks of partial sums are asked for at once:
    the stream, the normed rows and their bits in other company, against float64."""
    from gibbs_amd import ops
    bf = torch.bfloat16
    x, gain = rnd(n, hidden, scale=2.0), 1 + 0.1 * rnd(hidden, seed=2)
    delta = None if parts == 0 else (rnd(n, hidden, dtype=bf, seed=3) if parts == 1 else rnd(parts, n, hidden, seed=3))
    v = x.double() + (0 if parts == 0 else delta.double() if parts == 1 else delta.double().sum(0))
    y, alone = x.clone(), x[2:3].clone()
    out = ops.add_rmsnorm(y, delta, gain, 1e-5, bf)
    close(y, v, torch.float32, "stream")
    close(out, v * torch.rsqrt(v.pow(2).mean(1, keepdim=True) + 1e-5) * gain.double(), bf, "normed", bf16=4e-3)
    one = None if parts == 0 else delta[2:3].contiguous() if parts == 1 else delta[:, 2:3].contiguous()
    assert torch.equal(ops.add_rmsnorm(alone, one, gain, 1e-5, bf)[0], out[2]) and torch.equal(alone[0], y[2])


@pytest.mark.parametrize("n,o,i", [(1, 1, 128), (31, 129, 192), (33, 127, 128), (64, 4100, 2048), (49, 130, 320), (64, 128, 4160)])
@pytest.mark.parametrize("out_dtype", DT)
def test_gemm_bf16_of_few_rows(n, o, i, out_dtype):
    """Around the edges of 32 and 64 rows and of 128 features, two tiles of k and many, rows of the results that are no whole 16 bytes, and nothing
    written beside them."""
    from gibbs_amd import ops
    x, w = rnd(n, i, dtype=torch.bfloat16), rnd(o, i, dtype=torch.bfloat16, seed=1)
    room = torch.full((n + 1, o + 3), 77, dtype=out_dtype, device=DEV)
    got = ops.gemm_bf16(x, w, out_dtype, out=room[:n, :o])
    close(got, x.double() @ w.double().t(), out_dtype, "few rows", f32=2e-5, bf16=4e-3)
    assert (room[n] == 77).all() and (room[:, o:] == 77).all()
    whole = ops.gemm_bf16(x, w, out_dtype)
    assert torch.equal(whole, got)
    assert torch.equal(ops.gemm_bf16(x[:1].contiguous(), w, out_dtype)[0], whole[0])


@pytest.mark.parametrize("n,f,i", [(1, 8192, 2048), (8, 200, 512), (40, 128, 72), (64, 256, 1024), (64, 6200, 256),
                                   (36, 8192, 2048),                        # two tiles a workgroup
                                   (5, 4100, 104), (8, 52, 40), (11, 4090, 72), (14, 2200, 104), (9, 60, 136)])
def test_skinny_glu(n, f, i):
    from gibbs_amd import ops
    x, w = rnd(n, i, dtype=torch.bfloat16, scale=2.0), rnd(2 * f, i, dtype=torch.bfloat16, scale=0.05, seed=1)
    gu = (x.double() @ w.double().t()) * rms_scale(x, 1e-6)
    want = F.silu(gu[:, :f]) * gu[:, f:]
    got = ops.skinny_glu(x, w, rms_eps=1e-6)
    close(got, want, torch.bfloat16, "skinny_glu", bf16=6e-3)
    assert torch.equal(ops.skinny_glu(x, ops.PackedWeight(w, groups=2), rms_eps=1e-6), got), "tile-ordered weights: same sums"
    with pytest.raises(ops.KernelError, match="row groups"):
        ops.skinny_glu(x, ops.PackedWeight(w), rms_eps=1e-6)


@pytest.mark.parametrize("n,c,i,k,bias", [(1, 2048, 2048, 3, False), (8, 72, 96, 4, True), (20, 40, 64, 2, True), (64, 96, 128, 3, False),
                                          (13, 2056, 96, 3, True), (16, 2104, 64, 4, False), (11, 40, 64, 2, True),   # 9 to 16 rows
                                          (31, 1, 512, 3, False), (2, 1, 520, 4, True)])   # one channel: sums that cancel
def test_skinny_conv(n, c, i, k, bias):
    """In-projection + convolution of decoded tokens against the unfused kernels and the reference."""
    from gibbs_amd import ops
    x = rnd(n, i, dtype=torch.bfloat16, scale=2.0)
    w = rnd(3 * c, i, dtype=torch.bfloat16, scale=0.1, seed=1)
    taps, b = rnd(c, k, seed=4), (rnd(c, seed=5) if bias else None)
    slots = torch.randperm(n + 3)[:n].to(torch.int32).to(DEV)
    ctx = i32([j % (k + 1) for j in range(n)])             # 0 (fresh), shorter than the history, longer
    state = rnd(n + 3, k - 1, c, seed=6)
    state2, state3 = state.clone(), state.clone()
    y = ops.skinny_conv(x, w, taps, b, state, slots, ctx, rms_eps=1e-5)
    y3 = ops.skinny_conv(x, ops.PackedWeight(w, groups=3), taps, b, state3, slots, ctx, rms_eps=1e-5)
    assert torch.equal(y3, y) and torch.equal(state3, state), "tile-ordered weights: same sums"
    bcx = (x.double() @ w.double().t()) * rms_scale(x, 1e-5)
    B, C, X = bcx[:, :c], bcx[:, c:2 * c], bcx[:, 2 * c:]
    bx = B * X
    want_state = state2.double().clone()
    for r in range(n):
        hist = state2[slots[r]].double().clone()
        for j in range(k - 1):
            if int(ctx[r]) - (k - 1) + j < 0:
                hist[j] = 0
        window = torch.cat([hist, bx[r:r + 1]])
        cv = (window * taps.double().t()).sum(0) + (b.double() if bias else 0)
        close(y[r], C[r] * cv, torch.bfloat16, f"skinny_conv row {r}", bf16=8e-3)
        want_state[slots[r]] = window[1:]
    # All rows' states against one scale.  The new entry B * x is a product of two float32 sums over k, whose
    # rounding error follows the size of their terms, not of the sums: with one channel, a row whose B or x
    # cancels to almost nothing has a tiny state of its own and misses a bound taken from that row alone
    # (random shapes found such rows), though every value is as exact as float32 sums get.
    close(state, want_state, torch.float32, "state", f32=2e-5)
    untouched = [s for s in range(n + 3) if s not in slots.tolist()]
    assert torch.equal(state[untouched], state2[untouched])


def test_embed_and_residual_mirror():
    from gibbs_amd import ops
    table = rnd(50, 72, dtype=torch.bfloat16)
    mirror = torch.zeros(4, 72, dtype=torch.bfloat16, device=DEV)
    x = ops.embed(table, i32([3, 49, 0, 3]), 4, mirror=mirror)
    assert torch.equal(mirror.float(), x)
    d = rnd(4, 72, dtype=torch.bfloat16, seed=3)
    x0 = x.clone()
    ops.residual_add(x, d, mirror)
    assert torch.equal(x, x0 + d.float()) and torch.equal(mirror, x.to(torch.bfloat16))
    parts = rnd(3, 4, 72, seed=4)                                      # float32 partial sums, added in order
    x1 = x.clone()
    ops.residual_add(x, parts, mirror)
    assert torch.equal(x, ((x1 + parts[0]) + parts[1]) + parts[2]) and torch.equal(mirror, x.to(torch.bfloat16))
    out = ops.add_rmsnorm(x, None, None, 1e-5, torch.bfloat16)       # no gain
    close(out, F.rms_norm(x.double(), (72,), None, 1e-5), torch.bfloat16, "gain-free norm")


@pytest.mark.parametrize("kind", ["valu", "mfma", "mfma-merge-pass"])
@pytest.mark.parametrize("n_splits,table_len,waves", [(1, 0, 8), (4, 20, 4), (None, 1024, None)])   # rows at 699 and 32 beyond a table of 20
@pytest.mark.parametrize("variant", ["half_split", "interleaved"])
@pytest.mark.parametrize("nh,nkv,hd,rot,page,window", [(4, 2, 16, 16, 16, None), (32, 8, 64, 64, 16, None), (6, 1, 48, 32, 8, None),
                                                       (5, 5, 80, 80, 32, 37), (16, 2, 128, 128, 16, None), (24, 2, 32, 32, 16, None)])
def test_attention_decode_fused(nh, nkv, hd, rot, page, window, variant, n_splits, table_len, waves, kind):
    """The fused decode attention against the separate kernels: same pages afterwards, same output,
    for rows at a page's first slot, its last slot, position 0 and far into the cache."""
    from gibbs_amd import ops
    from gibbs_amd.parts.rope import rope_inv_freq
    dtype = torch.bfloat16
    seq_lens = [700, 1, 33, 16, 17]
    kp, vp, table, ks, vs = paged_setup(dtype, nkv, hd, page, seq_lens, 120, seed=7)
    n = len(seq_lens)
    pos, row_req = i32([l - 1 for l in seq_lens]), i32(list(range(n)))
    qkv = rnd(n, (nh + 2 * nkv) * hd, dtype=dtype, seed=9)
    qg, kg = rnd(hd, seed=1) * 0.1 + 1, rnd(hd, seed=2) * 0.1 + 1
    inv = torch.from_numpy(rope_inv_freq(rot, 10000.0, "f32")).to(DEV)
    scale = 1 / math.sqrt(hd)
    kp2, vp2, qkv2 = kp.clone(), vp.clone(), qkv.clone()
    ops.qk_rope_kv(qkv2, n, nh, nkv, hd, q_gain=qg, k_gain=kg, eps=1e-6, inv_freq=inv, rotary_dim=rot, variant=variant,
                   pos=pos, row_req=row_req, kpages=kp2, vpages=vp2, table=table, n_req=n)
    want = ops.attention_decode(qkv2, n, nh, nkv, hd, kp2, vp2, table, n, pos, row_req, scale, window, max_seq=700, n_splits=3)
    kp1, vp1 = kp.clone(), vp.clone()
    got = ops.attention_decode_fused(qkv, n, nh, nkv, hd, kp1, vp1, table, n, pos, row_req, scale, q_gain=qg,
                                     k_gain=kg, eps=1e-6, inv_freq=inv, rotary_dim=rot, variant=variant,
                                     window=window, max_seq=700, n_splits=n_splits, waves=waves, kind=kind,
                                     cos_sin=ops.rope_table(inv, table_len) if table_len else None)
    close(kp1, kp2, dtype, "new keys in the pages", bf16=8e-3)
    assert torch.equal(vp1, vp2)
    close(got, want, dtype, "fused decode attention", bf16=8e-3)


@pytest.mark.parametrize("n", [1, 8, 9, 16, 33, 64])
@pytest.mark.parametrize("o,i,products,apart", [(8, 64, 3, True), (72, 200, 4, True), (520, 40, 2, False), (4104, 96, 2, True)])
def test_several_products_of_one_size_in_a_launch(n, o, i, products, apart):
    """Every product's rows as they come from a launch of their own, to the bit: matrices in either tile order, one or two tiles of rows and
    more, rows of X shared or one's behind the other's, results side by side in wider rows."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import call, ptr, stream
    x = rnd(products if apart else 1, n, i, dtype=torch.bfloat16, seed=1)
    w = rnd(products * o, i, dtype=torch.bfloat16, seed=2)
    packed = ops.PackedWeight(w, groups=products)
    y = torch.zeros(n, products * o, dtype=torch.bfloat16, device=DEV)
    call("gibbs_skinny_store_many", ptr(x), n * i if apart else 0, ptr(packed.data), products, ptr(y), o, n, o, i, i, products * o, stream())
    for p in range(products):
        rows = x[p if apart else 0].contiguous()
        assert torch.equal(y[:, p * o:(p + 1) * o], ops.skinny_store(rows, ops.PackedWeight(w[p * o:(p + 1) * o].contiguous()))), p
        # (a bfloat16 result of float32 sums)
        close(y[:, p * o:(p + 1) * o], rows.double() @ w[p * o:(p + 1) * o].double().T, torch.bfloat16, f"product {p}", bf16=8e-3)


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("n,top,experts,identity,width,inner", [(1, 1, 1, 0, 8, 8), (3, 4, 5, 2, 72, 40), (16, 4, 16, 0, 264, 520), (16, 4, 4, 0, 1024, 136),
                                                                 (8, 8, 9, 3, 256, 64)])
def test_few_rows_experts_without_grouping(n, top, experts, identity, width, inner, weighted):
    """Places are the pairs' own numbers (-1: an identity expert), and every pair's gated and returned rows have the bits that the grouped
    products give them: one pair and 64, an expert that all rows choose, experts that none does, sizes beside the tiles and the
    stretches of k."""
    from gibbs_amd.ops.lib import call, dtype_code, library, ptr, stream
    bf = torch.bfloat16
    h, router = rnd(n, width, dtype=bf, seed=1), rnd(experts + identity, width, seed=2)
    wa, wb, wd = rnd(experts, inner, width, dtype=bf, seed=3), rnd(experts, inner, width, dtype=bf, seed=4), rnd(experts, width, inner, dtype=bf, seed=5)
    pairs = n * top
    new = lambda *shape, dtype=torch.int32: torch.full(shape, 77, dtype=dtype, device=DEV)
    chosen, weight, place = new(pairs), new(pairs, dtype=torch.float32), new(pairs)
    call("gibbs_moe_route_placed", ptr(h), width, dtype_code(bf), ptr(router), None, None, ptr(chosen), ptr(weight), None, ptr(place), experts, n, width,
         experts + identity, top, 1, 1.0, stream())
    own = torch.arange(pairs, dtype=torch.int32, device=DEV)
    assert torch.equal(place, torch.where(chosen < experts, own, -torch.ones_like(own)))
    tile = 16
    cap = int(library().gibbs_moe_capacity(pairs, experts, tile))
    order, at, tiles = new(cap), new(pairs), new(cap // tile)
    call("gibbs_moe_group", ptr(chosen), pairs, experts, tile, ptr(order), ptr(at), ptr(tiles), cap, stream())
    scale = ptr(weight) if weighted else None
    grouped, direct = new(cap, inner, dtype=bf), new(pairs, inner, dtype=bf)
    call("gibbs_moe_gemm_weighted", ptr(h), width, top, ptr(order), ptr(tiles), cap, tile, ptr(wa), ptr(wb), scale, ptr(grouped), inner, dtype_code(bf), inner, width, 0, stream())
    call("gibbs_moe_gemm_direct", ptr(h), width, top, ptr(chosen), pairs, experts, ptr(wa), ptr(wb), scale, ptr(direct), inner, inner, width, 0, stream())
    has = chosen < experts
    assert torch.equal(direct[has], grouped[at[has].long()])
    back, out = new(cap, width, dtype=bf), new(pairs, width, dtype=bf)
    call("gibbs_moe_gemm", ptr(grouped), inner, 0, ptr(order), ptr(tiles), cap, tile, ptr(wd), None, ptr(back), width, dtype_code(bf), width, inner, 0, stream())
    call("gibbs_moe_gemm_direct", ptr(direct), inner, top, ptr(chosen), pairs, experts, ptr(wd), None, None, ptr(out), width, width, inner, 0, stream())
    assert torch.equal(out[has], back[at[has].long()])
    # (against float64: sums of bfloat16 products in float32, a rounding to bfloat16 at the end)
    for i in torch.nonzero(has).flatten().tolist()[:6]:
        e, x, w = int(chosen[i]), h[i // top].double(), float(weight[i]) if weighted else 1.0
        g, u = w * (wa[e].double() @ x), w * (wb[e].double() @ x)
        close(direct[i], F.silu(g) * u, bf, f"pair {i}", bf16=8e-3)


@pytest.mark.parametrize("n,top,experts,width,inner", [(2, 3, 5, 2048, 40), (16, 4, 16, 2312, 72), (7, 2, 3, 4104, 33)])
def test_few_rows_experts_begin_at_different_k(n, top, experts, width, inner):
    """Rows of 2,048 values and more, whose blocks of features begin at k of their own: against float64, and choices below 0 and beyond the
    last expert have no result."""
    from gibbs_amd.ops.lib import call, ptr, stream
    bf, pairs = torch.bfloat16, n * top
    h, wa, wb = rnd(n, width, dtype=bf, seed=1), rnd(experts, inner, width, dtype=bf, seed=2) * 0.05, rnd(experts, inner, width, dtype=bf, seed=3) * 0.05
    chosen = torch.stack([torch.randperm(experts + 1, generator=torch.Generator().manual_seed(r))[:top] for r in range(n)]).int().view(-1)
    chosen[1::5] = torch.where(chosen[1::5] < 2, torch.full_like(chosen[1::5], -1), chosen[1::5])
    chosen = chosen.to(DEV)
    gated, back = torch.full((pairs, inner), 77, dtype=bf, device=DEV), torch.full((pairs, inner), 77, dtype=bf, device=DEV)
    own = rnd(pairs, width, dtype=bf, seed=4)
    call("gibbs_moe_gemm_direct", ptr(h), width, top, ptr(chosen), pairs, experts, ptr(wa), ptr(wb), None, ptr(gated), inner, inner, width, 0, stream())
    call("gibbs_moe_gemm_direct", ptr(own), width, top, ptr(chosen), pairs, experts, ptr(wa), None, None, ptr(back), inner, inner, width, 0, stream())
    for i, e in enumerate(chosen.tolist()):
        if not 0 <= e < experts:
            assert (gated[i] == 77).all() and (back[i] == 77).all()
            continue
        x = h[i // top].double()
        # (sums of bfloat16 products in float32, a rounding to bfloat16 at the end)
        close(gated[i], F.silu(wa[e].double() @ x) * (wb[e].double() @ x), bf, f"pair {i}", bf16=8e-3)
        close(back[i], wa[e].double() @ own[i].double(), bf, f"pair {i} back", bf16=8e-3)


@pytest.mark.parametrize("n,top,experts,width,inner", [(240, 2, 8, 72, 1160), (240, 2, 8, 264, 1304), (96, 8, 64, 64, 520), (17, 4, 300, 8, 152)])
def test_gated_experts_of_many_workgroups(n, top, experts, width, inner):
    """From the line on a workgroup takes 32 features: each pair's row has the bits that 16 give it (the product without grouping of 8 rows at a time), the last
    tile of features whole or not, experts of several tiles and of none."""
    from gibbs_amd.ops.lib import call, dtype_code, library, ptr, stream
    bf, pairs, tile = torch.bfloat16, n * top, 16
    h, wa, wb = rnd(n, width, dtype=bf, seed=1), rnd(experts, inner, width, dtype=bf, seed=2), rnd(experts, inner, width, dtype=bf, seed=3)
    chosen = torch.stack([torch.randperm(max(top, experts - 1), generator=torch.Generator().manual_seed(r))[:top] for r in range(n)]).int().to(DEV)
    cap = int(library().gibbs_moe_capacity(pairs, experts, tile))
    assert int(library().gibbs_moe_gated_features(cap // tile, inner)) == 32
    new = lambda *shape, dtype=torch.int32: torch.full(shape, 77, dtype=dtype, device=DEV)
    order, at, tiles = new(cap), new(pairs), new(cap // tile)
    call("gibbs_moe_group", ptr(chosen), pairs, experts, tile, ptr(order), ptr(at), ptr(tiles), cap, stream())
    grouped = new(cap, inner, dtype=bf)
    call("gibbs_moe_gemm_weighted", ptr(h), width, top, ptr(order), ptr(tiles), cap, tile, ptr(wa), ptr(wb), None, ptr(grouped), inner, dtype_code(bf), inner, width, 0, stream())
    for r in range(0, n, 8):
        few = min(8, n - r)
        direct = new(few * top, inner, dtype=bf)
        call("gibbs_moe_gemm_direct", ptr(h[r:]), width, top, ptr(chosen[r:]), few * top, experts, ptr(wa), ptr(wb), None, ptr(direct), inner, inner, width, 0, stream())
        assert torch.equal(direct, grouped[at[r * top:(r + few) * top].long()]), r
    # (against float64: sums of bfloat16 products in float32, a rounding to bfloat16 at the end)
    for i in (0, pairs // 2, pairs - 1):
        e, x = int(chosen.view(-1)[i]), h[i // top].double()
        close(grouped[int(at[i])], F.silu(wa[e].double() @ x) * (wb[e].double() @ x), bf, f"pair {i}", bf16=8e-3)


@pytest.mark.parametrize("parts", [1, 3, 9])
@pytest.mark.parametrize("hidden", [100, 1024, 2048, 5000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_sublayers_norm_sums_its_squares_in_one_order(dtype, hidden, parts):
    """x += norm(rows): of four squares the second is rounded and the others are added to it, then come a thread's stretches, lanes by
    halves of a wave, waves in turn.  The same in float32 here, to the bit, so that a row does not depend on how its kernel was compiled; one
    stretch a thread and several, whole rows and partial sums, what follows normed or read as it is."""
    from gibbs_amd.ops.lib import call, dtype_code, ptr, stream
    n, eps = 64, 1e-6
    rows = rnd(n, hidden, dtype=dtype, seed=1) if parts == 1 else rnd(parts, n, hidden, seed=1)
    x0, gain, gain_n = rnd(n, hidden, seed=2), rnd(hidden, seed=3), rnd(hidden, seed=4)
    f32, f64 = np.float32, np.float64
    fused = lambda a, b, c: (a.astype(f64) * b.astype(f64) + c.astype(f64)).astype(f32)
    v = np.zeros((n, hidden), f32)
    for part in (rows.float().view(-1, n, hidden).cpu().numpy()):
        v = v + part
    threads = 1024 if hidden >= 4096 else 512 if hidden >= 2048 else 256 if hidden >= 512 else 64
    stretches = -(-hidden // (4 * threads))
    four = np.zeros((n, stretches * threads * 4), f32)
    four[:, :hidden] = v
    a, b, c, d = np.moveaxis(four.reshape(n, stretches, threads, 4), 3, 0)
    squares = fused(d, d, fused(c, c, fused(a, a, b * b)))
    lanes = np.zeros((n, threads), f32)
    for s in range(stretches):
        lanes = lanes + squares[:, s]
    lanes = lanes.reshape(n, -1, 64)
    for half in (32, 16, 8, 4, 2, 1):
        lanes = lanes + lanes[:, :, np.arange(64) ^ half]
    total = np.zeros(n, f32)
    for w in range(lanes.shape[1]):
        total = total + lanes[:, w, 0]
    scale = (f32(1) / np.sqrt(total / f32(hidden) + f32(eps)))[:, None]
    want = torch.from_numpy(fused(v * scale, gain.cpu().numpy()[None], x0.cpu().numpy()))
    x, out = x0.clone(), torch.empty(n, hidden, dtype=dtype, device=DEV)
    call("gibbs_rmsnorm_rows_add_norm", ptr(x), ptr(rows), parts, n * hidden, ptr(gain), eps, ptr(gain_n), eps, ptr(out), dtype_code(dtype), n, hidden, stream())
    assert torch.equal(x.cpu(), want)
    x = x0.clone()
    call("gibbs_rmsnorm_rows_add_read", ptr(x), ptr(rows), parts, n * hidden, None, None, 0, None, None, ptr(gain), eps, 1, None, None, 0, None, ptr(out),
         dtype_code(dtype), n, hidden, stream())
    assert torch.equal(x.cpu(), want)
    assert torch.equal(out.cpu(), want.to(dtype))


@pytest.mark.parametrize("parts", [0, 1, 3])
@pytest.mark.parametrize("hidden", [4, 516, 2048, 5000])
def test_norm_that_leaves_a_mirror(hidden, parts):
    """x, the normed rows and x in bfloat16 in one kernel: the bits of the two that it stands for."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import call, dtype_code, ptr, stream
    n = 5
    x, gain = rnd(n, hidden, seed=1), rnd(hidden, seed=2)
    delta = None if parts == 0 else rnd(n, hidden, dtype=torch.bfloat16, seed=3) if parts == 1 else rnd(parts, n, hidden, seed=3)
    x1, out, mirror = x.clone(), torch.empty(n, hidden, dtype=torch.bfloat16, device=DEV), torch.empty(n, hidden, dtype=torch.bfloat16, device=DEV)
    want = ops.add_rmsnorm(x, delta, gain, 1e-5, torch.bfloat16)
    call("gibbs_add_rmsnorm_mirror", ptr(x1), ptr(delta), parts, n * hidden, ptr(gain), 1e-5, ptr(out), ptr(mirror), dtype_code(torch.bfloat16), n, hidden, stream())
    assert torch.equal(x1, x) and torch.equal(out, want) and torch.equal(mirror, x.to(torch.bfloat16))


@pytest.mark.parametrize("raw", [False, True])
@pytest.mark.parametrize("n_splits,waves", [(1, 4), (1, 8), (5, 4), (None, None)])
@pytest.mark.parametrize("nh,nkv,hd,page,window", [(2, 2, 64, 16, None), (4, 2, 64, 64, 33), (8, 1, 64, 16, 700), (1, 1, 128, 16, None),
                                                   (4, 2, 128, 32, 70), (8, 1, 128, 16, 31)])
def test_attention_decode_in_tiles(nh, nkv, hd, page, window, n_splits, waves, raw):
    """Heads of 64 and 128 in groups of 1 to 8, rows that end on either side of a tile of 32 keys and of a page, a row of more tiles than
    a wave holds page ids for (4,400 keys are 138 tiles: 35 a wave), windows that begin inside a tile; in the pages, everything
    that no row may see is NaN.  Raw rows also at positions behind the table of rotation factors."""
    from gibbs_amd import ops
    from gibbs_amd.parts.rope import rope_inv_freq
    dtype = torch.bfloat16
    seq_lens = [4400, 1, 16, 17, 32, 33, 96, 97]
    n = len(seq_lens)
    kp, vp, table, ks, vs = paged_setup(dtype, nkv, hd, page, seq_lens, 320, seed=13)
    kp[kp == 50], vp[vp == -50] = float("nan"), float("nan")
    pos = i32([l - 1 for l in seq_lens])
    scale = 1 / math.sqrt(hd)
    qkv = rnd(n, (nh + 2 * nkv) * hd, dtype=dtype, seed=9)
    if raw:
        inv = torch.from_numpy(rope_inv_freq(hd, 10000.0, "f32")).to(DEV)
        gains = rnd(hd, seed=1) * 0.1 + 1, rnd(hd, seed=2) * 0.1 + 1
        kp2, vp2, q = kp.clone(), vp.clone(), qkv.clone()
        ops.qk_rope_kv(q, n, nh, nkv, hd, q_gain=gains[0], k_gain=gains[1], eps=1e-6, inv_freq=inv, rotary_dim=hd, variant="half_split", pos=pos,
                       row_req=i32(list(range(n))), kpages=kp2, vpages=vp2, table=table, n_req=n)
        out = ops.attention_decode_fused(qkv, n, nh, nkv, hd, kp, vp, table, n, pos, i32(list(range(n))), scale, q_gain=gains[0], k_gain=gains[1], eps=1e-6,
                                         inv_freq=inv, rotary_dim=hd, variant="half_split", window=window, max_seq=4400, n_splits=n_splits, waves=waves,
                                         cos_sin=ops.rope_table(inv, 33))
        for r, l in enumerate(seq_lens):      # the new keys and values, and nothing else in the pages
            pg = table[r, (l - 1) // page].item()
            ks[r][l - 1], vs[r][l - 1] = kp2[pg, :, (l - 1) % page], vp2[pg, :, (l - 1) % page]
        close(kp.nan_to_num(0), kp2.nan_to_num(0), dtype, "new keys in the pages", bf16=8e-3)
        assert torch.equal(vp.nan_to_num(7), vp2.nan_to_num(7))
    else:
        q = qkv
        out = ops.attention_decode(q, n, nh, nkv, hd, kp, vp, table, n, pos, None, scale, window, max_seq=4400, n_splits=n_splits, waves=waves)
    for r, l in enumerate(seq_lens):
        want = attention_reference(q[r:r + 1, :nh * hd].view(1, nh, hd), ks[r], vs[r], [l - 1], scale, window)
        # (the weights and the output are bfloat16: 2^-9 of the largest value each, and 2^-8 for a raw row's keys and queries)
        close(out[r].view(1, nh, hd), want, dtype, f"row of {l} keys", bf16=1e-2)


@pytest.mark.parametrize("n_splits,waves,kind", [(1, 4, 0), (1, 8, 0), (3, 8, 4), (5, 4, 2)])
@pytest.mark.parametrize("nh,nkv,hd,page", [(2, 2, 64, 16), (4, 2, 64, 64), (8, 2, 64, 16), (8, 1, 64, 32), (1, 1, 128, 16), (4, 2, 128, 32), (8, 1, 128, 16)])
@pytest.mark.parametrize("what", ["raw", "plain", "bias", "sink", "capped", "chunk", "all", "short chunk"])
def test_tiles_give_the_bits_of_the_general_decode_kernel(nh, nkv, hd, page, n_splits, waves, kind, what):
    """A row's keys are shared out over slices and waves, and their results folded, as in the kernel for any shape (which output rows of
    an odd stride reach), so that a model's rows do not depend on which of the two takes a call.  Rows on either side of a tile and of a page,
    one of more tiles than a wave holds page ids for; what no row sees is NaN.  Prepared rows with a bias whose table ends before the row's
    keys do, a sink, capped scores and chunks, each also against float64 (a chunk inside which tiles do not begin: against that alone)."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import call, ptr, stream
    from gibbs_amd.parts.rope import rope_inv_freq
    bf = torch.bfloat16
    seq_lens = [4400, 1, 31, 32, 33, 96, 97, 1029]
    n, raw = len(seq_lens), what == "raw"
    kp, vp, table, ks, vs = paged_setup(bf, nkv, hd, page, seq_lens, 400, seed=3)
    kp[kp == 50], vp[vp == -50] = float("nan"), float("nan")
    pos = i32([l - 1 for l in seq_lens])
    scale = 1 / math.sqrt(hd)
    qkv = rnd(n, (nh + 2 * nkv) * hd, dtype=bf, seed=9)
    every = what == "all"
    bias = rnd(nh, 300, seed=4) / scale if what == "bias" or every else None
    sink = rnd(nh, seed=5) if what == "sink" or every else None
    softcap = 2.0 if what == "capped" or every else 0.0
    chunk = {"chunk": 1024, "all": 96, "short chunk": 180}.get(what, 0)
    inv = torch.from_numpy(rope_inv_freq(hd, 10000.0, "f32")).to(DEV)
    gains, factors = (rnd(hd, seed=1) * 0.1 + 1, rnd(hd, seed=2) * 0.1 + 1), ops.rope_table(inv, 1000)

    def run(ldo):
        out, k, v = torch.zeros(n, ldo, dtype=bf, device=DEV), kp.clone(), vp.clone()
        partial = torch.empty(n * nh * n_splits * (hd + 2), device=DEV)
        cache = (ptr(table), table.shape[1], page, kp.shape[0], n, nh, nkv, hd, qkv.shape[1], ldo, scale, 0, n_splits, waves, kind, 4400)
        if raw:
            call("gibbs_attention_decode_fused", ptr(qkv), ptr(k), ptr(v), ptr(out), ptr(partial), ptr(gains[0]), ptr(gains[1]), 1e-6, ptr(inv), hd, 0,
                 ptr(factors), 1000, ptr(pos), None, *cache, stream())
        else:
            call("gibbs_attention_decode_masked", ptr(qkv), ptr(k), ptr(v), ptr(out), ptr(partial), ptr(pos), None, *cache, ptr(bias), 300, ptr(sink), chunk,
                 softcap, stream())
        return out[:, :nh * hd], k, v

    got, general = run(nh * hd), run(nh * hd + 1)
    if chunk % 32 == 0:
        for a, b in zip(got, general):
            assert torch.equal(a.nan_to_num(7.0), b.nan_to_num(7.0))
    if raw:
        return
    for r, l in enumerate(seq_lens):
        lo = (l - 1) // chunk * chunk if chunk else 0
        kk, vv = (x[r][lo:].double().repeat_interleave(nh // nkv, 1) for x in (ks, vs))
        s = torch.einsum("hd,lhd->hl", qkv[r, :nh * hd].view(nh, hd).double(), kk) * scale
        s = softcap * torch.tanh(s / softcap) if softcap else s
        if bias is not None:
            s = s + bias.double()[:, (l - 1 - torch.arange(lo, l, device=DEV)).clamp(max=299)] * scale
        if sink is not None:
            s = torch.cat([s, sink.double()[:, None]], 1)
        want = torch.einsum("hl,lhd->hd", s.softmax(-1)[:, :l - lo], vv)
        # (the weights and the output are bfloat16: 2^-9 of the largest value each)
        close(got[0][r].view(nh, hd), want, bf, f"row of {l} keys", bf16=8e-3)


@pytest.mark.parametrize("gained", [False, True])
@pytest.mark.parametrize("nh,nkv,hd", [(32, 8, 64), (16, 8, 64), (8, 1, 64), (4, 4, 128), (16, 2, 128)])
def test_tiles_rotate_to_the_bit_as_the_general_decode_kernel(nh, nkv, hd, gained):
    """Enough rotated queries and keys that another rounding inside a rotation (which of its two products is rounded before the sum) shows in
    the bfloat16 keys in the pages and in the outputs: it moves one value in some 10,000."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import call, ptr, stream
    from gibbs_amd.parts.rope import rope_inv_freq
    bf, rows, page, keys = torch.bfloat16, 512, 16, 48
    inv = torch.from_numpy(rope_inv_freq(hd, 10000.0, "f32")).to(DEV)
    gains = (rnd(hd, seed=1) * 0.1 + 1, rnd(hd, seed=2) * 0.1 + 1) if gained else (None, None)
    factors = ops.rope_table(inv, keys)
    pages = rows * keys // page
    kp, vp = rnd(pages, nkv, page, hd, dtype=bf, seed=3), rnd(pages, nkv, page, hd, dtype=bf, seed=4)
    table = torch.arange(pages, dtype=torch.int32, device=DEV).view(rows, -1)
    pos = i32([5 + r % (keys - 5) for r in range(rows)])
    qkv = rnd(rows, (nh + 2 * nkv) * hd, dtype=bf, seed=5)

    def run(ldo):
        out, k, v = torch.zeros(rows, ldo, dtype=bf, device=DEV), kp.clone(), vp.clone()
        call("gibbs_attention_decode_fused", ptr(qkv), ptr(k), ptr(v), ptr(out), None, ptr(gains[0]), ptr(gains[1]), 1e-6, ptr(inv), hd, 0, ptr(factors), keys,
             ptr(pos), None, ptr(table), table.shape[1], page, pages, rows, nh, nkv, hd, qkv.shape[1], ldo, hd ** -0.5, 0, 1, 4, 0, keys, stream())
        return out[:, :nh * hd], k, v

    for a, b in zip(run(nh * hd), run(nh * hd + 1)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("rows,nh,nkv,max_seq,kind", [(32, 32, 8, 8192, "auto"), (64, 16, 4, 10368, "auto"), (16, 8, 8, 16384, "auto"), (64, 8, 8, 16384, "mfma")])
def test_decode_attention_of_many_rows_under_a_far_bound(rows, nh, nkv, max_seq, kind):
    """Rows that fill the chip, under a bound on their keys beyond the page ids that one slice has room for: a bias on the scores, and the matrix
    cores asked for, are taken with the slices of the rule.  (Rows share their pages: only the bound has to be far.)"""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import call, ptr, stream
    bf, hd, page, keys = torch.bfloat16, 64, 16, 300
    kp, vp, one, ks, vs = paged_setup(bf, nkv, hd, page, [keys], 24, seed=5)
    table = torch.zeros(rows, max_seq // page, dtype=torch.int32, device=DEV)
    table[:, :one.shape[1]] = one
    pos = i32([(keys - 1) if r % 2 else r for r in range(rows)])
    q, scale = rnd(rows, nh * hd, dtype=bf, seed=6), 0.125
    bias = rnd(nh, 64, seed=7) / scale if kind == "auto" else None
    n_splits, waves = ops.decode_splits(rows, nkv, nh // nkv, max_seq, hd, kind, page)
    partial = torch.empty(max(1, ops.slices_workspace(rows, nh, hd, n_splits)), device=DEV)
    out = torch.zeros(rows, nh * hd, dtype=bf, device=DEV)
    call("gibbs_attention_decode_masked", ptr(q), ptr(kp), ptr(vp), ptr(out), ptr(partial), ptr(pos), None, ptr(table), table.shape[1], page, kp.shape[0],
         rows, nh, nkv, hd, nh * hd, nh * hd, scale, 0, n_splits, waves, ops.DECODE_KINDS[kind], max_seq, ptr(bias), 64, None, 0, 0.0, stream())
    kk, vv = ks[0].double().repeat_interleave(nh // nkv, 1), vs[0].double().repeat_interleave(nh // nkv, 1)
    for r in range(rows):
        p = pos[r].item()
        s = torch.einsum("hd,lhd->hl", q[r].view(nh, hd).double(), kk[:p + 1]) * scale
        if bias is not None:
            s = s + bias.double()[:, (p - torch.arange(p + 1, device=DEV)).clamp(max=63)] * scale
        # (the weights and the output are bfloat16: 2^-9 of the largest value each)
        close(out[r].view(nh, hd), torch.einsum("hl,lhd->hd", s.softmax(-1), vv[:p + 1]), bf, f"row {r}", bf16=8e-3)


@pytest.mark.parametrize("n_rows,nh,nkv,hd,n_splits", [(64, 32, 8, 64, 8), (3, 6, 2, 48, 5), (2, 4, 1, 128, 40),
                                                       (4200, 8, 8, 16, 2)])
def test_slices_merged_by_the_last_to_finish_or_by_a_second_kernel(n_rows, nh, nkv, hd, n_splits):
    """The key slices of a row are merged by the workgroup that finishes last, through memory that the other
    workgroups wrote in the same kernel; a second kernel does the same arithmetic where it is asked for, or where
    rows x groups of heads exceed the counters (4,200 x 8).  Up to 8 slices both add in the same order: the results
    are equal bit for bit, call after call (the counters are left at zero, no partial result is read before it has
    arrived); beyond 8 they differ by rounding."""
    from gibbs_amd import ops
    dtype, page = torch.bfloat16, 16
    long_rows = n_rows <= 64
    seq_lens = [(900 + 37 * r) if long_rows else 20 + r % 13 for r in range(n_rows)]
    kp, vp, table, ks, vs = paged_setup(dtype, nkv, hd, page, seq_lens, sum(-(-l // page) for l in seq_lens) + 8, seed=3)
    pos = i32([l - 1 for l in seq_lens])
    scale = 1 / math.sqrt(hd)
    # (other queries in every call: a partial result left over from the call before would show)
    for call in range(12 if long_rows else 2):
        qc = rnd(n_rows, nh * hd, dtype=dtype, seed=4 + call) * (1 + call % 3)
        got = ops.attention_decode(qc, n_rows, nh, nkv, hd, kp, vp, table, n_rows, pos, None, scale, None,
                                   max_seq=max(seq_lens), n_splits=n_splits, waves=4, kind="mfma")
        want = ops.attention_decode(qc, n_rows, nh, nkv, hd, kp, vp, table, n_rows, pos, None, scale, None,
                                    max_seq=max(seq_lens), n_splits=n_splits, waves=4, kind="mfma-merge-pass")
        if n_splits <= 8:
            assert torch.equal(got, want), f"call {call}"
        else:
            close(got, want, dtype, f"merged in the kernel, call {call}", bf16=4e-3)
        for r in range(min(n_rows, 3)):
            ref = attention_reference(qc[r:r + 1].view(1, nh, hd), ks[r], vs[r], [seq_lens[r] - 1], scale, None)
            close(got[r].view(1, nh, hd), ref, dtype, f"row {r}, call {call}", bf16=1e-2)


def test_attention_block_table_segments():
    """Requests with more pages than the kernels keep in LDS at a time (pages of 2 tokens, 2,300
    keys): the fast kernels cross from one segment of the block table to the next."""
    from gibbs_amd import ops
    from gibbs_amd.parts.rope import rope_inv_freq
    dtype, nh, nkv, hd, page = torch.bfloat16, 2, 1, 32, 2
    seq_lens = [2300, 1100]
    kp, vp, table, ks, vs = paged_setup(dtype, nkv, hd, page, seq_lens, 1800, seed=5)
    scale = 1 / math.sqrt(hd)
    # prompt portions ending at the last key of each request
    q_lens = [130, 70]
    ctx = [s - q for s, q in zip(seq_lens, q_lens)]
    cu = np.concatenate([[0], np.cumsum(q_lens)])
    n = int(cu[-1])
    q = rnd(n, nh * hd, dtype=dtype, seed=9)
    out = ops.attention_prefill(q, n, nh, nkv, hd, kp, vp, table, 2, i32(cu), i32(ctx), scale)
    for r in range(2):
        rows = slice(int(cu[r]), int(cu[r + 1]))
        want = attention_reference(q[rows].view(-1, nh, hd), ks[r], vs[r], list(range(ctx[r], seq_lens[r])), scale, None)
        close(out[rows].view(-1, nh, hd), want, dtype, f"prefill over segments, request {r}", bf16=1e-2)
    # decoded rows at the last positions, one key slice and several
    pos, row_req = i32([l - 1 for l in seq_lens]), i32([0, 1])
    qd = rnd(2, nh * hd, dtype=dtype, seed=3)
    want = ops.attention_plain(qd, 2, nh, nkv, hd, kp, vp, table, 2, pos, row_req, scale)
    for ns in (1, 3):
        close(ops.attention_decode(qd, 2, nh, nkv, hd, kp, vp, table, 2, pos, row_req, scale, n_splits=ns), want, dtype,
              f"decode over segments, {ns} slices", bf16=1e-2)
        qkv = torch.cat([qd, rnd(2, 2 * nkv * hd, dtype=dtype, seed=4)], dim=1).contiguous()
        kp1, vp1, kp2, vp2, qkv2 = kp.clone(), vp.clone(), kp.clone(), vp.clone(), qkv.clone()
        ops.qk_rope_kv(qkv2, 2, nh, nkv, hd, q_gain=None, k_gain=None, eps=0.0, inv_freq=None, rotary_dim=0,
                       variant="half_split", pos=pos, row_req=row_req, kpages=kp2, vpages=vp2, table=table, n_req=2)
        ref = ops.attention_plain(qkv2, 2, nh, nkv, hd, kp2, vp2, table, 2, pos, row_req, scale)
        got = ops.attention_decode_fused(qkv, 2, nh, nkv, hd, kp1, vp1, table, 2, pos, row_req, scale, q_gain=None,
                                         k_gain=None, eps=0.0, inv_freq=None, rotary_dim=0, variant="half_split",
                                         n_splits=ns)
        close(got, ref, dtype, f"fused decode over segments, {ns} slices", bf16=1e-2)


def test_decode_tail_one_kernel():
    """The end of a captured decode step: next tokens (first largest logit, NaN never wins), the log, positions,
    cached lengths, draws and per-row step counts, and the tokens' embeddings as the next step's rows."""
    from gibbs_amd import ops
    n, V, hidden, cap = 5, 1001, 72, 4
    logits = rnd(n, V, seed=3)
    logits[1, 7] = logits[1, 900] = 50.0           # a tie: the first wins
    logits[2, 3] = float("nan")
    table = rnd(V, hidden, dtype=torch.bfloat16, seed=4)
    ids, pos, ctx = i32([9] * n), i32([10, 20, 30, 40, 50]), i32([10, 20, 30, 40, 50])
    log, steps = torch.full((cap, n), -1, dtype=torch.int32, device=DEV), i32([0, 1, 2, 3, 4])
    u, u_all = torch.zeros(n, device=DEV), rnd(cap, n, seed=5)
    x, mirror = torch.zeros(n, hidden, device=DEV), torch.zeros(n, hidden, dtype=torch.bfloat16, device=DEV)
    ops.decode_tail(logits, ids, pos, ctx, log, steps, u, u_all, n, table, x, mirror)
    want = torch.nan_to_num(logits, nan=-float("inf")).argmax(-1).int()
    want[1] = 7
    assert torch.equal(ids, want) and pos.tolist() == [11, 21, 31, 41, 51] and ctx.tolist() == pos.tolist()
    assert steps.tolist() == [1, 2, 3, 4, 5]
    for r in range(n):
        assert [int(log[s, r]) for s in range(cap)] == [int(want[r]) if s == r else -1 for s in range(cap)]   # row 4: beyond the log
        assert float(u[r]) == (float(u_all[r + 1, r]) if r + 1 < cap else 0.0)
    assert torch.equal(x, table[want.long()].float()) and torch.equal(mirror, table[want.long()])
    # tokens that a sampling kernel has put into ids; no embedding asked for
    ids2, steps2 = i32([4, 3, 2, 1, 0]), i32([0] * n)
    ops.decode_tail(None, ids2, pos, ctx, log, steps2, None, None, n)
    assert log[0].tolist() == [4, 3, 2, 1, 0] and pos.tolist() == [12, 22, 32, 42, 52] and ids2.tolist() == [4, 3, 2, 1, 0]


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh", "gelu", "relu"])
def test_activations_of_the_gated_kernels(dtype, activation):
    """The activation table in the stand-alone kernel (both precisions, vector and scalar variants) and in the
    epilogue of the fused decode product."""
    from gibbs_amd import ops
    act = {"silu": F.silu, "gelu_tanh": lambda g: F.gelu(g, approximate="tanh"), "gelu": F.gelu, "relu": F.relu}[activation]
    for f in (200, 203):
        gu = rnd(7, 2 * f, dtype=dtype, scale=2.0, seed=f)
        close(ops.glu(gu, activation), act(gu[:, :f].double()) * gu[:, f:].double(), dtype, f"glu {activation} {f}")
    if dtype == torch.bfloat16:
        x = rnd(5, 96, dtype=dtype, seed=1)
        w = rnd(2 * 48, 96, dtype=dtype, scale=0.2, seed=2)
        want = act(x.double() @ w[:48].double().T) * (x.double() @ w[48:].double().T)
        close(ops.skinny_glu(x, w, activation=activation), want, dtype, f"skinny_glu {activation}")
    with pytest.raises(ops.KernelError, match="not implemented"):
        ops.glu(rnd(2, 8, dtype=dtype), "softsign")


@pytest.mark.parametrize("dtype", DT)
def test_attention_plain_with_score_slopes(dtype):
    """A linear bias on the scores by distance: slope[h] * (key position - query position)."""
    from gibbs_amd import ops
    nh, nkv, hd, page = 6, 2, 32, 8
    seq_lens = [70, 9]
    kp, vp, table, ks, vs = paged_setup(dtype, nkv, hd, page, seq_lens, 24, seed=3)
    rows = [(0, list(range(60, 70))), (1, [8])]
    pos, row_req = i32([p for _, ps in rows for p in ps]), i32([r for r, ps in rows for _ in ps])
    n = pos.numel()
    q = rnd(n, nh * hd, dtype=dtype, seed=9)
    slopes = torch.tensor([0.5 ** (h + 1) for h in range(nh)], dtype=torch.float32, device=DEV)
    out = ops.attention_plain(q, n, nh, nkv, hd, kp, vp, table, 2, pos, row_req, hd ** -0.5, slopes=slopes)
    at = 0
    for r, ps in rows:
        kk, vv = ks[r].double().repeat_interleave(nh // nkv, 1), vs[r].double().repeat_interleave(nh // nkv, 1)
        for i, p in enumerate(ps):
            s = torch.einsum("hd,lhd->hl", q[at + i].double().view(nh, hd), kk[:p + 1]) * hd ** -0.5
            s = s + slopes.double()[:, None] * (torch.arange(p + 1, device=DEV) - p)[None, :]
            want = torch.einsum("hl,lhd->hd", s.softmax(-1), vv[:p + 1])
            close(out[at + i].view(nh, hd), want, dtype, f"slopes request {r} position {p}", f32=2e-5, bf16=1e-2)
        at += len(ps)
