"""Row-invariant linear layer (sd_linear) and RMSNorm (sd_rms_norm) on the GPU.

Bar: the linear layer's outputs are the bf16 rounding of fp32 dot products (within one bf16 unit of the float64
dot product plus the fp32 accumulation bound, at least 99.9 % equal to it rounded: the library GEMM's
contract); the norm's residual output is bit-exact against the oracle (layernorm.py:28-38) and its normalised
output differs from the oracle only by the order of the sum of squares (at least 99.5 % bit-exact, the rest
within one bf16 unit). Both give bitwise the same row whatever the number of rows in the call, which the
library GEMM (o_proj, gate_up_proj and down_proj shapes) and reductions do not.
"""
import pytest
import torch

from nanovllm_amd.layers.activation import silu_and_mul
from nanovllm_amd.layers.layernorm import RMSNorm, rms_norm
from nanovllm_amd.layers.linear import RowInvariantLinear
from oracle import qk_norm_rope as onr

pytestmark = pytest.mark.gpu

QWEN3_8B = [("qkv_proj", 4096, 6144), ("o_proj", 4096, 4096), ("gate_up_proj", 4096, 24576),
            ("down_proj", 12288, 4096)]


def _ulp_bf16(x: torch.Tensor) -> torch.Tensor:
    a = x.abs().float().clamp_min(2.0 ** -126)
    return torch.exp2(torch.floor(torch.log2(a)) - 7)


def _check_rows(x, w, y, rows):
    xd, wd = x.cpu().double()[rows], w.cpu().double()
    ref = xd @ wd.T
    mag = xd.abs() @ wd.abs().T
    ours = y.cpu()[rows].double()
    bound = _ulp_bf16(ref.float()).double() + x.size(1) * 2.0 ** -24 * mag
    worst = ((ours - ref).abs() / bound).max().item()
    exact = (ours.float() == ref.float().to(torch.bfloat16).float()).float().mean().item()
    print(f"vs float64: worst {worst:.3f} of the bound, {exact * 100:.3f} % equal to the rounded float64", flush=True)
    assert worst <= 1.0 and exact >= 0.999


@pytest.mark.parametrize("M,N,K", [(5, 1000, 256), (70, 2053, 192), (330, 6144, 4096), (64, 4096, 12288),
                                   (1300, 4096, 12288), (700, 2053, 192)])
def test_linear_vs_float64(device, M, N, K):
    g = torch.Generator(device=device).manual_seed(M + N)
    x = torch.randn(M, K, device=device, generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device=device, generator=g) * K ** -0.5).to(torch.bfloat16)
    y = RowInvariantLinear(w)(x)
    _check_rows(x, w, y, list(range(0, M, max(1, M // 6))) + [M - 1])


# 300 tiles: 256 of one range of k and 44 of five, unequal ones of S / 5 steps
@pytest.mark.parametrize("name,K,N", QWEN3_8B + [("partly_split", 128, 76800)])
def test_linear_rows_independent_of_row_count(device, name, K, N):
    g = torch.Generator(device=device).manual_seed(K + N)
    x = torch.randn(2048, K, device=device, generator=g).to(torch.bfloat16)
    lin = RowInvariantLinear((torch.randn(N, K, device=device, generator=g) * K ** -0.5).to(torch.bfloat16))
    probes = [0, 1, 63, 127, 128, 319, 320, 1000, 1215, 2047]
    alone = {r: lin(x[r:r + 1]) for r in probes}    # each row in a call of its own
    for M in (2, 16, 64, 80, 320, 325, 1216, 2048):
        y = lin(x[:M])
        for r in probes:
            if r < M:
                assert torch.equal(y[r:r + 1], alone[r]), f"{name}: row {r} differs at {M} rows"
    # a strided input (a column slice of a wider buffer) gives the same rows
    wide = torch.zeros(64, K + 64, dtype=torch.bfloat16, device=device)
    wide[:, :K] = x[:64]
    assert torch.equal(lin(wide[:, :K]), lin(x[:64]))


def test_linear_vs_library_gemm(device):
    g = torch.Generator(device=device).manual_seed(3)
    x = torch.randn(320, 4096, device=device, generator=g).to(torch.bfloat16)
    w = (torch.randn(6144, 4096, device=device, generator=g) * 4096 ** -0.5).to(torch.bfloat16)
    ours, lib = RowInvariantLinear(w)(x), torch.nn.functional.linear(x, w)
    same = (ours == lib).float().mean().item()
    big = ((ours.float() - lib.float()).abs() > _ulp_bf16(torch.maximum(ours.float().abs(), lib.float().abs())) + 1e-3)
    print(f"vs F.linear: {same * 100:.3f} % identical", flush=True)
    assert same >= 0.99 and int(big.sum()) == 0


@pytest.mark.parametrize("H", [4096, 1024, 1000, 12288])
def test_rms_norm_vs_oracle(device, H):
    g = torch.Generator().manual_seed(H)
    x = (torch.randn(37, H, generator=g) * 2).to(torch.bfloat16)
    r = torch.randn(37, H, generator=g).to(torch.bfloat16)
    w = (1 + 0.1 * torch.randn(H, generator=g)).to(torch.bfloat16)
    for residual in (None, r):
        if residual is None:
            got = rms_norm(x.to(device), w.to(device), 1e-6).cpu()
            want = onr.rms_norm(x, w, 1e-6)
        else:
            got, got_res = (t.cpu() for t in rms_norm(x.to(device), w.to(device), 1e-6, residual.to(device)))
            want, want_res = onr.add_rms_norm(x, residual, w, 1e-6)
            assert torch.equal(got_res, want_res)
        same = (got == want).float().mean().item()
        diff = (got.float() - want.float()).abs()
        assert same >= 0.995 and bool((diff <= _ulp_bf16(want.float())).all()), (same, float(diff.max()))


def test_rms_norm_rows_independent_of_row_count_and_in_place(device):
    H = 4096
    g = torch.Generator(device=device).manual_seed(9)
    x = torch.randn(2048, H, device=device, generator=g).to(torch.bfloat16)
    r = torch.randn(2048, H, device=device, generator=g).to(torch.bfloat16)
    norm = RMSNorm(H).to(device)
    norm.weight.data = (1 + 0.1 * torch.randn(H, device=device, generator=g)).to(torch.bfloat16)
    first, first_res = norm(x[:1], r[:1])
    for M in (16, 64, 320, 2048):
        out, res = norm(x[:M], r[:M])
        assert torch.equal(out[:1], first) and torch.equal(res[:1], first_res)
    # in place: out over x, the new residual over the old one (as a fused residual stream uses it)
    xi, ri = x[:64].clone(), r[:64].clone()
    want_out, want_res = norm(x[:64], r[:64])
    rms_norm(xi, norm.weight.data, norm.eps, ri, out=xi, residual_out=ri)
    assert torch.equal(xi, want_out) and torch.equal(ri, want_res)


# Edges of the row-invariant GEMM's kernels (which sizes run which is sd_linear_kernel's answer; test_capi.py checks that
# each kernel is among these with its main loop, steps left behind it and a half stage): rows one short of, at and past
# the workgroups' rows, columns that are no multiple of the two-step stages or of the steps ahead, weight rows that end
# inside a tile and inside a store of four, outputs at aligned rows and at unaligned ones.
EDGES = [(1000, 32), (515, 96), (2053, 160), (4096, 544), (6150, 256), (24576, 64), (4096, 1056), (6150, 1056),
         (12290, 1056), (24579, 1056), (49155, 1056), (131075, 544), (4098, 4096)]
EDGE_ROWS = (15, 16, 17, 63, 64, 65, 79, 80, 81, 128, 159, 160, 161, 255, 256, 257, 300, 640, 1100)


# Every row equals its row in calls of at most 16 rows (bitwise), and some of those the float64 product within the bound.
@pytest.mark.parametrize("N,K", EDGES)
def test_linear_kernel_edges(device, N, K):
    g = torch.Generator(device=device).manual_seed(N + K)
    x = torch.randn(1100, K, device=device, generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device=device, generator=g) * K ** -0.5).to(torch.bfloat16)
    lin = RowInvariantLinear(w)
    want = torch.cat([lin(x[r:r + 16]) for r in range(0, 1100, 16)])
    part = slice(0, N) if N < 30000 else slice(N - 2000, N)
    _check_rows(x, w[part], want[:, part], [0, 15, 16, 1099])
    for M in EDGE_ROWS:
        print(f"M={M} N={N} K={K}", flush=True)
        assert torch.equal(lin(x[:M]), want[:M]), f"{M} rows"
        wide = torch.full((M, N + 3), 7.0, dtype=torch.bfloat16, device=device)   # rows not 8-byte aligned
        assert torch.equal(lin(x[:M], out=wide[:, 1:1 + N]), want[:M]), f"{M} rows"
        assert bool((wide[:, 0] == 7).all()) and bool((wide[:, 1 + N:] == 7).all())


# The same bits wherever the output's rows start: multiples of 16, 8 and 2 bytes (a store of 8, 4 and 1 entries), at
# every kernel, a weight that ends inside a store and nothing written beside the rows.
@pytest.mark.parametrize("N,K", [(1003, 96), (4094, 544), (24577, 64), (6144, 256)])
def test_linear_output_alignment(device, N, K):
    g = torch.Generator(device=device).manual_seed(N)
    x = torch.randn(600, K, device=device, generator=g).to(torch.bfloat16)
    lin = RowInvariantLinear((torch.randn(N, K, device=device, generator=g) * K ** -0.5).to(torch.bfloat16))
    width = -(-(N + 16) // 8) * 8
    for M in (3, 16, 40, 80, 160, 300, 600):
        want = lin(x[:M])
        for at, row in ((8, width), (4, width), (8, width + 4), (4, width + 4), (2, width), (3, width + 1)):
            print(f"M={M} N={N} K={K} offset {at} row {row}", flush=True)
            buf = torch.full((M, row), 7.0, dtype=torch.bfloat16, device=device)
            lin(x[:M], out=buf[:, at:at + N])
            assert torch.equal(buf[:, at:at + N], want)
            assert bool((buf[:, :at] == 7).all()) and bool((buf[:, at + N:] == 7).all())


# x and out in one buffer: a row copy (the workspace) only where they share memory. [x | out] and [out | x] side by side
# don't, also with other rows between (x from row 2 on); one shared column, or out running into x's next row, does.
@pytest.mark.parametrize("M", [3, 100])
@pytest.mark.parametrize("xat,oat,row,shift,copied", [(0, 96, 352, 0, False), (256, 0, 352, 0, False), (0, 96, 352, 2, False),
                                                      (256, 0, 352, 2, False), (0, 88, 352, 0, True), (256, 8, 352, 0, True),
                                                      (0, 96, 344, 2, True), (0, 0, 352, 0, True)])
def test_linear_column_slices_of_one_buffer(device, monkeypatch, M, xat, oat, row, shift, copied):
    from nanovllm_amd import _lib
    g = torch.Generator(device=device).manual_seed(M + xat)
    lin = RowInvariantLinear((torch.randn(256, 96, device=device, generator=g) / 10).to(torch.bfloat16))
    flat = torch.zeros((M + shift + 1) * row + 512, dtype=torch.bfloat16, device=device)
    x = flat.as_strided((M, 96), (row, 1), shift * row + xat)
    out = flat.as_strided((M, 256), (row, 1), oat)
    x.copy_(torch.randn(M, 96, device=device, generator=g).to(torch.bfloat16))
    want = lin(x)
    ws = torch.full((1 << 16,), 0x5a, dtype=torch.uint8, device=device)
    monkeypatch.setattr(_lib, "workspace", lambda n, dev, tag="": ws)
    assert torch.equal(lin(x, out=out), want)
    assert bool((ws != 0x5a).any()) == copied


def _ranges(N, K):
    """The layer's rule: packed tiles of 256 rows from `full` on are summed in n ranges of k (sd_linear's contract)."""
    tiles = -(-N // 256)
    tail = tiles - (tiles - 1) // 256 * 256
    n = 1 if 2 * tail > 256 else min(8, 256 // tail, K // 64)
    return (tiles, 1) if n < 2 else (tiles - tail, n)


# How an output is summed, made visible: a weight row holds 2^28 in the first column, -2^28 in the last and quarters
# between, in each range but the first for 4 m of its steps of 32 columns before the last. A range of its own keeps its
# 32 m, and every sum on the way is exact (a multiple of 32 below 2^28 + 2^24); added to 2^28 step by step, the 8 of a
# step are less than half a unit of 32 and all are lost. So outputs are 32 times the sum of m with the ranges and 0 in
# a tile of one. Every kernel and workgroup shape, ranges that end anywhere in the steps ahead, rows of unlike signs.
@pytest.mark.parametrize("N,K", [(1000, 1056), (4096, 4096), (4096, 12288), (6144, 1184), (24576, 4096), (76800, 1568),
                                 (151936, 1024), (33000, 512)])
def test_linear_sums_ranges_of_k(device, N, K):
    full, n = _ranges(N, K)
    S = K // 32
    w = torch.zeros(K, dtype=torch.float64)
    total = 0
    for r in range(1, n):
        begin, end = r * S // n, (r + 1) * S // n
        m = (end - begin - 1) // 4
        w[32 * begin:32 * (begin + 4 * m)] = 0.25
        total += 32 * m
    assert n == 1 or total > 0
    w[0], w[K - 1] = 2.0 ** 28, -2.0 ** 28
    single = torch.zeros(K, dtype=torch.float64)             # a tile of one range: quarters everywhere, all lost
    single[0], single[32:K - 32], single[K - 1] = 2.0 ** 28, 0.25, -2.0 ** 28
    scale = torch.tensor([1.0, -2.0, 4.0], dtype=torch.float64)[torch.arange(N) % 3]
    cut = min(N, 256 * full)
    weight = torch.empty(N, K, dtype=torch.bfloat16, device=device)
    weight[:cut] = (scale[:cut, None].to(device) * single.to(device)).to(torch.bfloat16)
    weight[cut:] = (scale[cut:, None].to(device) * w.to(device)).to(torch.bfloat16)
    want = (scale * total * (torch.arange(N) >= cut)).to(torch.bfloat16).to(device)
    lin = RowInvariantLinear(weight)
    sign = (1.0 - 2.0 * (torch.arange(1168) % 2)).to(torch.bfloat16).to(device)
    x = sign[:, None].expand(1168, K).contiguous()
    for M in (1, 16, 17, 64, 80, 160, 320, 600, 1168) if N < 100000 else (5, 20, 64, 320):
        print(f"M={M} N={N} K={K} ranges={n} from tile {full}", flush=True)
        y = lin(x[:M])
        assert torch.equal(y.float(), (sign[:M, None] * want).float()), f"M={M}"


def test_linear_output_over_its_input(device):
    g = torch.Generator(device=device).manual_seed(5)
    lin = RowInvariantLinear((torch.randn(512, 512, device=device, generator=g) / 23).to(torch.bfloat16))
    for M in (3, 100, 700):
        x = torch.randn(M, 512, device=device, generator=g).to(torch.bfloat16)
        want = lin(x)
        assert torch.equal(lin(x, out=x), want)


# SiLU-and-multiply against the eager operations in float64 with their two roundings: the fp32 silu is within a few
# units of 2^-24, so its bf16 rounding moves by at most one unit and only where it lies that close to a midpoint.
@pytest.mark.parametrize("M,half", [(1, 8), (5, 2056), (80, 12288), (3, 2048)])
def test_silu_and_mul(device, M, half):
    g = torch.Generator(device=device).manual_seed(half)
    wide = (4 * torch.randn(M, 2 * half + 8, device=device, generator=g)).to(torch.bfloat16)
    x = wide[:, :2 * half]                                    # a row stride past the row
    x[0, :6] = torch.tensor([0.0, -0.0, 200.0, -200.0, float("inf"), float("nan")])
    gate, up = x.double().chunk(2, -1)
    want = ((gate / (1 + torch.exp(-gate))).to(torch.bfloat16).double() * up).to(torch.bfloat16)
    got = silu_and_mul(x)
    ok = (got.view(torch.int16) == want.view(torch.int16)) | (got.isnan() & want.isnan()) | (got == want)
    assert ok.float().mean().item() >= 0.999
    finite = want.isfinite()
    assert bool(((got.float() - want.float()).abs()[finite] <= 2 * _ulp_bf16(want.float())[finite]).all())
    assert torch.equal(silu_and_mul(x[:1])[0].view(torch.int16), got[0].view(torch.int16))
