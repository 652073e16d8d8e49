"""GPU parity of the int4 kernels (quantise, dequantise, M=1 GEMV) against the CPU oracle.

Bar: quantised values / scales / zeros and dequantised weights bit-exact; GEMV within the
fp32-accumulation bound of an fp64 brute force, rounded to bf16.
"""
import pytest
import torch

from tests.helpers import gemm_bound, log

pytestmark = pytest.mark.gpu

SHAPES = [(3584, 2560), (2560, 2560), (16384, 2560), (2560, 8192), (8, 128), (24, 384)]


def _weights(n, k, seed, kind="normal"):
    g = torch.Generator().manual_seed(seed)
    w = (torch.randn(n, k, generator=g) * 0.02)
    if kind == "edge":
        w = w.view(n, k // 128, 128)
        w[0, :] = 0.25                       # constant group -> scale clamp 1e-6
        w[1 % n, 0] = -1.0                   # outlier
        w[-1, -1, :64] = 3.0                 # two-valued group
        w = w.view(n, k)
    return w.to(torch.bfloat16)


@pytest.mark.parametrize("n,k", SHAPES)
def test_quantize_bit_exact(dev, n, k):
    from flint_amd.quantize import quantize_int4, unpack_q, unpack_sz
    from oracle import quant
    for kind in ("normal", "edge"):
        log(f"quantize n={n} k={k} kind={kind}")
        w = _weights(n, k, 1, kind)
        q, sz = quantize_int4(w.to(dev))
        torch.cuda.synchronize()
        qo, so, zo = quant.group_quantize(w)
        assert torch.equal(unpack_q(q).cpu(), qo)
        s, z = unpack_sz(sz)
        assert torch.equal(s.cpu().view(torch.int16), so.view(torch.int16))
        assert torch.equal(z.cpu().view(torch.int16), zo.view(torch.int16))


@pytest.mark.parametrize("matrix_cores", [False, True])
@pytest.mark.parametrize("n,k", SHAPES)
def test_dequant_bit_exact(dev, n, k, matrix_cores):
    """Both device forms of the dequantisation (vector ALUs; 4x4x4 MFMAs lane by lane, the decode
    GEMVs') give the oracle's bits, edge groups (scale clamp, outlier, two values) included."""
    from flint_amd.quantize import quantize_int4, dequantize_int4
    from oracle import quant
    w = _weights(n, k, 2, "edge")
    log(f"dequant n={n} k={k} matrix_cores={matrix_cores}")
    q, sz = quantize_int4(w.to(dev))
    dq = dequantize_int4(q, sz, matrix_cores).cpu()
    ref = quant.dq_linear_weight(w)
    assert torch.equal(dq.view(torch.int16), ref.view(torch.int16))


def test_dequant_mx_extreme_scales(dev):
    """The matrix-core form on hand-set (scale, zero) words across the bf16 range -- tiny and huge
    scales, zeros of both signs and magnitudes that make the fp32 add round -- against the vector
    form, every nibble value in every position."""
    from flint_amd.quantize import dequantize_int4
    g = torch.Generator().manual_seed(11)
    n, k = 64, 512
    q = torch.randint(-2**31, 2**31 - 1, (n, k // 8), generator=g, dtype=torch.int64).to(torch.int32)
    q[0] = 0x76543210
    q[1] = -0x789abcdf   # 0x87654321 as int32
    s = torch.tensor([1e-30, 3e-8, 1e-6, 2.5e-3, 0.02, 1.0, 7.5, 3e4, 1e30], dtype=torch.float32)
    z = torch.tensor([0.0, -0.0, 1e-30, -2.5e-3, 0.6, -1.0, 200.0, -3e4, 1e30], dtype=torch.float32)
    si = torch.randint(0, len(s), (n, k // 128), generator=g)
    zi = torch.randint(0, len(z), (n, k // 128), generator=g)
    sb = s[si].to(torch.bfloat16).view(torch.int16).to(torch.int32) & 0xFFFF
    zb = z[zi].to(torch.bfloat16).view(torch.int16).to(torch.int32) & 0xFFFF
    sz = (sb | (zb << 16)).to(torch.int32)
    a = dequantize_int4(q.to(dev), sz.to(dev), False).cpu()
    b = dequantize_int4(q.to(dev), sz.to(dev), True).cpu()
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("n,k", SHAPES)
def test_gemv_vs_fp64(dev, n, k):
    from flint_amd.quantize import quantize_int4, gemv_int4
    from oracle import quant
    w = _weights(n, k, 3)
    g = torch.Generator().manual_seed(4)
    x = torch.randn(k, generator=g).to(torch.bfloat16)
    log(f"gemv n={n} k={k}")
    q, sz = quantize_int4(w.to(dev))
    y = gemv_int4(q, sz, x.to(dev)).cpu()
    dq = quant.dq_linear_weight(w).double()
    ref = dq @ x.double()
    # fp32 accumulation of k products: |err| <= k * 2^-24 * sum|x*w|, plus bf16 output rounding
    bound = k * 2.0 ** -24 * (dq.abs() @ x.double().abs()) + ref.abs() * 2.0 ** -8 + 1e-30
    err = (y.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
    # rounded results agree with the fp64 reference rounded once except at rare rounding ties
    mism = (y != ref.float().to(torch.bfloat16)).float().mean().item()
    log(f"  bf16 mismatch rate vs fp64-rounded: {mism:.2e}")
    assert mism < 2e-3


def test_gemv_matches_oracle_linear(dev):
    """Same contract as the oracle's F.linear on dequantised weights (the reference linear)."""
    from flint_amd.quantize import quantize_int4, gemv_int4
    from oracle import quant
    n, k = 16384, 2560
    w = _weights(n, k, 5)
    x = torch.randn(k, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16)
    q, sz = quantize_int4(w.to(dev))
    y = gemv_int4(q, sz, x.to(dev)).cpu()
    ref = torch.nn.functional.linear(x.view(1, -1), quant.dq_linear_weight(w)).view(-1)
    diff = (y.float() - ref.float()).abs().max().item()
    mism = (y != ref).float().mean().item()
    log(f"gemv vs oracle linear: max|diff|={diff:.3e} mismatch={mism:.2e}")
    assert mism < 2e-3 and diff < 2e-2


GEMM_CASES = [(3584, 2560, 5), (2560, 8192, 8), (16384, 2560, 16), (24, 384, 3), (8, 128, 1),
              (2560, 2560, 2),
              # the second 16-row activation block (tokens 16..31), with N not a multiple of 16
              (3584, 2560, 17), (2568, 8192, 24), (1000, 2560, 32), (24, 384, 32)]


@pytest.mark.parametrize("n,k,m", GEMM_CASES)
def test_gemm_vs_fp64(dev, n, k, m):
    """M-row int4 GEMM on the matrix cores (verify's weight-read-once product): every output within
    the fp32-accumulation bound of the exact product with the bit-exact dequantised weights."""
    from flint_amd.quantize import quantize_int4, gemm_int4
    from oracle import quant
    w = _weights(n, k, 7)
    g = torch.Generator().manual_seed(8)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    log(f"gemm n={n} k={k} m={m}")
    q, sz = quantize_int4(w.to(dev))
    y = gemm_int4(q, sz, x.to(dev)).cpu()
    assert y.shape == (m, n)
    dq = quant.dq_linear_weight(w).double()
    ref = x.double() @ dq.t()
    bound = k * 2.0 ** -24 * (x.double().abs() @ dq.abs().t()) + ref.abs() * 2.0 ** -8 + 1e-30
    err = (y.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
    mism = (y != ref.float().to(torch.bfloat16)).float().mean().item()
    log(f"  bf16 mismatch rate vs fp64-rounded: {mism:.2e}")
    assert mism < 2e-3


@pytest.mark.parametrize("m", [8, 32])
def test_gemm_rows_match_gemv(dev, m):
    """Row m of the M-row GEMM equals the M=1 GEMV of x[m] up to fp32 summation order."""
    from flint_amd.quantize import quantize_int4, gemm_int4, gemv_int4
    n, k = 3584, 2560
    w = _weights(n, k, 9)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(10)).to(torch.bfloat16)
    q, sz = quantize_int4(w.to(dev))
    y = gemm_int4(q, sz, x.to(dev)).cpu()
    for i in range(m):
        yv = gemv_int4(q, sz, x[i].contiguous().to(dev)).cpu()
        d = (y[i].float() - yv.float()).abs()
        assert float(d.max()) <= float(yv.float().abs().max()) * 2.0 ** -7
        assert float((d > 0).float().mean()) < 2e-3


@pytest.mark.parametrize("lead", [(1,), (8,), (2, 16), (32,), (3, 25)])
def test_weight_only_int4_linear(dev, lead):
    """WeightOnlyInt4Linear (the drop-in for reference engine/quantize.py:483-525) at M = 1
    (the GEMV), M up to 32 (one GEMM launch, leading dimensions flattened) and M = 75 (three
    launches of up to 32 rows, as gpt-fast's prefill passes a whole prompt) against the oracle's
    linear on the dequantised weights; its buffers hold the quantised values exactly."""
    from flint_amd.quantize import WeightOnlyInt4Linear, unpack_q, unpack_sz
    from oracle import quant
    n, k = 2560, 2560
    w = _weights(n, k, 12)
    mod = WeightOnlyInt4Linear.from_float(w.to(dev))
    qo, so, zo = quant.group_quantize(w)
    assert torch.equal(unpack_q(mod.weight).cpu(), qo)
    s, z = unpack_sz(mod.scales_and_zeros)
    assert torch.equal(s.cpu().view(torch.int16), so.view(torch.int16))
    assert torch.equal(z.cpu().view(torch.int16), zo.view(torch.int16))
    g = torch.Generator().manual_seed(13)
    x = torch.randn(*lead, k, generator=g).to(torch.bfloat16)
    y = mod(x.to(dev)).cpu()
    assert y.shape == (*lead, n) and y.dtype == torch.bfloat16
    ref = torch.nn.functional.linear(x.reshape(-1, k), quant.dq_linear_weight(w)).view(*lead, n)
    diff = (y.float() - ref.float()).abs().max().item()
    mism = (y != ref).float().mean().item()
    log(f"WeightOnlyInt4Linear lead={lead}: max|diff|={diff:.3e} mismatch={mism:.2e}")
    assert mism < 2e-3 and diff <= 2.0 ** -7 * float(ref.float().abs().max())
    with pytest.raises(Exception):
        mod(torch.zeros(4, k + 128, dtype=torch.bfloat16, device=dev))  # wrong inner dimension


def _check_gemm(y, x, dq):
    ref, bound = gemm_bound(x, dq)
    d = (y.double() - ref).abs()
    log(f"gemm {tuple(x.shape)} -> {y.shape[1]}: max|d| {float(d.max()):.3e}, largest share of its bound {float((d / bound).max()):.3f}")
    assert bool((d <= bound).all())


@pytest.mark.parametrize("m,n,k", [(33, 64, 128), (64, 63, 384), (65, 2570, 2560), (127, 130, 8192), (129, 16385, 256),
                                   (300, 16384, 128), (2049, 2048, 384), (8193, 65, 128), (400, 16385, 128),
                                   (1100, 8200, 384), (2049, 4100, 256), (333, 2570, 1408), (130, 3400, 4352),
                                   (300, 3500, 2304), (2, 4097, 384), (16, 8193, 128), (9, 14350, 640), (17, 4097, 1152),
                                   (32, 8193, 640), (9, 12270, 2688), (16, 12300, 1536), (400, 14400, 384), (448, 14340, 256),
                                   (520, 13000, 1536), (520, 13000, 1664), (1100, 10900, 384)])
def test_gemm_rows(dev, m, n, k):
    """fl_gemm_rows_int4 at the edges of its tiles (64 and 128 rows of both operands, and 128 x 256 where
    at least 224 of those fill the chip, beyond 256 from 384 or 13 groups on: 400 x 14400, 520 x 13000 x 1664, 1100 x 10900), of its ways, its K parts
    and its launches of 8192 rows, and fl_gemm_int4 past 256, 512 and 768 tiles of 16 weight rows, N odd and not, into an output that is not 8-byte aligned
    too: fp32 sums of exact products, so a result may differ from the oracle's only where another
    order of the sum rounds to the neighbouring bf16 value."""
    from flint_amd.quantize import dequantize_int4, gemm_int4, quantize_int4
    w = _weights(n, k, 21, "edge").to(dev)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(22)).to(torch.bfloat16).to(dev)
    q, sz = quantize_int4(w)
    y = gemm_int4(q, sz, x)
    _check_gemm(y, x, dequantize_int4(q, sz))
    buf = torch.zeros(m * n + 3, dtype=torch.bfloat16, device=dev)
    gemm_int4(q, sz, x, buf[1:1 + m * n].view(m, n))
    assert torch.equal(buf[1:1 + m * n].view(m, n), y) and not buf[:1].any() and not buf[1 + m * n:].any()


@pytest.mark.parametrize("m,n,k", [(2, 5, 128), (16, 131073, 128), (9, 2561, 1280), (9, 2561, 1408), (3, 12305, 2560),
                                   (3, 12305, 2688), (16, 13000, 1280), (16, 13109, 1280), (17, 2561, 768), (17, 2561, 896),
                                   (32, 5440, 768), (32, 5500, 768), (25, 20003, 256), (17, 16384, 384)])
def test_gemm_few_groups(dev, m, n, k):
    """fl_gemm_int4 on both sides of each line between its two kernels (few K groups: k_gemm): 10 and 20
    groups, 131072 products (by 16 rows and 128 columns) up to 16 rows; 2 and 6 groups, 65536 beyond."""
    from flint_amd.quantize import dequantize_int4, gemm_int4, quantize_int4
    w = _weights(n, k, 23, "edge").to(dev)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(24)).to(torch.bfloat16).to(dev)
    q, sz = quantize_int4(w)
    _check_gemm(gemm_int4(q, sz, x), x, dequantize_int4(q, sz))


def test_scales_and_zeros_gptfast_layout(dev):
    """scales_and_zeros_gptfast gives gpt-fast's [K/128, N, 2] bf16 tensor
    (reference engine/quantize.py:79-93 pack_scales_and_zeros) of the same values the oracle
    packs."""
    from flint_amd.quantize import quantize_int4, scales_and_zeros_gptfast
    from oracle import quant
    n, k = 384, 1024
    w = _weights(n, k, 14, "edge")
    q, sz = quantize_int4(w.to(dev))
    got = scales_and_zeros_gptfast(sz).cpu()
    _, so, zo = quant.group_quantize(w)
    ref = quant.pack_scales_and_zeros(so, zo)
    assert got.shape == (k // 128, n, 2) and got.dtype == torch.bfloat16
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
    # the reference's definition: entry [g, n] = (scale, zero) of row n, group g
    for g, r in ((0, 0), (3, 17), (7, n - 1)):
        assert got[g, r, 0].view(torch.int16) == so[r, g].view(torch.int16)
        assert got[g, r, 1].view(torch.int16) == zo[r, g].view(torch.int16)


TILED_SHAPES = [(3584, 2560), (16384, 2560), (2560, 8192), (16, 128), (48, 384), (32, 16384)]


def _tiled(q, n, k):
    from flint_amd import _lib
    qt = torch.empty(n // 16, k // 128, 64, 4, dtype=torch.int32, device=q.device)
    _lib.call("fl_tile_int4", _lib.ptr(q), _lib.ptr(qt), n, k, _lib.stream_ptr())
    return qt


@pytest.mark.parametrize("n,k", TILED_SHAPES)
def test_tiled_dequant_bit_exact(dev, n, k):
    """The matrix-core dequantisation (fl_tile_int4 + fl_dequant_int4_tiled: D1 = (128+q) diag(s)
    - 136 s, round, D2 = I a + z, round) gives gpt-fast's bf16(bf16((q-8) s) + z) bit for bit,
    edge groups included (constant group, outlier, two-valued group)."""
    from flint_amd import _lib
    from flint_amd.quantize import quantize_int4
    from oracle import quant
    w = _weights(n, k, 21, "edge")
    log(f"tiled dequant n={n} k={k}")
    q, sz = quantize_int4(w.to(dev))
    qt = _tiled(q, n, k)
    out = torch.empty(n, k, dtype=torch.bfloat16, device=dev)
    _lib.call("fl_dequant_int4_tiled", _lib.ptr(qt), _lib.ptr(sz), _lib.ptr(out), n, k, _lib.stream_ptr())
    ref = quant.dq_linear_weight(w)
    got = out.cpu()
    bad = (got.view(torch.int16) != ref.view(torch.int16))
    if bool(bad.any()):
        idx = bad.nonzero()[:12].tolist()
        rows = bad.nonzero()[:, 0] % 16
        cols = bad.nonzero()[:, 1] % 128
        log(f"  {int(bad.sum())} of {bad.numel()} differ; rows mod 16 {torch.bincount(rows, minlength=16).tolist()}; "
            f"cols mod 16 {torch.bincount(cols % 16, minlength=16).tolist()}; cols // 16 {torch.bincount(cols // 16, minlength=8).tolist()}")
        for r, c in idx:
            log(f"  [{r},{c}] got {float(got[r, c])} want {float(ref[r, c])}")
    assert not bool(bad.any())


@pytest.mark.parametrize("n,k", TILED_SHAPES)
def test_tiled_gemv_vs_fp64(dev, n, k):
    """The matrix-core GEMV within the fp32-accumulation bound of the exact product, and equal to
    the row-layout GEMV up to fp32 summation order."""
    from flint_amd import _lib
    from flint_amd.quantize import quantize_int4, gemv_int4
    from oracle import quant
    w = _weights(n, k, 22)
    x = torch.randn(k, generator=torch.Generator().manual_seed(23)).to(torch.bfloat16)
    log(f"tiled gemv n={n} k={k}")
    q, sz = quantize_int4(w.to(dev))
    qt = _tiled(q, n, k)
    y = torch.empty(n, dtype=torch.bfloat16, device=dev)
    _lib.call("fl_gemv_int4_tiled", _lib.ptr(qt), _lib.ptr(sz), _lib.ptr(x.to(dev)), _lib.ptr(y), n, k,
              _lib.stream_ptr())
    y = y.cpu()
    dq = quant.dq_linear_weight(w).double()
    ref = dq @ x.double()
    bound = k * 2.0 ** -24 * (dq.abs() @ x.double().abs()) + ref.abs() * 2.0 ** -8 + 1e-30
    err = (y.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
    mism = (y != ref.float().to(torch.bfloat16)).float().mean().item()
    yr = gemv_int4(q, sz, x.to(dev)).cpu()
    log(f"  bf16 mismatch vs fp64-rounded {mism:.2e}, vs row-layout GEMV {(y != yr).float().mean().item():.2e}")
    assert mism < 2e-3


@pytest.mark.parametrize("kind", ["scales", "offset", "constant", "tiny", "inf"])
def test_quantize_wide_range(dev, kind):
    """k_quantize divides by a reciprocal and a correction where nothing can overflow and by a true
    division elsewhere: groups across the bf16 range (both paths within one wave's rows), large offsets,
    constant and subnormal groups, and groups holding an infinity, against the same steps in
    torch (each a bf16 operation). Rows that do not fill a workgroup."""
    from flint_amd.quantize import quantize_int4, unpack_q, unpack_sz
    g = torch.Generator(device=dev).manual_seed(31)
    n, k = 173, 640
    w = torch.randn(n, k, generator=g, device=dev)
    if kind == "scales":
        w *= torch.exp2(torch.randint(-100, 120, (n, 1), generator=g, device=dev).float())
    elif kind == "offset":
        w = w * 1e-3 + 1000.0 * torch.randn(n, k // 128, generator=g, device=dev).repeat_interleave(128, 1)
    elif kind == "constant":
        w = torch.randn(n, k // 128, generator=g, device=dev).repeat_interleave(128, 1)
    elif kind == "tiny":
        w *= 2.0 ** -130
    elif kind == "inf":
        w[::3, 77] = float("inf")
    w = w.to(torch.bfloat16).contiguous()
    x = w.view(-1, 128)
    mx, mn = x.amax(1, keepdim=True), x.amin(1, keepdim=True)
    s = (mx - mn).clamp(min=1e-6) / 15
    z = mn + s * 8
    t = ((x - (z - s * 8)) / s).round().clamp(0, 15)
    fine = torch.isfinite(t).all(1).view(n, -1)  # torch's int32 of a NaN is undefined
    q, sz = quantize_int4(w)
    got = unpack_q(q).view(n, -1, 128)
    assert torch.equal(got[fine], t.nan_to_num(0).to(torch.int32).view(n, -1, 128)[fine])
    gs, gz = unpack_sz(sz)
    assert torch.equal(gs[fine].view(torch.int16), s.view(n, -1)[fine].view(torch.int16))
    assert torch.equal(gz[fine].view(torch.int16), z.view(n, -1)[fine].view(torch.int16))
    assert bool(fine.all()) == (kind != "inf")


def test_quantize_nan(dev):
    """A group of only NaN has a NaN zero point (torch's min of it) and the scale of an empty range; in a
    group with other values NaN takes no part in the range and becomes 0. The other groups of the wave
    are what they are without it."""
    from flint_amd.quantize import quantize_int4, unpack_q, unpack_sz
    n, k = 37, 384
    w = _weights(n, k, 32).to(dev)
    base_q, base_sz = quantize_int4(w)
    bad = w.clone()
    bad[3, :128] = float("nan")
    bad[::5, 256:384] = float("nan")
    some = torch.zeros(n, k, dtype=torch.bool, device=dev)
    some[7, 0], some[8, 131], some[9, 128:255] = True, True, True
    bad[some] = float("nan")
    q, sz = quantize_int4(bad)
    gone = torch.isnan(bad.view(n, -1, 128)).all(2)
    s, z = unpack_sz(sz)
    v = unpack_q(q).view(n, -1, 128)
    assert bool(torch.isnan(z[gone]).all()) and not bool(v[gone].any())
    tiny = torch.tensor(1e-6, dtype=torch.bfloat16, device=dev) / 15
    assert bool((s[gone] == tiny).all())
    part = some.view(n, -1, 128).any(2)
    clean = ~gone & ~part
    assert torch.equal(v[clean], unpack_q(base_q).view(n, -1, 128)[clean])
    assert torch.equal(sz[clean], base_sz[clean])
    fill = torch.where(some, bad.view(n, -1, 128).nan_to_num(-1e9).amax(2).repeat_interleave(128, 1), w)
    fq, fsz = quantize_int4(fill.to(torch.bfloat16))
    assert torch.equal(sz[part], fsz[part]) and not bool(unpack_q(q)[some].any())
    keep = part.repeat_interleave(128, 1) & ~some
    assert torch.equal(unpack_q(q)[keep], unpack_q(fq)[keep])


@pytest.mark.parametrize("n,k", [(16, 128), (32, 256), (48, 640), (16, 16384), (160, 1152)])
def test_tile_layout(dev, n, k):
    """fl_tile_int4 at group counts that do and do not fill its workgroups of four, against the layout
    as the header states it."""
    from flint_amd.quantize import tile_int4, unpack_q
    q = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 8), generator=torch.Generator().manual_seed(n + k), dtype=torch.int64)
    q = q.to(torch.int32)
    v = unpack_q(q).view(n // 16, 16, k // 128, 128).to(torch.int64)
    want = torch.zeros(n // 16, k // 128, 64, 4, dtype=torch.int64)
    for l in range(64):
        p, c = (l // 4) % 4, 4 * (l // 16) + l % 4
        for half in range(2):
            for t in range(8):
                pair = v[:, 4 * p + 2 * half, :, c + 16 * t] | v[:, 4 * p + 2 * half + 1, :, c + 16 * t] << 16
                want[:, :, l, 2 * half + t // 4] |= pair << (4 * (t % 4))
    got = tile_int4(q.to(dev)).cpu().view(n // 16, k // 128, 64, 4).to(torch.int64) & 0xFFFFFFFF
    assert torch.equal(got, want)


@pytest.mark.parametrize("shape", [(1,), (1, 1), (5,), (2, 16), (33,), (4, 100)])
def test_linear_module_call(dev, shape):
    """WeightOnlyInt4Linear's single-call forward gives the general path's bits, on another stream and
    under graph capture too; a strided input, fp32, a subclass and an empty batch take the general path."""
    from flint_amd import quantize as Q
    n, k = 2570, 640
    mod = Q.WeightOnlyInt4Linear.from_float(_weights(n, k, 41).to(dev))
    x = torch.randn(*shape, k, generator=torch.Generator().manual_seed(42)).to(torch.bfloat16).to(dev)
    assert Q._linear_fast is not None
    x2 = x.view(-1, k)
    want = (Q.gemv_int4(mod.weight, mod.scales_and_zeros, x2[0]).view(1, n) if x2.shape[0] == 1
            else Q.gemm_int4(mod.weight, mod.scales_and_zeros, x2)).view(*shape, n)
    assert torch.equal(mod(x), want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = mod(x)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(y, want)
    wide = torch.zeros(*shape, k + 8, dtype=torch.bfloat16, device=dev)
    wide[..., :k] = x
    assert torch.equal(mod(wide[..., :k]), want) and torch.equal(mod(x.float()), want)
    assert torch.equal(mod(torch.nn.Parameter(x, requires_grad=False)), want)
    assert mod(x[:0]).shape == (0, *shape[1:], n)
    with pytest.raises(ValueError):
        mod(x.cpu())
    g = torch.cuda.CUDAGraph()
    xs = x.clone()
    with torch.cuda.graph(g):
        y = mod(xs)
    for i in range(3):
        xs.copy_(x * (i + 1))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, mod(x * (i + 1)))


def test_linear_without_workspace(dev):
    """Where memory has no room for the part sums of more than 32 rows, the call runs in launches of 32
    rows instead, through the module's single-call forward and through gemm_int4."""
    from flint_amd import _lib
    from flint_amd import quantize as Q
    m, n, k = 100, 2560, 8192  # 4 MB of part sums, a result of 512 KB
    need = _lib.ctypes.c_int64()
    _lib.call("fl_gemm_rows_workspace", m, n, k, _lib.ctypes.byref(need))
    assert need.value > 2 << 20
    mod = Q.WeightOnlyInt4Linear.from_float(_weights(n, k, 51).to(dev))
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(52)).to(torch.bfloat16).to(dev)
    want = torch.cat([Q.gemm_int4(mod.weight, mod.scales_and_zeros, x[r:r + 32].contiguous()) for r in range(0, m, 32)])
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    # room for the result in segments of the allocator that stay; no new segments, the larger ones filled up
    parts = [torch.empty(900 << 10, dtype=torch.uint8, device=dev) for _ in range(8)]
    del parts[::2]
    torch.cuda.set_per_process_memory_fraction(0.0)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            for _ in range(1000):
                parts.append(torch.empty(2 << 20, dtype=torch.uint8, device=dev))
        got, got2 = mod(x), Q.gemm_int4(mod.weight, mod.scales_and_zeros, x)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(got, want) and torch.equal(got2, want)
