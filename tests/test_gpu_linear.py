"""GPU parity of the decode projections: smla_linear, smla_rope and smla_o_proj.

* ``smla_rope`` equals the oracle's float32 rotation (golden-pinned) bit for bit, forward and
  inverse, bf16 and fp32.
* ``smla_linear`` equals the float64 product of the same bf16 operands within the float32
  accumulation error (1e-5 of sum |x||w|, far below what a dropped K slice or a wrong row would
  change), plus half a bf16 ulp when the output is bf16; with fp32 operands (the tiled GEMM only)
  within (K + 8) 2^-23 of sum |x||w|, twice the textbook bound of a K-term fp32 dot product.
  Up to 8 bf16 rows run the weight-streaming kernel, other shapes the tiled MFMA GEMM
  (ragged token and output tiles, K tails, groups, fp32 operands, split K ranges).
* ``smla_o_proj`` with the fused inverse RoPE equals, bit for bit, the standalone inverse rotation
  followed by the unrotated projection, and the oracle's o_project within bf16 tolerance.
"""
import numpy as np
import pytest
import torch

from conftest import announce
from oracle import mla as omla
from oracle import norm_rope as onr

pytestmark = pytest.mark.gpu


def _check_linear(got, x, w, G, out_dtype):
    x64, w64 = x.double().numpy(), w.double().numpy()
    T, GK = x64.shape
    K = GK // G
    N = w64.shape[0] // G
    ref = np.concatenate([x64[:, g * K:(g + 1) * K] @ w64[g * N:(g + 1) * N].T for g in range(G)], axis=1)
    mag = np.concatenate([np.abs(x64[:, g * K:(g + 1) * K]) @ np.abs(w64[g * N:(g + 1) * N]).T for g in range(G)],
                         axis=1)
    acc_tol = (K + 8) * 2.0 ** -23 if x.dtype == torch.float32 else 1e-5
    tol = acc_tol * mag + (np.abs(ref) * 2.0 ** -8 if out_dtype == torch.bfloat16 else 0.0)
    err = np.abs(got.double().cpu().numpy() - ref)
    assert np.all(err <= tol), f"max err {err.max():.3e}, worst ratio {(err / np.maximum(tol, 1e-30)).max():.3f}"


@pytest.mark.parametrize("T,G,N,K,out_dtype", [
    (8, 8, 1024, 4096, torch.bfloat16),      # o_grouped's grouped product at decode (LDS form)
    (12, 8, 1024, 4096, torch.bfloat16),     # the same width in the register form (T > 8)
    (8, 1, 4096, 8192, torch.float32),       # its second product (8 waves x 16 steps)
    (9, 1, 4096, 8192, torch.float32),       # register form
    (1, 1, 256, 4096, torch.float32),
    (3, 2, 48, 512, torch.float32),          # one wave per workgroup
    (16, 2, 64, 1024, torch.bfloat16),       # short K slices: the guarded last batch
    (17, 1, 128, 512, torch.float32),        # two token tiles, one ragged
    (32, 4, 32, 2048, torch.bfloat16),
    # the LDS form over 8192 rows: 2 and 4 waves, one wave with K = 512
    (5, 1, 8192, 1024, torch.float32),
    (8, 4, 2048, 2048, torch.bfloat16),
    (2, 1, 8192, 512, torch.float32),
    # the tiled MFMA GEMM
    (768, 1, 21760, 512, torch.float32),       # 256 x 256 DMA tiles: 3 x 85 of them
    (520, 2, 11000, 576, torch.bfloat16),      # the same, ragged tokens and outputs, two groups
    (64, 1, 1024, 4096, torch.float32),
    (4096, 1, 1024, 4096, torch.bfloat16),     # prefill's q_down
    (300, 1, 200, 520, torch.float32),         # ragged token and output tiles, a K tail
    (100, 8, 1024, 4096, torch.bfloat16),      # o_grouped's grouped product at prefill
    (33, 2, 48, 24, torch.float32),            # K shorter than one step
])
@pytest.mark.parametrize("operands", [torch.bfloat16, torch.float32])
def test_linear_vs_fp64(dev, T, G, N, K, out_dtype, operands):
    from smla import ops
    announce(f"linear T={T} G={G} N={N} K={K} out={out_dtype} operands={operands}")
    g = torch.Generator().manual_seed(T * 7 + G + N + K)
    x = torch.randn(T, G * K, generator=g).to(operands)
    w = (torch.randn(G * N, K, generator=g) * 0.05).to(operands)
    y = ops.linear_op(x.to(dev), w.to(dev), G, out_dtype)
    torch.cuda.synchronize()
    assert y.dtype == out_dtype and y.shape == (T, G * N)
    _check_linear(y.float(), x, w, G, out_dtype)


@pytest.mark.parametrize("T,G,N,K", [
    # one case or more per tile form of the bf16 GEMM, with ragged tokens and outputs; N not a multiple
    # of 8 (4) takes the element-wise stores of bf16 (fp32) outputs
    (9, 1, 48, 128),         # two K steps, one 256 x 256 tile mostly past the edges
    (40, 1, 72, 192),        # three steps, 128 x 256
    (70, 1, 333, 512),       # 64 x 64, odd N
    (65, 3, 90, 1152),       # 64 x 64, four splits of 4 or 5 steps, three groups
    (33, 1, 1000, 2048),     # 64 x 64, eight splits
    (150, 1, 520, 4160),     # eight splits of a range they do not divide
    (130, 2, 4100, 320),     # 64 x 64 over many tiles, five steps
    (300, 1, 4104, 4096),    # 128 x 128, two splits
    (420, 1, 4090, 8192),    # the same, N not a multiple of 4
    (1300, 1, 2050, 2048),   # 128 x 128
    (700, 8, 1000, 1024),    # 128 x 256, eight groups
    (257, 1, 32776, 256),    # 128 x 256, one token past two tiles
    (513, 1, 33000, 128),    # 256 x 256, two steps
])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_linear_tile_forms(dev, T, G, N, K, out_dtype):
    from smla import ops
    announce(f"linear tile forms T={T} G={G} N={N} K={K} out={out_dtype}")
    g = torch.Generator(device=dev).manual_seed(T + N + K)
    x = torch.randn(T, G * K, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(G * N, K, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    y = ops.linear_op(x, w, G, out_dtype)
    x64, w64 = x.double().view(T, G, K), w.double().view(G, N, K)
    for i in range(G):       # the bounds of _check_linear, evaluated on the GPU
        ref, mag = x64[:, i] @ w64[i].t(), x64[:, i].abs() @ w64[i].abs().t()
        tol = 1e-5 * mag + (ref.abs() * 2.0 ** -8 if out_dtype == torch.bfloat16 else 0.0)
        assert bool(((y[:, i * N:(i + 1) * N].double() - ref).abs() <= tol).all())


@pytest.mark.parametrize("T,G,N,K", [
    (1300, 8, 1024, 4096),   # 6 token tiles of 256: groups of 4 and 2, the last tile ragged
    (2305, 2, 1500, 16384),  # two groups, ragged outputs
    (1100, 16, 700, 2048),
    (4000, 1, 1024, 32768),  # one group: no pairs
])
def test_linear_rows_64k_apart(dev, T, G, N, K):
    """Rows of x 64 KB apart take the tiles of two groups side by side: every tile of every group is there."""
    test_linear_tile_forms(dev, T, G, N, K, torch.bfloat16)


@pytest.mark.parametrize("T,G,N,K", [
    # both sides of the lines between the weight-streaming kernels and the tiled GEMM
    (16, 1, 8192, 512), (9, 1, 8208, 512),            # 512 and 513 workgroups of 16 outputs
    (9, 2, 4096, 4096), (16, 1, 8192, 4608),          # 512 x 4096 and beyond
    (12, 1, 1536, 4096), (12, 1, 1552, 4096),         # few outputs of a long K
    (17, 1, 4096, 2048), (17, 1, 4112, 2048), (32, 1, 4096, 2560),
    (32, 1, 1024, 2048), (32, 1, 1040, 2048),
])
def test_linear_few_rows(dev, T, G, N, K):
    test_linear_tile_forms(dev, T, G, N, K, torch.float32)


@pytest.mark.parametrize("T,G,N,K", [
    (1, 1, 1024, 4096),      # 64 x 64 tiles, eight splits
    (70, 1, 333, 512),       # odd N: element-wise stores
    (129, 2, 136, 64),       # two steps of 32 k: 128 x 128 tiles, one token past the first
    (65, 3, 90, 160),        # five steps, three groups
    (700, 1, 2050, 1056),    # 128 x 128 tiles, ragged
])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_linear_fp32_tiles(dev, T, G, N, K, out_dtype):
    """fp32 operands on the bf16 matrix cores (three bf16 parts per value), by the bound of an fp32
    dot product."""
    from smla import ops
    announce(f"linear fp32 T={T} G={G} N={N} K={K} out={out_dtype}")
    g = torch.Generator().manual_seed(T + N + K)
    x = torch.randn(T, G * K, generator=g) * torch.exp2(torch.randint(-20, 20, (T, 1), generator=g).float())
    w = torch.randn(G * N, K, generator=g) * 0.05
    y = ops.linear_op(x.to(dev), w.to(dev), G, out_dtype)
    _check_linear(y.float(), x, w, G, out_dtype)


@pytest.mark.parametrize("T,N,K", [(64, 1024, 64), (300, 1024, 1024), (2046, 2048, 4096), (1024, 4096, 8192)])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_linear_fp32_one_sign(dev, T, N, K, sign):
    """Sums of one sign, where a term that falls below the accumulator's last place is lost every time and
    not only now and then.  K / 16 roundings of partial sums that grow evenly, each off by at most
    2^-24 of its partial sum, are 2^-24 sqrt(K / 48) of the result together (2-norm); the last addition
    and the terms that three bf16 parts leave out are 2^-24 each.  All of it is noise: the mean is at most
    the last two."""
    from smla import ops
    announce(f"linear fp32 one sign T={T} N={N} K={K}")
    g = torch.Generator(device=dev).manual_seed(T + K)
    x, w = torch.rand(T, K, generator=g, device=dev), torch.rand(N, K, generator=g, device=dev) * sign
    ref = x.double() @ w.double().t()
    err = (ops.linear_op(x, w, 1, torch.float32).double() - ref) / ref
    assert err.square().mean().sqrt().item() <= 2.0 ** -24 * ((K / 48) ** 0.5 + 2)
    assert abs(err.mean().item()) <= 2.0 ** -23


@pytest.mark.parametrize("T,N,K", [(40, 130, 4096), (300, 600, 96)])    # with and without splits
def test_linear_fp32_special_values(dev, T, N, K):
    """Infinities, NaN, values whose bf16 rounding overflows and subnormals come out as fp32 arithmetic
    gives them: the same places infinite and NaN, the rest within the fp32 bound and the rounding of a
    subnormal result."""
    from smla import ops
    announce(f"linear fp32 special values T={T} N={N} K={K}")
    g = torch.Generator().manual_seed(T)
    x, w = torch.randn(T, K, generator=g), torch.randn(N, K, generator=g) * 0.05
    x[0, 3], x[1, 5], x[2, 7], x[3, 9] = float("inf"), float("nan"), 3.4028234e38, -3.4e38
    x[4] *= 1e-36
    x[5] *= 1e-40
    w[4, 3] = 0.0                                   # inf * 0
    w[6, 11], x[6, 11] = float("-inf"), 2.0
    y = ops.linear_op(x.to(dev), w.to(dev), 1, torch.float32).cpu()
    ref = x.double() @ w.double().t()
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(torch.isinf(y), inf) and torch.equal(y[inf].double(), ref[inf])
    ok = torch.isfinite(ref)
    xf, wf = torch.nan_to_num(x.double(), 0, 0, 0), torch.nan_to_num(w.double(), 0, 0, 0)
    tol = (K + 8) * 2.0 ** -23 * (xf.abs() @ wf.abs().t()) + K * 2.0 ** -149
    assert bool(((y.double() - ref).abs()[ok] <= tol[ok]).all())


@pytest.mark.parametrize("N,K", [(130, 4096), (1030, 96)])       # 64 x 64 tiles with splits, 128 x 128
def test_linear_fp32_every_magnitude(dev, N, K):
    """Rows of every binary magnitude an fp32 operand can have, the smallest subnormal to the largest that
    leaves the sums finite: the fp32 bound throughout, plus what a result below 2^-126 is rounded by."""
    from smla import ops
    announce(f"linear fp32 magnitudes N={N} K={K}")
    g = torch.Generator().manual_seed(K)
    e = torch.arange(-149, 119).double()
    x = (torch.randn(e.numel(), K, generator=g).double() * torch.exp2(e)[:, None]).float()
    w = torch.randn(N, K, generator=g) * 0.05
    for a, b in ((x, w), (w, x)):
        y = ops.linear_op(a.to(dev), b.to(dev), 1, torch.float32).cpu().double()
        ref, mag = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
        assert bool(((y - ref).abs() <= (K + 8) * 2.0 ** -23 * mag + 16 * 2.0 ** -150).all())


def test_linear_fp32_single_products(dev):
    """Sums of one term: the split leaves out at most 2^-24 of a product and one addition rounds."""
    from smla import ops
    announce("linear fp32 single products")
    g = torch.Generator(device=dev).manual_seed(8)
    K = 1024
    x = torch.diag(1.0 + torch.rand(K, generator=g, device=dev))
    w = 1.0 + torch.rand(2048, K, generator=g, device=dev)
    y = ops.linear_op(x, w, 1, torch.float32).double()
    ref = x.diagonal().double()[:, None] * w.double().t()
    assert ((y - ref).abs() / ref).max().item() <= 2.0 ** -23


@pytest.mark.parametrize("T,N,K", [(300, 600, 8192), (1024, 2048, 4096)])
def test_linear_fp32_infinity_costs_no_cliff(dev, T, N, K):
    """One infinite weight makes a column of the result non-finite, which the fp32 MFMAs compute again block
    by block: that work is at most the product's own at a third of its rate (8 times with its start and
    its loads' latency), not a serial chain per output (40 times and more)."""
    from smla import ops
    announce(f"linear fp32 with an infinity T={T} N={N} K={K}")
    g = torch.Generator(device=dev).manual_seed(T)
    x, w = torch.randn(T, K, generator=g, device=dev), torch.randn(N, K, generator=g, device=dev)
    bad = w.clone()
    bad[5, 0] = float("inf")

    def us(weight):
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(6)]
        ops.linear_op(x, weight, 1, torch.float32)
        for e in ev:
            e.record()
            ops.linear_op(x, weight, 1, torch.float32)
        torch.cuda.synchronize()
        return min(a.elapsed_time(b) for a, b in zip(ev, ev[1:]))

    y = ops.linear_op(x, bad, 1, torch.float32)
    assert bool(torch.isinf(y[:, 5]).all()) and bool(torch.isfinite(y[:, :5]).all())
    assert us(bad) <= 8 * us(w)


@pytest.mark.parametrize("T,G,N,K", [(9, 1, 64, 4096), (17, 2, 48, 4096), (32, 1, 512, 4096), (100, 1, 1024, 4096)])
def test_linear_without_workspace(dev, T, G, N, K):
    """smla_linear (no workspace): 9 to 32 rows whose GEMM would split K run the weight-streaming
    kernel, more rows the GEMM without the split; both as exact as with a workspace."""
    from smla import _lib
    announce(f"linear without workspace T={T} G={G} N={N} K={K}")
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, G * K, generator=g).to(torch.bfloat16)
    w = (torch.randn(G * N, K, generator=g) * 0.05).to(torch.bfloat16)
    xd, wd, y = x.to(dev), w.to(dev), torch.empty(T, G * N, device=dev)
    assert _lib.lib().smla_linear_workspace(T, G, N, K, _lib.BF16) > 0
    _lib.call("smla_linear", xd.data_ptr(), _lib.BF16, wd.data_ptr(), _lib.BF16, T, G, N, K, y.data_ptr(), _lib.F32,
              torch.cuda.current_stream().cuda_stream)
    _check_linear(y, x, w, G, torch.float32)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("inverse", [False, True])
def test_rope_bit_exact(dev, dt, inverse):
    from smla import norm_rope as snr
    from smla import ops
    announce(f"rope dtype={dt} inverse={inverse}")
    g = torch.Generator().manual_seed(2)
    T, H, D, rd = 9, 64, 512, 64
    x = torch.randn(T, H, D, generator=g).to(dt)
    pos = torch.randint(0, 65536, (T,), generator=g, dtype=torch.int32)
    pos[0] = 0
    cos_t, sin_t = snr.rope_tables(rd, 65536, device=dev)
    got = x.to(dev)
    ops.rope_op_(got, pos.to(dev), cos_t, sin_t, inverse)
    cis = torch.complex(cos_t.cpu()[pos.long()], sin_t.cpu()[pos.long()])
    ref = x.clone()
    ref[..., D - rd:] = onr.apply_rotary_emb(x[None, :, :, D - rd:], cis, inverse=inverse)[0]
    assert torch.equal(got.cpu(), ref)


@pytest.mark.parametrize("T", [1, 8, 20, 40, 300])
def test_o_proj_fused_rope(dev, T):
    from smla import norm_rope as snr
    from smla import ops
    announce(f"o_proj T={T}")
    g = torch.Generator().manual_seed(T)
    H, D, rd, G, R, dim = 64, 512, 64, 8, 1024, 4096
    o = torch.randn(T, H, D, generator=g).to(torch.bfloat16)
    wa = (torch.randn(G * R, H * D // G, generator=g) * 0.02).to(torch.bfloat16)
    wb = (torch.randn(dim, G * R, generator=g) * 0.02).to(torch.bfloat16)
    pos = torch.randint(0, 65536, (T,), generator=g, dtype=torch.int32)
    cos_t, sin_t = snr.rope_tables(rd, 65536, device=dev)
    od, wad, wbd, posd = o.to(dev), wa.to(dev), wb.to(dev), pos.to(dev)
    fused = ops.o_proj_op(od, posd, cos_t, sin_t, wad, wbd, G, torch.float32)
    # the same rotation done first by the standalone kernel: identical operands, identical result
    rot = od.clone()
    ops.rope_op_(rot, posd, cos_t, sin_t, True)
    two = ops.o_proj_op(rot, None, None, None, wad, wbd, G, torch.float32)
    assert torch.equal(fused, two)
    # against the oracle (float64 products, bf16 intermediate)
    ref = omla.o_project(o, pos, cos_t.cpu(), sin_t.cpu(), wa.float().numpy(), wb.float().numpy(), G)
    np.testing.assert_allclose(fused.cpu().double().numpy(), ref, rtol=1e-2, atol=2e-2 * np.abs(ref).max())


@pytest.mark.parametrize("T", [600, 2048])
def test_o_proj_fused_rope_wide(dev, T):
    """The grouped product on the DMA tiles (600 tokens: 128 x 128, 2048: 256 x 256) with the
    inverse RoPE applied in LDS: equal to the standalone rotation followed by the plain product bit
    for bit, and to the oracle on a sample of tokens (each token's output depends on that token
    alone)."""
    from smla import norm_rope as snr
    from smla import ops
    announce(f"o_proj T={T} (DMA tiles with RoPE)")
    g = torch.Generator().manual_seed(T)
    H, D, rd, G, R, dim = 64, 512, 64, 8, 1024, 4096
    o = torch.randn(T, H, D, generator=g).to(torch.bfloat16)
    wa = (torch.randn(G * R, H * D // G, generator=g) * 0.02).to(torch.bfloat16)
    wb = (torch.randn(dim, G * R, generator=g) * 0.02).to(torch.bfloat16)
    pos = torch.randint(0, 65536, (T,), generator=g, dtype=torch.int32)
    cos_t, sin_t = snr.rope_tables(rd, 65536, device=dev)
    od, wad, wbd, posd = o.to(dev), wa.to(dev), wb.to(dev), pos.to(dev)
    fused = ops.o_proj_op(od, posd, cos_t, sin_t, wad, wbd, G, torch.float32)
    rot = od.clone()
    ops.rope_op_(rot, posd, cos_t, sin_t, True)
    two = ops.o_proj_op(rot, None, None, None, wad, wbd, G, torch.float32)
    assert torch.equal(fused, two)
    idx = torch.tensor([0, 1, 127, 128, 255, 256, T // 2, T - 2, T - 1])
    ref = omla.o_project(o[idx], pos[idx], cos_t.cpu(), sin_t.cpu(), wa.float().numpy(), wb.float().numpy(), G)
    np.testing.assert_allclose(fused.cpu()[idx].double().numpy(), ref, rtol=1e-2, atol=2e-2 * np.abs(ref).max())


@pytest.mark.parametrize("T", [520, 2048])
def test_o_proj_token_anywhere(dev, T):
    """One token's output has the same bits wherever it stands in a prompt (rows of o 64 KB apart, tiles
    of 128 x 128 and 256 x 256): every output is one accumulation chain in k order."""
    from smla import norm_rope as snr
    from smla import ops
    announce(f"o_proj T={T}, one token repeated")
    g = torch.Generator(device=dev).manual_seed(T)
    o = torch.randn(1, 64, 512, generator=g, device=dev).to(torch.bfloat16).expand(T, -1, -1).contiguous()
    wa = (torch.randn(8192, 4096, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    wb = (torch.randn(4096, 8192, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    cos_t, sin_t = snr.rope_tables(64, 4096, device=dev)
    pos = torch.full((T,), 1234, dtype=torch.int32, device=dev)
    y = ops.o_proj_op(o, pos, cos_t, sin_t, wa, wb, 8, torch.float32)
    assert torch.equal(y, y[:1].expand(T, -1))


@pytest.mark.parametrize("T", [40, 300])
@pytest.mark.parametrize("H,D,G", [(8, 64, 1), (12, 192, 2), (4, 320, 2)])
def test_o_proj_fused_rope_head_dims(dev, T, H, D, G):
    """Heads of 1, 3 and 5 K steps of 64 (not only the layer's 8): the fused rotation finds each head's
    last 64 dims, with and without a split K range."""
    from smla import norm_rope as snr
    from smla import ops
    announce(f"o_proj T={T} heads={H} head_dim={D} groups={G}")
    g = torch.Generator(device=dev).manual_seed(T + D)
    o = torch.randn(T, H, D, generator=g, device=dev).to(torch.bfloat16)
    wa = (torch.randn(G * 128, H * D // G, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    wb = (torch.randn(256, G * 128, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    pos = torch.randint(0, 4096, (T,), generator=g, device=dev, dtype=torch.int32)
    cos_t, sin_t = snr.rope_tables(64, 4096, device=dev)
    rot = o.clone()
    ops.rope_op_(rot, pos, cos_t, sin_t, True)
    assert not torch.equal(rot, o)
    fused = ops.o_proj_op(o, pos, cos_t, sin_t, wa, wb, G, torch.float32)
    assert torch.equal(fused, ops.o_proj_op(rot, None, None, None, wa, wb, G, torch.float32))


def test_mla_mirror_routes(dev):
    """mla.linear / o_grouped / o_project run the weight-streaming kernels at decode shapes and the
    tiled GEMM beyond; both agree with the oracle."""
    from smla import mla
    from smla import norm_rope as snr
    announce("mla mirror")
    g = torch.Generator().manual_seed(5)
    H, D, G, R, dim = 64, 512, 8, 1024, 4096
    wa = (torch.randn(G * R, H * D // G, generator=g) * 0.02).to(torch.bfloat16)
    wb = (torch.randn(dim, G * R, generator=g) * 0.02).to(torch.bfloat16)
    cos_t, sin_t = snr.rope_tables(64, 65536, device=dev)
    for T in (4, 40):                  # decode kernel, then the GEMM path
        o = torch.randn(T, H, D, generator=g).to(torch.bfloat16)
        pos = torch.randint(0, 65536, (T,), generator=g, dtype=torch.int32)
        y = mla.o_project(o.to(dev), pos.to(dev), cos_t, sin_t, wa.to(dev), wb.to(dev))
        ref = omla.o_project(o, pos, cos_t.cpu(), sin_t.cpu(), wa.float().numpy(), wb.float().numpy(), G)
        np.testing.assert_allclose(y.cpu().double().numpy(), ref, rtol=2e-2, atol=2e-2 * np.abs(ref).max())
    x = torch.randn(3, 4096, generator=g).to(torch.bfloat16)
    W = (torch.randn(1024, 4096, generator=g) * 0.02).to(torch.bfloat16)
    y = mla.linear(x.to(dev), W.to(dev))
    np.testing.assert_allclose(y.cpu().double().numpy(), omla.linear(x.float().numpy(), W.float().numpy()),
                               rtol=2e-2, atol=2e-2)


def test_o_proj_graph_replays(dev):
    """The fused output path captured in a HIP graph: every replay, with eager work and
    synchronisations between replays, equals the eager result bit for bit."""
    from smla import norm_rope as snr
    from smla import ops
    announce("o_proj graph replay")
    g = torch.Generator().manual_seed(12)
    T, H, D, G, R, dim = 8, 64, 512, 8, 1024, 4096
    o = torch.randn(T, H, D, generator=g).to(torch.bfloat16).to(dev)
    wa = (torch.randn(G * R, H * D // G, generator=g) * 0.02).to(torch.bfloat16).to(dev)
    wb = (torch.randn(dim, G * R, generator=g) * 0.02).to(torch.bfloat16).to(dev)
    pos = torch.randint(0, 65536, (T,), generator=g, dtype=torch.int32).to(dev)
    cos_t, sin_t = snr.rope_tables(64, 65536, device=dev)
    eager = ops.o_proj_op(o, pos, cos_t, sin_t, wa, wb, G, torch.bfloat16)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.o_proj_op(o, pos, cos_t, sin_t, wa, wb, G, torch.bfloat16)
    for r in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {r}"
        ops.o_proj_op(o, pos, cos_t, sin_t, wa, wb, G, torch.bfloat16)     # eager work between replays
        torch.cuda.synchronize()


def _split_case(dev, dt):
    """A product whose plan splits K (checked), and the output path with a workspace."""
    from smla import _lib
    from smla import norm_rope as snr
    g = torch.Generator(device=dev).manual_seed(21)
    T, N, K = 64, 1024, 4096
    assert _lib.lib().smla_linear_workspace(T, 1, N, K, _lib.BF16 if dt == torch.bfloat16 else _lib.F32) > 0
    assert _lib.lib().smla_o_proj_workspace(T, 64, 512, 8, 1024, 4096) > 0
    x = torch.randn(T, K, generator=g, device=dev).to(dt)
    w = (torch.randn(N, K, generator=g, device=dev) * 0.05).to(dt)
    o = torch.randn(T, 64, 512, generator=g, device=dev).to(torch.bfloat16)
    wa = (torch.randn(8192, 4096, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    wb = (torch.randn(4096, 8192, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    pos = torch.randint(0, 4096, (T,), generator=g, device=dev, dtype=torch.int32)
    return x, w, (o, pos, *snr.rope_tables(64, 4096, device=dev), wa, wb, 8, torch.bfloat16)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_split_products_graph_replays(dev, dt):
    """Products with split K ranges captured in a HIP graph, their workspaces from the graph's pool: every
    replay, with eager work and synchronisations between replays, equals the eager result bit for bit."""
    from smla import ops
    announce(f"split products graph replay {dt}")
    x, w, op_args = _split_case(dev, dt)
    run = lambda: (ops.linear_op(x, w, 1, torch.float32), ops.o_proj_op(*op_args))  # noqa: E731
    eager = run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run()
    for r in range(3):
        for t in out:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, eager)), f"replay {r}"
        run()                                               # eager work between replays
        torch.cuda.synchronize()


def test_split_products_on_streams(dev):
    """The same products issued on two streams in turn, each call with a workspace of its own."""
    from smla import ops
    announce("split products on two streams")
    x, w, op_args = _split_case(dev, torch.bfloat16)
    eager = (ops.linear_op(x, w, 1, torch.float32), ops.o_proj_op(*op_args))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(dev) for _ in range(2)]
    got = []
    for _ in range(10):
        for st in streams:
            with torch.cuda.stream(st):
                got.append((ops.linear_op(x, w, 1, torch.float32), ops.o_proj_op(*op_args)))
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for pair in got for a, b in zip(pair, eager))


@pytest.mark.parametrize("shape,dt", [((2, 5, 64), torch.float32), ((2, 5, 8, 64), torch.bfloat16),
                                      ((1, 7, 64, 64), torch.float32)])
@pytest.mark.parametrize("inverse", [False, True])
def test_apply_rotary_emb_mirror(dev, shape, dt, inverse):
    """smla.norm_rope.apply_rotary_emb (ref_torch/norm_rope.py:53-62 signature, on smla_rope) equals
    the oracle's rotation bit for bit."""
    from smla import norm_rope as snr
    announce(f"apply_rotary_emb {shape} {dt} inverse={inverse}")
    g = torch.Generator().manual_seed(sum(shape))
    x = torch.randn(*shape, generator=g).to(dt)
    cis = onr.precompute_freqs_cis(shape[-1], shape[1], 65536, 160000.0, 16, 32, 1)
    got = snr.apply_rotary_emb(x.to(dev), cis.to(dev), inverse=inverse).cpu()
    ref = onr.apply_rotary_emb(x, cis, inverse=inverse)
    assert got.dtype == x.dtype and torch.equal(got, ref)


@pytest.mark.parametrize("T,K,dt", [(20, 4096, torch.bfloat16), (100, 4096, torch.bfloat16), (40, 4096, torch.float32)])
def test_linear_unaligned_workspace(dev, T, K, dt):
    """A workspace that 16-byte accesses cannot use is not used: the result of smla_linear, and the bytes of the
    workspace as they were."""
    from smla import _lib
    announce(f"linear, workspace at 4 bytes T={T} K={K} {dt}")
    g = torch.Generator(device=dev).manual_seed(T)
    N, code = 1000 if T > 32 else 1024, _lib.BF16 if dt == torch.bfloat16 else _lib.F32
    x = torch.randn(T, K, generator=g, device=dev).to(dt)
    w = (torch.randn(N, K, generator=g, device=dev) * 0.05).to(dt)
    y, ref = torch.empty(T, N, device=dev), torch.empty(T, N, device=dev)
    need = _lib.lib().smla_linear_workspace(T, 1, N, K, code)
    assert need > 0
    ws = torch.full((need + 16,), 9, dtype=torch.uint8, device=dev)
    st = torch.cuda.current_stream().cuda_stream
    args = (x.data_ptr(), code, w.data_ptr(), code, T, 1, N, K)
    _lib.call("smla_linear", *args, ref.data_ptr(), _lib.F32, st)
    _lib.call("smla_linear_ws", *args, y.data_ptr(), _lib.F32, ws.data_ptr() + 4, need, st)
    assert torch.equal(y, ref) and bool((ws == 9).all())
    _check_linear(y, x.cpu(), w.cpu(), 1, torch.float32)


def test_ops_eager_route(dev):
    """Plain CUDA tensors skip the registered op and give its result; whatever needs the op (a
    differentiated input, forward-mode level, functorch transform, fake tensors, a tracer, a CPU
    tensor) still reaches it."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    from smla import ops
    announce("ops eager route")
    x = torch.randn(4, 512, device=dev).to(torch.bfloat16)
    w = torch.randn(64, 512, device=dev).to(torch.bfloat16)
    args = (x, w, 1, torch.float32)
    seen = []

    def probe(a):
        seen.append(ops._eager((a, w, 1, torch.float32)))
        return a

    assert ops._eager(args)
    assert torch.equal(ops.linear_op(*args), ops.linear_op.op(*args))
    leaf = x.clone().requires_grad_()
    probe(leaf)
    assert ops.linear_op(leaf, w, 1, torch.float32).requires_grad
    torch.func.vmap(probe)(x[None])
    with torch.autograd.forward_ad.dual_level():
        probe(x)
    with FakeTensorMode() as mode:
        fake = mode.from_tensor(x)
        probe(fake)
        assert ops.linear_op(fake, mode.from_tensor(w), 1, torch.float32).shape == (4, 64)
    torch.jit.trace(probe, (x,), check_trace=False)
    probe(x.cpu())
    assert len(seen) >= 6 and not any(seen)
    with torch.no_grad():
        assert ops._eager((leaf, w, 1, torch.float32))


def test_ops_eager_route_negative_bit(dev):
    """A tensor with the negative bit set (its memory holds the negated values) gives the op's result."""
    from smla import ops
    announce("ops eager route, negative bit")
    x = torch.randn(4, 512, device=dev)
    w = torch.randn(64, 512, device=dev)
    neg = torch._neg_view(x)
    assert neg.is_neg() and neg.is_contiguous()
    assert torch.equal(ops.linear_op(neg, w, 1, torch.float32), ops.linear_op(-x, w, 1, torch.float32))
    idx = ops.topk_op(torch._neg_view(x), 8, None, 0)
    assert torch.equal(idx, ops.topk_op(-x, 8, None, 0))


def test_ops_eager_route_keeps_the_op(dev):
    """Under a profiler the call is listed by the op's name, the op's own methods are there, and an op that a
    caller has extended is used from then on."""
    from smla import ops
    announce("ops eager route, profiler and methods")
    x, w = torch.randn(4, 512, device=dev), torch.randn(64, 512, device=dev)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        ops.linear_op(x, w, 1, torch.float32)
    assert any(e.key == "smla::linear" for e in prof.key_averages())

    @torch.library.custom_op("smla_test::twice", mutates_args=(), device_types="cuda")
    def twice(a: torch.Tensor) -> torch.Tensor:
        return 2 * a

    called = []

    def body(a):
        called.append(a)
        return 2 * a

    op = ops._with_eager_route(twice, body)
    assert torch.equal(op(x), 2 * x) and len(called) == 1
    op.register_autograd(lambda ctx, g: 2 * g)
    leaf = x.clone().requires_grad_()
    op(leaf).sum().backward()
    assert torch.equal(leaf.grad, torch.full_like(x, 2.0))
    assert torch.equal(op(x), 2 * x) and len(called) == 1
