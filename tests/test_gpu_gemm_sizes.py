"""The GEMM kernels at the sizes where their tiles, remainders and dispatch
rules change, against 64-bit products of the same values."""
import pytest
import torch

pytestmark = pytest.mark.gpu

dev = "cuda"


def say(*a):
    print("[case]", *a, flush=True)


# K off and on the matrix kernels' grid (20, 40: the SIMT kernel); rows and
# channels around the 16-, 32- and 64-wide tiles, channel counts not a
# multiple of 4 (element-wise stores), more row tiles than CUs
@pytest.mark.parametrize("n,k,n_out", [(1, 32, 8), (16, 64, 16), (17, 96, 17), (16, 32, 66),
                                       (17, 32, 33), (33, 512, 64), (64, 96, 130), (65, 256, 1000),
                                       (5000, 32, 8), (2100, 64, 640), (40, 20, 48), (129, 40, 70)])
def test_f32_linear_tile_edges(n, k, n_out):
    from spider_moe_amd import ForgeConfig
    from spider_moe_amd.forge import ForgeGEMM
    say("f32 linear", n, k, n_out)
    g = torch.Generator().manual_seed(n * 7 + k + n_out)
    x = torch.randn(n, k, generator=g)
    w = torch.randn(n_out, k, generator=g)
    b = torch.randn(n_out, generator=g)
    y = ForgeGEMM(ForgeConfig()).linear(x.to(dev), w.to(dev), b.to(dev)).cpu().double()
    ref = x.double() @ w.double().t() + b.double()
    # k products and k + 1 sums in f32, in any order: each at most 2^-24 off,
    # relative to the sum of magnitudes
    bound = (2 * k + 2) * 2.0 ** -24 * (x.abs().double() @ w.abs().double().t() + b.abs().double())
    assert bool(((y - ref).abs() <= bound).all())


# experts with no rows, one row and partial tiles; top_k 1 leaves groups of
# about n / e rows: 4 and 16 (16-row tiles), 17 and 100 (32- and 64-row tiles)
@pytest.mark.parametrize("n,h,u,e,k", [(32, 64, 96, 8, 1), (128, 32, 64, 8, 1), (136, 64, 128, 8, 1),
                                       (400, 96, 160, 8, 2), (3000, 64, 320, 5, 2)])
def test_f32_grouped_tile_edges(n, h, u, e, k):
    from spider_moe_amd import sparse_expert_delta
    say("f32 grouped", n, h, u, e, k)
    g = torch.Generator().manual_seed(n + h + u)
    x = torch.randn(1, n, h, generator=g)
    idx = torch.randint(0, e - 1, (n, k), generator=g)  # the last expert stays empty ...
    idx[0, 0] = e - 1                                   # ... but for one row
    idx[1:, 0] = torch.where(idx[1:, 0] == 1, torch.zeros(()).long(), idx[1:, 0])  # expert 1: k > 1 only
    wt = torch.rand(n, k, generator=g) + 0.1
    wu, bu = torch.randn(e, u, h, generator=g) * h ** -0.5, torch.randn(e, u, generator=g)
    wd, bd = torch.randn(e, h, u, generator=g) * u ** -0.5, torch.randn(e, h, generator=g)
    y = sparse_expert_delta(x.to(dev), idx.view(1, n, k).to(dev), wt.view(1, n, k).to(dev), wu.to(dev),
                            bu.to(dev), wd.to(dev), bd.to(dev), num_experts=e, top_k=k).cpu().double()[0]
    ref = torch.zeros(n, h, dtype=torch.float64)
    mag = torch.zeros(n, h, dtype=torch.float64)
    for j in range(k):
        for x_ in range(e):
            r = (idx[:, j] == x_).nonzero().squeeze(-1)
            a = torch.nn.functional.gelu(x[0, r].double() @ wu[x_].double().t() + bu[x_].double())
            ref[r] += (a @ wd[x_].double().t() + bd[x_].double()) * wt[r, j:j + 1].double()
            mag[r] += (a.abs() @ wd[x_].abs().double().t() + bd[x_].abs().double()) * wt[r, j:j + 1].double()
    # the down product's sums as above; an up activation of size ~1 is off by
    # its own sums (h terms) and by erf's 1.5e-7, which the down weights carry on
    up_err = (2 * h + 2) * 2.0 ** -24 * 4 * h ** 0.5 + 2e-7
    bound = (2 * u + 8) * 2.0 ** -24 * mag + up_err * u ** 0.5 * wt.sum(-1, keepdim=True).double()
    assert bool(((y - ref).abs() <= bound).all())


# 33-255 rows per group on average, and any row count of fp8 / int4 without
# tile copies: groups of 0, 1, 64, 65, .. rows (tiles of 64 and 128 rows), K
# of one to five 64-k stages and channels off the 128-wide strips; 140 rows
# per group on average: (192, 320) makes fewer 64 x 128 tiles than CUs (64 x
# 64 tiles), (128, 2696) more (3 stages), (64, 5312) more than two per CU (2
# stages), (128, 456) a partial strip; a third of the rows, (128, 2696): the
# 64-row SwiGLU tiles.  int4 has 64-k scale groups here: the down products of
# U 2752 and 5312 (43 and 83 along K) run on the general kernel, and a third
# of the rows on the int4 stream kernel (test_grouped_mid_int4_scales has the
# scale table's sizes)
@pytest.mark.parametrize("h,u,part", [(192, 320, 1), (128, 2696, 1), (64, 5312, 1), (128, 456, 1),
                                      (128, 2696, 3)])
@pytest.mark.parametrize("fmt,act", [("bf16", "gelu"), ("bf16", "swiglu"), ("fp8", "gelu"),
                                     ("fp8", "swiglu"), ("int4", "gelu"), ("int4", "swiglu")])
def test_grouped_mid_rows(fmt, act, h, u, part):
    from spider_moe_amd import _native as n8
    from spider_moe_amd.quant import (interleave_gate_up, interleave_gate_up_rows,
                                      quantize_fp8_per_channel, quantize_int4)
    from test_gpu_kernels import _experts_struct, _run_delta
    # the down product's K is u: whole 64-k stages, or (2696, 456) bf16 on the
    # vector kernel; fp8 needs 32-k and int4 whole scale groups
    if u % 64 and (fmt != "bf16" or act == "swiglu"):
        u += -u % 64
    say("grouped mid", fmt, act, h, u, part)
    g = torch.Generator().manual_seed(h + u)
    rows = [r // part for r in (0, 3, 64, 65, 260, 300, 129, 300)]
    e, n = len(rows), sum(rows)
    idx = torch.cat([torch.full((r,), x, dtype=torch.int32) for x, r in enumerate(rows)])
    idx = idx[torch.randperm(n, generator=g)].view(n, 1)
    w = torch.rand(n, 1, generator=g) + 0.1
    x = torch.randn(n, h, generator=g).to(torch.bfloat16)
    nup = 2 * u if act == "swiglu" else u
    mats = [torch.randn(e, nup, h, generator=g) * h ** -0.5, torch.randn(e, h, u, generator=g) * u ** -0.5]
    bu, bd = torch.randn(e, u, generator=g) * 0.1, torch.randn(e, h, generator=g) * 0.1
    vals, dev_w, dev_s, kw = [], [], [], {}
    for i, m in enumerate(mats):
        pair = act == "swiglu" and i == 0
        if fmt == "bf16":
            q, s = m.to(torch.bfloat16), None
            vals.append(q.double())
        elif fmt == "fp8":
            q, s = quantize_fp8_per_channel(m)
            q = q.view(torch.float8_e4m3fn)
            vals.append(q.float().double() * s.view(e, -1, 1).double())
            q, s = q.view(torch.uint8), s.view(e, -1).float()
        else:
            p4 = quantize_int4(m, 64, torch.float16)
            q, s = p4.packed, p4.scales
            b = q.view(torch.uint8).int()
            nib = torch.stack([b & 15, b >> 4], -1).view(m.shape)
            nib = torch.where(nib > 7, nib - 16, nib).float()
            # the kernels multiply bf16(q * scale)
            vals.append((nib * s.float().repeat_interleave(64, -1)).to(torch.bfloat16).double())
        dev_w.append((interleave_gate_up(q[:, :u], q[:, u:]) if pair else q).contiguous().to(dev))
        if s is not None and fmt == "fp8":
            s = interleave_gate_up_rows(s[:, :u], s[:, u:]) if pair else s
        elif s is not None:
            s = interleave_gate_up(s[:, :u], s[:, u:]) if pair else s
        dev_s.append(None if s is None else s.contiguous().to(dev))
    if fmt != "bf16":
        kw = dict(s_up=dev_s[0], s_down=dev_s[1], scale_dtype=n8.F16 if fmt == "int4" else n8.F32)
    if fmt == "int4":
        kw["group"] = 64
    bu_d, bd_d = bu.to(dev), bd.to(dev)
    code = {"bf16": n8.BF16, "fp8": n8.FP8_E4M3, "int4": n8.INT4}[fmt]
    ex = _experts_struct(n8, code, n8.ACT_SWIGLU if act == "swiglu" else n8.ACT_GELU, e, h, u, *dev_w,
                         b_up=bu_d, b_down=bd_d, **kw)
    y = _run_delta(n8, ex, x.to(dev), idx.to(dev), w.to(dev)).double()
    xd = x.double()
    for i in range(e):
        r = (idx[:, 0] == i).nonzero().squeeze(-1)
        if not len(r):
            continue
        up = xd[r] @ vals[0][i].t()
        if act == "swiglu":
            a = torch.nn.functional.silu(up[:, :u]) * (up[:, u:] + bu[i].double())
        else:
            a = torch.nn.functional.gelu(up + bu[i].double())
        wt = w[r].double()
        ref = (a @ vals[1][i].t() + bd[i].double()) * wt
        mag = (a.abs() @ vals[1][i].abs().t() + bd[i].abs().double()) * wt
        # bf16 activations and rows: 2^-9 of each product and of the result;
        # f32 sums of u and h terms and the f32 activation functions: far below
        bound = (2.0 ** -9 + (2 * u + 2 * h) * 2.0 ** -24 + 1e-5) * mag + 2.0 ** -9 * ref.abs() + 1e-6
        bad = (y[r] - ref).abs() > 1.01 * bound
        assert not bool(bad.any()), (i, float(((y[r] - ref).abs() / bound).max()))


# one group: f32 results (16-byte stores), fp8 codes on a bf16 input, K tails
# and channels not a multiple of 4 (the general kernel)
@pytest.mark.parametrize("n,k,n_out", [(65, 64, 128), (130, 320, 132), (500, 2816, 1024), (129, 192, 130),
                                       (200, 96, 256), (2100, 128, 2052)])
@pytest.mark.parametrize("fp8", [False, True])
def test_linear_mid_rows(n, k, n_out, fp8):
    from spider_moe_amd.forge import ForgeConfig, ForgeGEMM
    from spider_moe_amd.quant import quantize_fp8_per_tensor
    say("linear mid", n, k, n_out, fp8)
    g = torch.Generator().manual_seed(n + k + n_out)
    x = torch.randn(n, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(n_out, k, generator=g) * k ** -0.5).to(torch.bfloat16)
    b = torch.randn(n_out, generator=g).to(torch.bfloat16)
    y = ForgeGEMM(ForgeConfig(gemm_fp8=fp8)).linear(x.to(dev), w.to(dev), b.to(dev)).cpu().double()
    wv = w.double()
    if fp8:
        codes, scale = quantize_fp8_per_tensor(w)
        wv = codes.view(torch.float8_e4m3fn).float().double() * scale.double()
    ref = x.double() @ wv.t() + b.double()
    # f32 sums of k products, the result rounded to bf16
    bound = 2.0 ** -8 * ref.abs() + (2 * k + 4) * 2.0 ** -24 * (x.abs().double() @ wv.abs().t() + b.abs().double())
    assert bool(((y - ref).abs() <= bound).all())


# decode steps on int4 experts with their tile copy: slices past N_out (H 192,
# U 448), K split over 1, 2 and 4 waves (K 128, 448, 832), groups found by
# lookup (fewer than two rows per expert on average) and directly, scales of
# both types, one per 64 and 128 k
@pytest.mark.parametrize("n,h,u,act", [(1, 192, 448, "gelu"), (7, 832, 128, "swiglu"), (9, 128, 832, "gelu"),
                                       (40, 448, 192, "swiglu"), (100, 832, 448, "gelu")])
@pytest.mark.parametrize("group,sdt", [(64, torch.float16), (64, torch.float32), (128, torch.float16)])
def test_decode_int4_tiles(n, h, u, act, group, sdt):
    from spider_moe_amd import _native as n8
    from spider_moe_amd.quant import interleave_gate_up, quantize_int4
    from test_gpu_kernels import _experts_struct, _run_delta
    if h % group or u % group:
        h, u = -(-h // group) * group, -(-u // group) * group
    say("decode int4 tiles", n, h, u, act, group, sdt)
    e, k = 8, 2
    g = torch.Generator().manual_seed(n + h + u + group)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16)
    idx = torch.stack([torch.randperm(e - 1, generator=g)[:k] for _ in range(n)]).to(torch.int32)
    w = torch.rand(n, k, generator=g) + 0.1
    nup = 2 * u if act == "swiglu" else u
    vals, codes, tiles, scales = [], [], [], []
    for i, (rows, cols) in enumerate(((nup, h), (h, u))):
        q = quantize_int4(torch.randn(e, rows, cols, generator=g) * cols ** -0.5, group, sdt)
        b = q.packed.view(torch.uint8).int()
        nib = torch.stack([b & 15, b >> 4], -1).view(e, rows, cols)
        nib = torch.where(nib > 7, nib - 16, nib).float()
        vals.append((nib * q.scales.float().repeat_interleave(group, -1)).to(torch.bfloat16).double())
        pair = act == "swiglu" and i == 0
        c, s = q.packed, q.scales
        if pair:
            c, s = interleave_gate_up(c[:, :u], c[:, u:]), interleave_gate_up(s[:, :u], s[:, u:])
        codes.append(c.contiguous().to(dev))
        scales.append(s.contiguous().to(dev))
        out = torch.empty_like(codes[-1])
        n8.check(n8.lib().smoe_pack_int4_qtiles(codes[-1].data_ptr(), e, rows, cols, out.data_ptr(),
                                                n8.stream_of(torch.device(dev))), "pack_int4_qtiles")
        tiles.append(out)
    bu, bd = torch.randn(e, u, generator=g) * 0.1, torch.randn(e, h, generator=g) * 0.1
    bu_d, bd_d = bu.to(dev), bd.to(dev)
    ex = _experts_struct(n8, n8.INT4, n8.ACT_SWIGLU if act == "swiglu" else n8.ACT_GELU, e, h, u, *codes,
                         s_up=scales[0], s_down=scales[1], b_up=bu_d, b_down=bd_d, group=group,
                         scale_dtype=n8.F16 if sdt == torch.float16 else n8.F32)
    plain = _run_delta(n8, ex, x.to(dev), idx.to(dev), w.to(dev)).double()
    ex.w_up_tiles, ex.w_down_tiles = tiles[0].data_ptr(), tiles[1].data_ptr()
    tiled = _run_delta(n8, ex, x.to(dev), idx.to(dev), w.to(dev)).double()
    ref, bound = torch.zeros(n, h).double(), torch.zeros(n, h).double()
    for t in range(n):
        for j in range(k):
            i = int(idx[t, j])
            up = x[t].double() @ vals[0][i].t()
            if act == "swiglu":
                a = torch.nn.functional.silu(up[:u]) * (up[u:] + bu[i].double())
            else:
                a = torch.nn.functional.gelu(up + bu[i].double())
            r = (a @ vals[1][i].t() + bd[i].double()) * w[t, j].double()
            mag = (a.abs() @ vals[1][i].abs().t() + bd[i].abs().double()) * w[t, j].double()
            ref[t] += r
            # bf16 activations and rows: 2^-9 of each product and of the row
            bound[t] += (2.0 ** -9 + (2 * u + 2 * h) * 2.0 ** -24 + 1e-5) * mag + 2.0 ** -9 * r.abs() + 1e-6
    for y in (plain, tiled):
        assert bool(((y - ref).abs() <= 1.01 * bound).all()), float(((y - ref).abs() / bound).max())


# fp8 x fp8: row and channel tiles of 128 with remainders, one to five 256-k
# pads, bf16 results in whole 16-byte chunks (staged) and not (direct), inputs
# whose rows are (8 | k) and are not whole vectors
@pytest.mark.parametrize("n,k,n_out", [(1, 256, 128), (127, 100, 8), (128, 1024, 136), (129, 1000, 132),
                                       (300, 7, 130), (257, 1288, 264), (2500, 256, 1416)])
@pytest.mark.parametrize("act", [None, "gelu"])
def test_fp8fp8_tile_edges(n, k, n_out, act):
    from spider_moe_amd.forge import ForgeConfig, ForgeGEMM
    from spider_moe_amd.quant import quantize_fp8_per_tensor
    say("fp8 x fp8", n, k, n_out, act)
    g = torch.Generator().manual_seed(n + k + n_out)
    x = torch.randn(n, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(n_out, k, generator=g) * k ** -0.5).to(torch.bfloat16)
    b = torch.randn(n_out, generator=g)
    y = ForgeGEMM(ForgeConfig(gemm_fp8=True))._run_fp8fp8(x.to(dev), w.to(dev), b.to(dev), act).cpu().double()
    (xq, xs), (wq, ws) = quantize_fp8_per_tensor(x), quantize_fp8_per_tensor(w)
    xv = xq.view(torch.float8_e4m3fn).float().double() * xs.double()
    wv = wq.view(torch.float8_e4m3fn).float().double() * ws.double()
    ref = xv @ wv.t() + b.double()
    # the instruction drops what lies 2^-14 below a 128-block's largest product,
    # of each product; f32 sums of the blocks; GELU's slope is below 1.13;
    # results rounded to bf16 with it
    blocks = -(-k // 128)
    err = (min(k, 128) * blocks * 2.0 ** -14 * xv.abs().amax(1, keepdim=True) * wv.abs().amax(1)
           + (blocks + 3) * 2.0 ** -24 * (xv.abs() @ wv.abs().t() + b.abs().double()))
    if act:
        ref, err = torch.nn.functional.gelu(ref), 1.13 * err + 2.0 ** -8 * torch.nn.functional.gelu(ref).abs() + 1e-6
    assert bool(((y - ref).abs() <= err).all()), float(((y - ref).abs() / err).max())


# the merge + rank launch (K <= 16, more than one chunk) with the one-launch
# finish (4096 tokens over 16 groups) and past it, against the oracle's plan
@pytest.mark.parametrize("n,k,e", [(64, 2, 200), (65, 1, 1), (65, 16, 64), (129, 2, 16), (130, 16, 17),
                                   (4096, 4, 16), (4097, 4, 16), (300, 17, 16), (200, 3, 256)])
def test_merged_plan_edges(n, k, e):
    import test_gpu_kernels
    test_gpu_kernels.test_dispatch_plan_bit_exact(n, k, e)


def _whole_experts(fmt, act, up, down, group=128, tiles=False):
    """Experts on whole-number weights in -8 .. 7, which every format holds
    exactly (scales 1): up [e, nup, h] (SwiGLU: gate, then up), down [e, h, u]."""
    from spider_moe_amd import _native as n8
    from spider_moe_amd.quant import interleave_gate_up
    from test_gpu_kernels import _experts_struct
    e, h, u = down.shape
    if act == "swiglu":
        up = interleave_gate_up(up[:, :u], up[:, u:])
    keep, kw = [], {}
    for name, m in (("up", up), ("down", down)):
        if fmt == "bf16":
            keep.append(m.to(torch.bfloat16).contiguous().to(dev))
        elif fmt == "fp8":
            keep.append(m.float().to(torch.float8_e4m3fn).view(torch.uint8).contiguous().to(dev))
            kw["s_" + name] = torch.ones(m.shape[:2], device=dev)
        else:
            q = m.int() & 15
            keep.append((q[..., ::2] | q[..., 1::2] << 4).to(torch.uint8).contiguous().to(dev))
            kw["s_" + name] = torch.ones(*m.shape[:2], m.shape[2] // group, dtype=torch.float16, device=dev)
    if fmt != "bf16":
        kw["scale_dtype"] = n8.F16 if fmt == "int4" else n8.F32
    if fmt == "int4":
        kw["group"] = group
    code = {"bf16": n8.BF16, "fp8": n8.FP8_E4M3, "int4": n8.INT4}[fmt]
    ex = _experts_struct(n8, code, n8.ACT_SWIGLU if act == "swiglu" else n8.ACT_GELU, e, h, u, *keep, **kw)
    if tiles:  # int4
        for name, m, w in (("up", up, keep[0]), ("down", down, keep[1])):
            t = torch.empty_like(w)
            n8.check(n8.lib().smoe_pack_int4_qtiles(w.data_ptr(), e, m.shape[1], m.shape[2], t.data_ptr(),
                                                    n8.stream_of(torch.device(dev))), "pack_int4_qtiles")
            setattr(ex, f"w_{name}_tiles", t.data_ptr())
            keep.append(t)
    return ex, (keep, kw)


def _whole_weights(g, e, h, u, act):
    nup = 2 * u if act == "swiglu" else u
    return (torch.randint(-8, 8, (e, nup, h), generator=g), torch.randint(-8, 8, (e, h, u), generator=g))


# 33-128 rows per group: every format sums a 64-k step in the order of the
# int4 stream kernel (MFMAs over the low and the high 8 of 16 consecutive k),
# so weights that all three hold exactly give the same bits.  36, 97 and 128
# rows per group on average, 0 to 300 in one; 11 and 2 steps of K
@pytest.mark.parametrize("n,h,u", [(288, 256, 704), (776, 128, 1408), (1024, 640, 256)])
@pytest.mark.parametrize("act", ["gelu", "swiglu"])
def test_grouped_mid_rows_sum_order(n, h, u, act):
    from spider_moe_amd import _native as n8
    from test_gpu_kernels import _run_delta
    say("mid rows, sum order", n, h, u, act)
    g = torch.Generator().manual_seed(n + u)
    e, group = 8, 64 if u % 128 else 128
    ids = torch.multinomial(torch.tensor([.3, .25, .15, .1, .1, .06, .04, 0.]), n, True, generator=g)
    up, down = _whole_weights(g, e, h, u, act)
    x = (torch.randn(n, h, generator=g) * 0.05).to(torch.bfloat16)
    w = torch.rand(n, 1, generator=g) + 0.1
    got = []
    for fmt in ("int4", "bf16", "fp8"):
        ex, keep = _whole_experts(fmt, act, up, down, group)
        got.append(_run_delta(n8, ex, x.to(dev), ids.int().view(n, 1).to(dev), w.to(dev)))
    assert bool(got[0].isfinite().all()) and float(got[0].abs().max()) > 0
    for y in got[1:]:
        assert torch.equal(y, got[0]), float((y != got[0]).float().mean())


# decode steps on int4 experts: the same bits from the packed rows and from
# the tile copy (K split over 1, 2 and 4 waves, groups looked up and direct)
@pytest.mark.parametrize("n,h,u", [(1, 128, 448), (7, 1024, 704), (40, 832, 192), (60, 448, 1408),
                                   (100, 704, 448)])
@pytest.mark.parametrize("act", ["gelu", "swiglu"])
def test_decode_int4_tiles_sum_order(n, h, u, act):
    from spider_moe_amd import _native as n8
    from test_gpu_kernels import _run_delta
    say("decode int4 tiles, sum order", n, h, u, act)
    g = torch.Generator().manual_seed(n + h + u)
    e, k = 8, 2
    idx = torch.stack([torch.randperm(e - 1, generator=g)[:k] for _ in range(n)]).int()
    up, down = _whole_weights(g, e, h, u, act)
    x = (torch.randn(n, h, generator=g) * 0.05).to(torch.bfloat16)
    w = torch.rand(n, k, generator=g) + 0.1
    got = []
    for tiles in (False, True):
        ex, keep = _whole_experts("int4", act, up, down, 64, tiles)
        got.append(_run_delta(n8, ex, x.to(dev), idx.to(dev), w.to(dev)))
    assert torch.equal(*got), float((got[0] != got[1]).float().mean())


# int4 experts whose codes or biases lie off 16-byte boundaries, at the row
# counts of the int4 stream kernel (16-byte loads): a kernel without them
@pytest.mark.parametrize("off", ["codes", "bias"])
def test_int4_stream_unaligned_operands(off):
    from spider_moe_amd import _native as n8
    from test_gpu_kernels import _run_delta
    say("int4 stream, unaligned", off)
    e, n, h, u = 4, 300, 256, 320
    g = torch.Generator().manual_seed(3)
    idx = torch.randint(0, e, (n, 1), generator=g).int()
    up, down = _whole_weights(g, e, h, u, "gelu")
    x = (torch.randn(n, h, generator=g) * 0.05).to(torch.bfloat16)
    w = torch.rand(n, 1, generator=g) + 0.1
    ex, (mats, kw) = _whole_experts("int4", "gelu", up, down, 64)
    bu, bd = torch.randn(e, u, generator=g), torch.randn(e, h, generator=g)
    bias = [torch.nn.functional.pad(b.flatten(), (1, 0)).to(dev)[1:] for b in (bu, bd)]
    if off == "codes":
        mats = [torch.nn.functional.pad(m.flatten(), (8, 0))[8:] for m in mats]
        bias = [b.clone() for b in bias]
        ex.w_up, ex.w_down = mats[0].data_ptr(), mats[1].data_ptr()
    ex.b_up, ex.b_down = bias[0].data_ptr(), bias[1].data_ptr()
    assert ex.w_up % 16 == (8 if off == "codes" else 0) and ex.b_up % 16 == (0 if off == "codes" else 4)
    y = _run_delta(n8, ex, x.to(dev), idx.to(dev), w.to(dev)).double()
    for i in range(e):
        r = (idx[:, 0] == i).nonzero().squeeze(-1)
        a = torch.nn.functional.gelu(x[r].double() @ up[i].double().t() + bu[i].double())
        ref = (a @ down[i].double().t() + bd[i].double()) * w[r].double()
        mag = (a.abs() @ down[i].abs().double().t() + bd[i].abs().double()) * w[r].double()
        # bf16 (8 significant bits: 2^-8) activations, of each product, and rows;
        # f32 sums of u and h terms and the f32 activation: far below
        bound = (2.0 ** -8 + (2 * u + 2 * h) * 2.0 ** -24 + 1e-5) * mag + 2.0 ** -8 * ref.abs() + 1e-6
        assert bool(((y[r] - ref).abs() <= bound).all()), float(((y[r] - ref).abs() / bound).max())


# 33-128 rows per group, bf16 rows of an odd number of 8-byte pieces: the same
# bits as with 4 channels more (the down weights pick one channel each, so the
# delta is the up product's row, scaled)
@pytest.mark.parametrize("n,h,u", [(160, 320, 324), (500, 128, 1004)])
def test_grouped_mid_rows_four_channel_stores(n, h, u):
    from spider_moe_amd import _native as n8
    from test_gpu_kernels import _experts_struct, _run_delta
    say("mid rows, 4-channel stores", n, h, u)
    g = torch.Generator().manual_seed(n + u)
    e = 4
    idx = torch.multinomial(torch.tensor([.5, .3, .2, 0.]), n, True, generator=g).int().view(n, 1)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16)
    w = torch.rand(n, 1, generator=g) + 0.1
    up = (torch.randn(e, u + 4, h, generator=g) * h ** -0.5).to(torch.bfloat16)
    bu = torch.randn(e, u + 4, generator=g)
    got = []
    for c in (u, u + 4):
        down = torch.zeros(e, h, c, dtype=torch.bfloat16)
        down[:, torch.arange(h), torch.arange(h) + u - h] = 1
        keep = [t.contiguous().to(dev) for t in (up[:, :c], down, bu[:, :c])]
        ex = _experts_struct(n8, n8.BF16, n8.ACT_GELU, e, h, c, keep[0], keep[1], b_up=keep[2])
        got.append(_run_delta(n8, ex, x.to(dev), idx.to(dev), w.to(dev)))
    assert float(got[0].abs().max()) > 0 and torch.equal(*got), float((got[0] != got[1]).float().mean())


# int4 at 140 rows per group without tile copies: scale tables of one to 32
# groups along the down product's K, the most that the tiles hold (64 x 32, 128 x
# 22), and 33 (the general kernel), scales of both types
@pytest.mark.parametrize("u,group", [(128, 128), (192, 64), (2048, 64), (2816, 128), (4096, 128), (2112, 64)])
@pytest.mark.parametrize("sdt", [torch.float16, torch.float32])
def test_grouped_mid_int4_scales(u, group, sdt):
    from spider_moe_amd import _native as n8
    from spider_moe_amd.quant import quantize_int4
    from test_gpu_kernels import _experts_struct, _run_delta
    say("int4 mid scales", u, group, sdt)
    g = torch.Generator().manual_seed(u + group)
    h, rows = 128, [300, 130, 0, 260, 65, 300, 1, 64]
    e, n = len(rows), sum(rows)
    idx = torch.cat([torch.full((r,), x, dtype=torch.int32) for x, r in enumerate(rows)])
    idx = idx[torch.randperm(n, generator=g)].view(n, 1)
    x, w = torch.randn(n, h, generator=g).to(torch.bfloat16), torch.rand(n, 1, generator=g) + 0.1
    bu, bd = torch.randn(e, u, generator=g) * 0.1, torch.randn(e, h, generator=g) * 0.1
    vals, packed, scales = [], [], []
    for o, k in ((u, h), (h, u)):
        # magnitudes that differ from one scale group to the next
        m = torch.randn(e, o, k, generator=g) * k ** -0.5 * (torch.rand(e, o, k // group, 1, generator=g) * 4 + 0.1) \
            .expand(-1, -1, -1, group).reshape(e, o, k)
        q = quantize_int4(m, group, sdt)
        b = q.packed.view(torch.uint8).int()
        nib = torch.stack([b & 15, b >> 4], -1).view(m.shape)
        nib = torch.where(nib > 7, nib - 16, nib).float()
        vals.append((nib * q.scales.float().repeat_interleave(group, -1)).to(torch.bfloat16).double())
        packed.append(q.packed.contiguous().to(dev))
        scales.append(q.scales.contiguous().to(dev))
    bias = [bu.to(dev), bd.to(dev)]
    ex = _experts_struct(n8, n8.INT4, n8.ACT_GELU, e, h, u, *packed, s_up=scales[0], s_down=scales[1],
                         b_up=bias[0], b_down=bias[1], group=group,
                         scale_dtype=n8.F16 if sdt == torch.float16 else n8.F32)
    y = _run_delta(n8, ex, x.to(dev), idx.to(dev), w.to(dev)).double()
    for i in range(e):
        r = (idx[:, 0] == i).nonzero().squeeze(-1)
        if not len(r):
            continue
        a = torch.nn.functional.gelu(x[r].double() @ vals[0][i].t() + bu[i].double())
        ref = (a @ vals[1][i].t() + bd[i].double()) * w[r].double()
        mag = (a.abs() @ vals[1][i].abs().t() + bd[i].abs().double()) * w[r].double()
        # as in test_int4_stream_unaligned_operands
        bound = (2.0 ** -8 + (2 * u + 2 * h) * 2.0 ** -24 + 1e-5) * mag + 2.0 ** -8 * ref.abs() + 1e-6
        assert bool(((y[r] - ref).abs() <= bound).all()), (i, float(((y[r] - ref).abs() / bound).max()))
