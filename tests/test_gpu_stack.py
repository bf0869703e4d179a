"""xdna::qwen3_stack on the MI355X: its HIP kernels against float64 references, and the fused op
through torch.compile against the oracle (oracle/qwen3_stack.py, pinned to transformers'
Qwen3Model) and against the model run eagerly in float32 (the reference's own check, 10%).

Tolerances: the kernels round to bf16 (GEMM operands, q / k / v, attention probabilities), so
element checks allow 2 bf16 ulps and sequence checks a relative norm of 2e-2 (bf16 carries 8 bits:
a relative error of ~4e-3 per rounding, accumulated over the layers); the fused op against the fp32
model uses the reference test's 8% bound for its bfp16 NPU path.
"""
import pytest
import torch

from models import Stack, prefix_mask, rel_err
from oracle import qwen3_stack as Q

pytestmark = pytest.mark.gpu

BF16_ULP = 2.0 ** -7


def _close_bf16(got, want, ulps=2):
    """|got - want| <= ulps bf16 ulps of |want| (plus a floor for values near 0)."""
    got, want = got.double().cpu(), want.double().cpu()
    tol = ulps * BF16_ULP * want.abs() + 1e-6
    bad = (got - want).abs() > tol
    assert not bool(bad.any()), f"{int(bad.sum())} of {want.numel()} values differ, max {float((got - want).abs().max())}"


def test_rmsnorm_bf16(gpu):
    from torch_xdna import kernels

    g = torch.Generator().manual_seed(1)
    x = torch.randn(37, 1024, generator=g) * 3
    w = 1 + 0.1 * torch.randn(1024, generator=g)
    for wt in (w, w.to(torch.bfloat16)):
        y = kernels.rmsnorm_bf16(x.to(gpu), wt.to(gpu), 1e-6)
        _close_bf16(y, Q.rms_norm(x.double(), wt.double(), 1e-6))


def test_add_rmsnorm_bf16(gpu):
    """The residual add fused into the norm: x after the launch equals x + a in float32 (torch's CPU sum),
    and the normalized output equals the separate add then norm launches bit for bit (and the float64
    norm of x + a within the bf16 tolerance), for d of 1024 and 4096 and both weight dtypes."""
    from torch_xdna import kernels

    g = torch.Generator().manual_seed(11)
    for d in (1024, 4096):
        x = torch.randn(41, d, generator=g) * 3
        a = torch.randn(41, d, generator=g)
        w = 1 + 0.1 * torch.randn(d, generator=g)
        for wt in (w, w.to(torch.bfloat16)):
            xf = x.to(gpu)
            y = kernels.add_rmsnorm_bf16(xf, a.to(gpu), wt.to(gpu), 1e-6)
            assert torch.equal(xf.cpu(), x + a)
            xs = x.to(gpu)
            kernels.add_(xs, a.to(gpu))
            assert torch.equal(y, kernels.rmsnorm_bf16(xs, wt.to(gpu), 1e-6)), (d, wt.dtype)
            _close_bf16(y, Q.rms_norm((x + a).double(), wt.double(), 1e-6))


@pytest.mark.parametrize("tile", ["t64x64", "t32x64k4", "t128x128", "t256x256w8", "small_w2", "gemv_w4", "seg4_r2"])
def test_gemm_bf16_silu(gpu, tile):
    """The gate|up GEMM with SiLU(gate) * up in its epilogue, on the interleaved weight, against the float32
    GEMM of the concatenated weight then the separate SiLU kernel, with the same tile forced on both (their
    float sums then match), bit for bit; rows from 1 to 486, ragged rows and K, and the one-row and few-row
    tiles, which the fused form replaces by the small-M kernel (there only the float64 bound is checked)."""
    from torch_xdna import kernels

    kernels.use_tuned(False)
    kernels.tile_clear()
    try:
        g = torch.Generator().manual_seed(5)
        for m, inter, k in [(1, 3072, 1024), (5, 256, 1024), (16, 260, 40), (70, 3072, 1024), (486, 3072, 1024)]:
            x = (torch.randn(m, k, generator=g)).to(torch.bfloat16)
            gate = (torch.randn(inter, k, generator=g) * 0.05).to(torch.bfloat16)
            up = (torch.randn(inter, k, generator=g) * 0.05).to(torch.bfloat16)
            kernels.tile_set("bf16", m, 2 * inter, k, tile)
            xg = x.to(gpu)
            y = kernels.mm_bf16_silu(xg, kernels.gate_up_interleaved(gate, up).to(gpu))
            assert y.shape == (m, inter) and y.dtype == torch.bfloat16
            ref = kernels.silu_mul_bf16(kernels.mm_bf16(xg, torch.cat([gate, up]).to(gpu), None, torch.float32))
            if not tile.startswith(("gemv", "seg4")):
                assert torch.equal(y, ref), (tile, m, inter, k)
            gd, ud = x.double() @ gate.double().t(), x.double() @ up.double().t()
            want = torch.nn.functional.silu(gd) * ud
            err = (y.double().cpu() - want).abs().max() / want.abs().max()
            assert err < 2e-2, (tile, m, inter, k, float(err))
            kernels.tile_set("bf16", m, 2 * inter, k, "auto")
    finally:
        kernels.tile_clear()
        kernels._tuned_applied = None


def test_qk_norm_rope(gpu):
    """q / k heads RMSNorm'd and rotated at each token's own position; v lands transposed at its column."""
    from torch_xdna import kernels

    g = torch.Generator().manual_seed(2)
    T, nh, nkv = 45, 16, 8
    qkv = torch.randn(T, (nh + 2 * nkv) * 128, generator=g)
    qw, kw = 1 + 0.1 * torch.randn(128, generator=g), 1 + 0.1 * torch.randn(128, generator=g)
    inv_freq = 1.0 / (1e6 ** (torch.arange(0, 128, 2, dtype=torch.float32) / 128))
    pos = torch.randint(0, 400, (T,), generator=g, dtype=torch.int32)
    vt_col = torch.randperm(T + 19, generator=g)[:T].to(torch.int32)
    vt = torch.zeros(nkv, 128, 64, dtype=torch.bfloat16, device=gpu)
    q, k = kernels.qk_norm_rope(qkv.to(gpu), nh, nkv, qw.to(gpu), kw.to(gpu), inv_freq.to(gpu), pos.to(gpu),
                                vt_col.to(gpu), 1e-6, vt)
    x = qkv.double()
    for heads, off, w, got in ((nh, 0, qw, q), (nkv, nh * 128, kw, k)):
        h = Q.rms_norm(x[:, off:off + heads * 128].view(T, heads, 128), w.double(), 1e-6)
        ang = pos.float()[:, None] * inv_freq[None, :]                         # float32 angles
        ang = torch.cat([ang, ang], -1)[:, None, :]
        rot = torch.cat([-h[..., 64:], h[..., :64]], -1)
        _close_bf16(got, h * ang.cos().double() + rot * ang.sin().double())
    v = qkv[:, (nh + nkv) * 128:].view(T, nkv, 128).to(torch.bfloat16)
    got_v = vt.cpu()[:, :, vt_col.long()].permute(2, 0, 1)
    assert torch.equal(got_v, v)


@pytest.mark.parametrize("d,rows", [(256, 3), (768, 70), (1280, 5), (4096, 2)])
@pytest.mark.parametrize("shift", [0, 1])
def test_rmsnorm_bf16_widths(gpu, d, rows, shift):
    """Row widths at the edges of the one-wave and four-wave forms, and operands one element past a 16-byte
    boundary: the norm and the add + norm within two bf16 ulps of float64, x after the add exactly x + a."""
    from torch_xdna import kernels

    g = torch.Generator().manual_seed(d + rows)

    def moved(t):
        buf = torch.empty(t.numel() + shift, dtype=t.dtype, device=gpu)
        buf[shift:].copy_(t.reshape(-1))
        return buf[shift:].view(t.shape)

    x, a = torch.randn(rows, d, generator=g), torch.randn(rows, d, generator=g)
    for wt in (torch.float32, torch.bfloat16, torch.float16):
        w = (1 + 0.1 * torch.randn(d, generator=g)).to(wt)
        _close_bf16(kernels.rmsnorm_bf16(moved(x), moved(w), 1e-6), Q.rms_norm(x.double(), w.double(), 1e-6))
        xg = moved(x)
        _close_bf16(kernels.add_rmsnorm_bf16(xg, moved(a), moved(w), 1e-6), Q.rms_norm((x + a).double(), w.double(), 1e-6))
        assert torch.equal(xg.cpu(), x + a)


@pytest.mark.parametrize("T,nh,nkv,perm", [(1, 16, 8, False), (31, 16, 8, False), (32, 4, 4, True), (33, 6, 1, False),
                                           (97, 3, 1, True)])
def test_qk_norm_rope_forms(gpu, T, nh, nkv, perm):
    """Token counts at the edges of the V copy's 32-token blocks, head counts off the eight half waves, V columns
    in order and permuted: q and k within two bf16 ulps of float64, V exactly the rounded values in their columns
    and nothing else written."""
    from torch_xdna import kernels

    g = torch.Generator().manual_seed(T + nh)
    qkv = torch.randn(T, (nh + 2 * nkv) * 128, generator=g)
    qw, kw = 1 + 0.1 * torch.randn(128, generator=g), 1 + 0.1 * torch.randn(128, generator=g)
    inv_freq = 1.0 / (1e6 ** (torch.arange(0, 128, 2, dtype=torch.float32) / 128))
    pos = torch.randint(0, 4096, (T,), generator=g, dtype=torch.int32)
    col = (torch.randperm(T + 24, generator=g)[:T] if perm else torch.arange(T) + 8).to(torch.int32)
    vt = torch.full((nkv, 128, T + 32), 7.0, dtype=torch.bfloat16, device=gpu)
    q, k = kernels.qk_norm_rope(qkv.to(gpu), nh, nkv, qw.to(gpu), kw.to(gpu), inv_freq.to(gpu), pos.to(gpu),
                                col.to(gpu), 1e-6, vt)
    x = qkv.double()
    for heads, off, w, got in ((nh, 0, qw, q), (nkv, nh * 128, kw, k)):
        h = Q.rms_norm(x[:, off:off + heads * 128].view(T, heads, 128), w.double(), 1e-6)
        ang = pos.float()[:, None] * inv_freq[None, :]
        ang = torch.cat([ang, ang], -1)[:, None, :]
        rot = torch.cat([-h[..., 64:], h[..., :64]], -1)
        # near-cancelling pairs: float32 errors of the two products (2^-22 of their size) under the two ulps
        err = (got.double().cpu() - (h * ang.cos().double() + rot * ang.sin().double())).abs()
        assert bool((err <= 2 * BF16_ULP * got.double().cpu().abs() + 1e-5).all())
    want = torch.full((nkv, 128, T + 32), 7.0, dtype=torch.bfloat16)
    want[:, :, col.long()] = qkv[:, (nh + nkv) * 128:].view(T, nkv, 128).to(torch.bfloat16).permute(1, 2, 0)
    assert torch.equal(vt.cpu(), want)


@pytest.mark.parametrize("lens", [[1], [31, 32, 33], [100, 65, 7], [257]])
def test_attention_bf16(gpu, lens):
    """Ragged sequences (partial and single query / key blocks): each sequence's heads against the
    float64 attention of the same bf16 q / k / v."""
    from torch_xdna import kernels

    g = torch.Generator().manual_seed(sum(lens))
    nh, nkv = 16, 8
    T = sum(lens)
    q = (torch.randn(T, nh, 128, generator=g) * 2).to(torch.bfloat16)
    k = (torch.randn(T, nkv, 128, generator=g) * 2).to(torch.bfloat16)
    v = torch.randn(T, nkv, 128, generator=g).to(torch.bfloat16)
    starts, vts, s, c = [], [], 0, 0
    for n in lens:
        starts.append(s)
        vts.append(c)
        s, c = s + n, c + -(-n // 32) * 32
    vt = torch.zeros(nkv, 128, -(-c // 8) * 8, dtype=torch.bfloat16)
    for n, s0, c0 in zip(lens, starts, vts):
        vt[:, :, c0:c0 + n] = v[s0:s0 + n].permute(1, 2, 0)
    i32 = dict(dtype=torch.int32, device=gpu)
    out = kernels.attention_bf16(q.to(gpu), k.to(gpu), vt.to(gpu), torch.tensor(starts, **i32),
                                 torch.tensor(lens, **i32), torch.tensor(vts, **i32), max(lens), 128 ** -0.5)
    out = out.cpu().double()
    for n, s0 in zip(lens, starts):
        want = Q.attention(q[s0:s0 + n].double(), k[s0:s0 + n].double(), v[s0:s0 + n].double())
        assert rel_err(out[s0:s0 + n], want) < 1e-2, n


@pytest.mark.parametrize("nh,nkv,scale,lens", [
    (16, 8, 128 ** -0.5, [2048]),                    # 128-row workgroups: whole tiles only
    (16, 8, 128 ** -0.5, [2049, 65, 1, 64]),         # a last tile of one key, sequences far below the longest
    (16, 8, -0.05, [1100, 1023, 130]),               # a negative scale
    (8, 8, 128 ** -0.5, [1999, 2500]),               # one q head per kv head
    (24, 8, 128 ** -0.5, [700, 701]),                # three
    (6, 1, 128 ** -0.5, [150, 3, 32, 33]),           # one kv head; 32-row workgroups with the keys split
    (16, 8, -0.05, [97, 128, 129]),
    (3, 3, 0.0, [40, 200])])                         # scale 0: the mean of V
def test_attention_bf16_forms(gpu, nh, nkv, scale, lens):
    """Both workgroup forms at the edges of their key tiles and row blocks, and head groupings, scale signs:
    each sequence against the float64 attention of the same bf16 values. P and the output are rounded to bf16
    (2^-9 relative each, averaged over the keys): 1e-2 in relative norm."""
    from torch_xdna import kernels

    g = torch.Generator().manual_seed(sum(lens) + nh)
    T = sum(lens)
    q = (torch.randn(T, nh, 128, generator=g) * 2).to(torch.bfloat16)
    k = (torch.randn(T, nkv, 128, generator=g) * 2).to(torch.bfloat16)
    v = torch.randn(T, nkv, 128, generator=g).to(torch.bfloat16)
    starts, vts, s, c = [], [], 0, 0
    for n in lens:
        starts.append(s)
        vts.append(c)
        s, c = s + n, c + -(-n // 32) * 32
    vt = torch.zeros(nkv, 128, c, dtype=torch.bfloat16)
    for n, s0, c0 in zip(lens, starts, vts):
        vt[:, :, c0:c0 + n] = v[s0:s0 + n].permute(1, 2, 0)
    i32 = dict(dtype=torch.int32, device=gpu)
    out = kernels.attention_bf16(q.to(gpu), k.to(gpu), vt.to(gpu), torch.tensor(starts, **i32),
                                 torch.tensor(lens, **i32), torch.tensor(vts, **i32), max(lens), scale)
    out = out.cpu().double()
    for n, s0 in zip(lens, starts):
        for h in range(nh):
            kv = h // (nh // nkv)
            p = torch.softmax(q[s0:s0 + n, h].double() @ k[s0:s0 + n, kv].double().t() * scale, dim=-1)
            assert rel_err(out[s0:s0 + n, h], p @ v[s0:s0 + n, kv].double()) < 1e-2, (n, h)


@pytest.mark.parametrize("nh,nkv,lens", [(16, 8, [1]), (16, 8, [32, 5, 31]), (6, 1, [17, 32]), (16, 8, [20] * 40), (16, 8, [33]),
                                         (16, 8, [64, 1, 32, 63]), (3, 3, [50] * 9), (6, 1, [64, 33]), (16, 8, [65, 20])])
def test_attention_short_sequences(gpu, nh, nkv, lens):
    """The forms of one wave (a longest sequence of up to 32 tokens), two (64) and four per row block, at their
    edges: as test_attention_bf16_forms."""
    test_attention_bf16_forms(gpu, nh, nkv, 128 ** -0.5, lens)


@pytest.mark.parametrize("n", [1536, 1999])
def test_attention_bf16_weights(gpu, n):
    """The 128-row form rounds its weights to bf16 against a maximum that follows every 32 keys: the output is that of the
    same online softmax in float64, rounded to bf16. What is left is the weights and outputs that float32 puts on the
    other side of a bf16 rounding boundary, 2^-14 of them for errors of 2^-24 of arguments up to 10 and steps of 2^-9, each
    2^-8 of itself: some 1e-4 in relative norm (a maximum per 64 keys is 1.1e-3 away)."""
    from torch_xdna import kernels

    nh, nkv, scale = 16, 8, 128 ** -0.5
    g = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(n, h, 128, generator=g).to(torch.bfloat16) for h in (nh, nkv, nkv))
    vt = torch.zeros(nkv, 128, -(-n // 32) * 32, dtype=torch.bfloat16)
    vt[:, :, :n] = v.permute(1, 2, 0)
    i32 = dict(dtype=torch.int32, device=gpu)
    out = kernels.attention_bf16(q.to(gpu), k.to(gpu), vt.to(gpu), torch.tensor([0], **i32), torch.tensor([n], **i32),
                                 torch.tensor([0], **i32), n, scale).cpu().double()
    for h in (0, 5, 15):
        s = q[:, h].double() @ k[:, h // 2].double().t() * scale
        m = torch.full((n, 1), -float("inf"), dtype=torch.float64)
        l, o = torch.zeros(n, 1, dtype=torch.float64), torch.zeros(n, 128, dtype=torch.float64)
        for b in range(0, n, 32):
            mn = torch.maximum(m, s[:, b:b + 32].amax(1, keepdim=True))
            p = torch.exp(s[:, b:b + 32] - mn)
            l = l * torch.exp(m - mn) + p.sum(1, keepdim=True)
            o = o * torch.exp(m - mn) + p.to(torch.bfloat16).double() @ v[b:b + 32, h // 2].double()
            m = mn
        assert rel_err(out[:, h], (o / l).to(torch.bfloat16).double()) < 4e-4, h


@pytest.mark.parametrize("n,keys,value,mixed", [
    (97, (0, 32), "-inf", 0), (200, (32, 64), "-inf", 0), (200, (96, 200), "-inf", 0), (300, (0, 299), "-inf", 0),
    (33, (0, 33), "-inf", 0),                                   # every key: no weights, NaN
    (200, (64, 96), "inf", 0), (200, (40, 41), "nan", 0), (130, (0, 128), "-inf", 1),
    (2048, (0, 64), "-inf", 0), (2049, (64, 2048), "-inf", 0), (2048, (0, 2048), "-inf", 0), (2048, (70, 71), "nan", 0),
    (2048, (0, 1000), "-inf", 1)])
def test_attention_infinite_scores(gpu, n, keys, value, mixed):
    """Scores of -inf (whole key tiles of them, first, last and all of a wave's), +inf and NaN, in both workgroup
    forms: every row as the float64 softmax has it, weight 0 for -inf, NaN where that is NaN. mixed: the
    even rows' queries turn the keys' -inf into +inf (NaN rows between finite ones)."""
    from torch_xdna import kernels

    nh, nkv = 16, 8
    g = torch.Generator().manual_seed(n + keys[0])
    q = torch.randn(n, nh, 128, generator=g).to(torch.bfloat16)
    k = torch.randn(n, nkv, 128, generator=g).to(torch.bfloat16)
    v = torch.randn(n, nkv, 128, generator=g).to(torch.bfloat16)
    q[:, :, 0] = 1.0                                            # times -inf: -inf
    if mixed:
        q[::2, :, 0] = -1.0
    k[:, :, 0] = 0.0
    k[keys[0]:keys[1], :, 0] = float(value)
    vt = torch.zeros(nkv, 128, -(-n // 32) * 32, dtype=torch.bfloat16)
    vt[:, :, :n] = v.permute(1, 2, 0)
    i32 = dict(dtype=torch.int32, device=gpu)
    out = kernels.attention_bf16(q.to(gpu), k.to(gpu), vt.to(gpu), torch.tensor([0], **i32), torch.tensor([n], **i32),
                                 torch.tensor([0], **i32), n, 128 ** -0.5).cpu().double()
    for h in range(nh):
        p = torch.softmax(q[:, h].double() @ k[:, h // 2].double().t() * 128 ** -0.5, dim=-1)
        want, got = p @ v[:, h // 2].double(), out[:, h]
        nan = want.isnan()
        assert torch.equal(got.isnan(), nan), h
        if not nan.all():       # the tolerance of test_attention_bf16_forms
            assert rel_err(got[~nan], want[~nan]) < 1e-2, h


def test_more_workgroups_than_a_launch(gpu):
    """Calls whose workgroups are more than one launch takes (2^24 of 256 threads): 2^21 + 3 short sequences of 8 kv
    heads, and 2^24 + 40 tokens of one head; what the last launch does is that of a call of its own."""
    from torch_xdna import kernels

    g = torch.Generator().manual_seed(2)
    rand = lambda *s: torch.randn(*s, generator=g)
    i32 = dict(dtype=torch.int32, device=gpu)
    q, k = (rand(40, 8, 128).to(torch.bfloat16).to(gpu) for _ in range(2))
    vt = rand(8, 128, 64).to(torch.bfloat16).to(gpu)
    nseq = 2 ** 21 + 3
    start, length = torch.zeros(nseq, **i32), torch.ones(nseq, **i32)
    start[-2:], length[-2:] = torch.tensor([1, 3], **i32), torch.tensor([2, 37], **i32)
    col = torch.zeros(nseq, **i32)
    col[-1] = 8
    out = kernels.attention_bf16(q, k, vt, start, length, col, 40, 128 ** -0.5)
    want = kernels.attention_bf16(q, k, vt, start[-3:].contiguous(), length[-3:].contiguous(), col[-3:].contiguous(), 40,
                                  128 ** -0.5)
    assert rel_err(out.double().cpu(), want.double().cpu()) < 1e-2     # the two forms: as test_attention_bf16_forms

    T = 2 ** 24 + 40
    qkv = torch.zeros(T, 3 * 128, device=gpu)
    qkv[-64:] = rand(64, 3 * 128).to(gpu)
    w, freq = (1 + 0.1 * rand(128)).to(gpu), (1.0 / (1e6 ** (torch.arange(0, 128, 2) / 128))).to(gpu)
    pos, col = torch.zeros(T, **i32), torch.zeros(T, **i32)
    pos[-64:], col[-64:] = torch.arange(64, **i32), torch.arange(64, **i32)
    qkv[:-64, 256:] = qkv[-64, 256:]                                   # all other tokens' V go to column 0 too
    vt = torch.zeros(1, 128, 64, dtype=torch.bfloat16, device=gpu)
    got = kernels.qk_norm_rope(qkv, 1, 1, w, w, freq, pos, col, 1e-6, vt)
    vt2 = torch.zeros_like(vt)
    want = kernels.qk_norm_rope(qkv[-64:], 1, 1, w, w, freq, pos[-64:], col[-64:], 1e-6, vt2)
    assert torch.equal(got[0][-64:], want[0]) and torch.equal(got[1][-64:], want[1]) and torch.equal(vt, vt2)


def test_silu_mul_and_add(gpu):
    from torch_xdna import kernels

    g = torch.Generator().manual_seed(3)
    gu = torch.randn(29, 2 * 3072, generator=g) * 3
    y = kernels.silu_mul_bf16(gu.to(gpu))
    gd = gu.double()
    _close_bf16(y, torch.nn.functional.silu(gd[:, :3072]) * gd[:, 3072:])
    a, b = torch.randn(1000, generator=g), torch.randn(1000, generator=g)
    ag = a.to(gpu)
    kernels.add_(ag, b.to(gpu))
    assert torch.equal(ag.cpu(), a + b)


def _stats():
    from torch_xdna import runtime

    return runtime.stats.as_dict()


def _compiled(net):
    from torch_xdna import runtime

    torch._dynamo.reset()
    runtime.stats.reset()
    return torch.compile(net, backend="xdna", options={"fallback": "eager"})


NAME = "qwen3 stack 2 layers -> 1000"


def test_stack_fused(gpu):
    """Three sequences of a 2-layer stack + biased head in one fused call: close to the oracle and to
    the fp32 model, padding rows zero, the first call checked; a causal mask runs the plain graph."""
    torch.manual_seed(4)
    net = Stack(layers=2, out=1000, bias=True).eval().to(gpu)
    L, lens = 100, [100, 70, 37]
    x = torch.randn(3, L, 1024, device=gpu)
    mask = prefix_mask(lens, L, gpu)
    m = _compiled(net)
    with torch.no_grad():
        y, ref = m(x, mask), net(x, mask)
    s = _stats()
    assert s["stacks"] == {f"{NAME} on gpu": 1} and not s["fallbacks"], s
    assert len(s["checks"]) == 1 and s["checks"][0][1] < 0.05, s["checks"]
    layers, norm, inv_freq = Q.model_weights(net.llm)
    for b, n in enumerate(lens):
        want = Q.stack_forward(x[b, :n], layers, norm, net.head.weight, net.head.bias, inv_freq)
        assert rel_err(y[b, :n].cpu(), want) < 2e-2, (b, n)
        assert rel_err(y[b, :n], ref[b, :n]) < 0.08
    assert not y[1, 70:].any() and not y[2, 37:].any(), "padding rows are not zero"
    causal = torch.tril(torch.ones(L, L, dtype=torch.bool, device=gpu)).expand(3, 1, L, L).contiguous()
    with torch.no_grad():
        y2, ref2 = m(x, causal), net(x, causal)
    assert _stats()["stacks"] == {f"{NAME} on gpu": 1, f"{NAME} on cpu": 1}
    assert rel_err(y2, ref2) < 0.05


def test_stack_silent_wrong(gpu, monkeypatch):
    """A stack whose GPU output is wrong fails its first-call check and runs the plain graph from then
    on (the reference's case_stack_silent_wrong)."""
    from torch_xdna import kernels

    real = kernels.mm_bf16

    def corrupt(a, w, bias, out_dtype):
        y = real(a, w, bias, out_dtype)
        return y * 1.5 if w.shape[0] == 1000 else y       # the head

    monkeypatch.setattr(kernels, "mm_bf16", corrupt)
    torch.manual_seed(6)
    net = Stack(layers=2, out=1000).eval().to(gpu)
    x, mask = torch.randn(2, 64, 1024, device=gpu), prefix_mask([64, 50], 64, gpu)
    m = _compiled(net)
    with torch.no_grad():
        y, ref = m(x, mask), net(x, mask)
        m(x, mask)
    s = _stats()
    assert len(s["fallbacks"]) == 1 and "disagrees with the model" in s["fallbacks"][0][1], s["fallbacks"]
    assert s["stacks"] == {f"{NAME} on cpu": 2}, s["stacks"]
    assert max(rel_err(y[0], ref[0]), rel_err(y[1, :50], ref[1, :50])) < 0.05


def test_stack_graph_replays(gpu, monkeypatch):
    """The HIP graph of a call shape (captured on its second call) replays with new inputs: every
    replay equals the eager run of the same inputs bit for bit, with other GPU work and syncs between
    the replays."""
    from torch_xdna import Config, stack

    torch.manual_seed(7)
    net = Stack(layers=2, out=300).eval().to(gpu)
    weights = {}
    for i, Lr in enumerate(net.llm.layers):
        at, mlp = Lr.self_attn, Lr.mlp
        for key, t in dict(q=at.q_proj.weight, k=at.k_proj.weight, v=at.v_proj.weight, o=at.o_proj.weight,
                           gate=mlp.gate_proj.weight, up=mlp.up_proj.weight, down=mlp.down_proj.weight,
                           input_norm=Lr.input_layernorm.weight, post_norm=Lr.post_attention_layernorm.weight,
                           q_norm=at.q_norm.weight, k_norm=at.k_norm.weight).items():
            weights[(i, key)] = t
    weights.update(norm=net.llm.norm.weight, head=net.head.weight, inv_freq=net.llm.rotary_emb.inv_freq)
    sid = stack.register(stack.Plan([], None, None, 1, None, weights, None, 2, 300, stack.MAX_TOKENS))
    cfg = Config(policy="gpu")
    lens, L = [40, 23], 40
    mask = prefix_mask(lens, L, gpu)
    xs = [torch.randn(2, L, 1024, device=gpu) for _ in range(4)]
    with torch.no_grad():
        monkeypatch.setattr(stack, "USE_GRAPHS", False)
        want = [stack.run(cfg, sid, x, mask) for x in xs]
        stack._stacks[sid].shapes.clear()
        monkeypatch.setattr(stack, "USE_GRAPHS", True)
        for rep in range(3):
            for x, w in zip(xs, want):
                got = stack.run(cfg, sid, x, mask)
                torch.cuda.synchronize()
                assert torch.equal(got, w), f"replay {rep} differs from the eager run"
                _ = (torch.randn(256, 256, device=gpu) @ torch.randn(256, 256, device=gpu)).sum().item()
    assert stack._stacks[sid].shapes[(tuple(lens), L, torch.float32, xs[0].device)].graph is not None
