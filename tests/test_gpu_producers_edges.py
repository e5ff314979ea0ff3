"""The producers' kernels at the edges of their tiles, against the float64 oracle: the convolution's blocks of 8 and 16
time steps and tiles of 64, channel counts that leave lanes of a wave past the channels, parameters in every type (read
and written in it by the kernels), and the gates' backward with heads that do not divide a workgroup's 256 lanes, more
heads than that, and one or several rows a lane.  Bounds: a result rounded once to a type of p significant bits is off
by at most 2^-p of itself, and float32 sums and exponentials before it by a few 2^-24 of their terms; the bar is 2^-p
plus 2^-20 of the 2-norm (eight such roundings of terms that cancel by half)."""
import pytest
import torch

from macai.gated_delta import _native as N
from macai.layer import conv_qkv, gates
from oracle import producers as P
from oracle.gdr import rel

pytestmark = pytest.mark.gpu
F64 = torch.float64
BITS = {torch.float32: 24, torch.bfloat16: 8, torch.float16: 11}


def _draw(shape, dtype, gen, scale=1.0):
    return (torch.randn(shape, generator=gen, dtype=F64) * scale).to(dtype)


def _compare(fused, ref, xs, gen):
    leaves = [x.cuda().requires_grad_(True) for x in xs]
    exact = [x.to(F64).requires_grad_(True) for x in xs]
    outs, refs = fused(*leaves), ref(*exact)
    ups = [_draw(o.shape, o.dtype, gen) for o in outs]
    got = list(outs) + list(torch.autograd.grad(outs, leaves, [u.cuda() for u in ups]))
    want = list(refs) + list(torch.autograd.grad(refs, exact, [u.to(F64) for u in ups]))
    for i, (x, y) in enumerate(zip(got, want)):
        e = rel(x.detach().cpu().double(), y.detach())
        assert e < 2.0 ** -BITS[x.dtype] + 2.0 ** -20, (i, x.dtype, e)


@pytest.mark.parametrize("dtype,wdtype", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32),
                                          (torch.float16, torch.bfloat16), (torch.float32, torch.float16)])
@pytest.mark.parametrize("T", [1, 3, 8, 16, 17, 61, 64, 65, 130])
def test_conv_blocks_and_channels(T, dtype, wdtype):
    print("case conv edges", T, dtype, wdtype, flush=True)
    gen = torch.Generator().manual_seed(T)
    for kd, dk, rep, dv, repeat in ((8, 8, 1, 8, False), (72, 24, 2, 16, True), (256, 64, 1, 64, False)):
        C = 2 * kd + kd // dk * rep * dv
        x, w = _draw((2, T, C), dtype, gen), _draw((C, 1, 4), wdtype, gen, 0.3)
        _compare(lambda a, b: conv_qkv(a, b, kd, dk, rep, dv, repeat, dtype),
                 lambda a, b: P.conv_qkv(a, b, kd, dk, rep, dv, repeat), [x, w], gen)


@pytest.mark.parametrize("dtype,v_dtype", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32),
                                           (torch.float16, torch.bfloat16), (torch.float32, torch.bfloat16),
                                           (torch.float32, torch.float32)])
@pytest.mark.parametrize("T", [1, 17, 61, 64, 130])
def test_conv_backward_on_both_forms(T, dtype, v_dtype):
    """The backward over many tiles (past 1,024 workgroups, every type's line) against the float64 oracle, and its first
    two rows by themselves, over few: the same dx bit for bit."""
    print("case conv forms", T, dtype, v_dtype, flush=True)
    gen = torch.Generator().manual_seed(T)
    kd, dk, rep, dv, repeat = 8, 8, 2, 8, True
    x, w = _draw((1030, T, 32), dtype, gen), _draw((32, 1, 4), torch.float32, gen, 0.3)
    fused = lambda a, b: conv_qkv(a, b, kd, dk, rep, dv, repeat, v_dtype)
    _compare(fused, lambda a, b: P.conv_qkv(a, b, kd, dk, rep, dv, repeat), [x, w], gen)
    ups = [_draw(o.shape, o.dtype, gen).cuda() for o in fused(x.cuda(), w.cuda())]
    dx = []
    for n in (len(x), 2):
        leaf, weight = x[:n].cuda().requires_grad_(True), w.cuda().requires_grad_(True)
        dx.append(torch.autograd.grad(fused(leaf, weight), [leaf, weight], [u[:n].contiguous() for u in ups])[0])
    assert torch.equal(dx[0][:2], dx[1])


@pytest.mark.parametrize("dtype,ptypes", [(torch.bfloat16, (torch.bfloat16, torch.bfloat16)),
                                          (torch.float32, (torch.float32, torch.float32)),
                                          (torch.bfloat16, (torch.float32, torch.float16))])
@pytest.mark.parametrize("rows,H", [(1, 1), (5, 3), (700, 48), (3, 256), (2, 257), (600, 300), (9000, 16)])
def test_gates_rows_and_heads(rows, H, dtype, ptypes):
    print("case gates edges", rows, H, dtype, ptypes, flush=True)
    gen = torch.Generator().manual_seed(rows + H)
    xs = [_draw((rows, H), dtype, gen), _draw((rows, H), dtype, gen, 3.0), _draw((H,), ptypes[0], gen),
          _draw((H,), ptypes[1], gen)]
    _compare(gates, P.gates, xs, gen)


@pytest.mark.parametrize("ptypes", [(torch.float32, torch.float32), (torch.bfloat16, torch.float16)])
@pytest.mark.parametrize("rows,H", [(512, 16), (576, 16), (577, 16), (577, 64), (2048, 1), (2049, 1), (1024, 2), (1025, 2),
                                    (2048, 3), (2049, 3), (2560, 65), (2561, 65), (4096, 257), (4097, 257), (2600, 8)])
def test_gates_parameter_gradients_on_both_forms(rows, H, ptypes):
    """Both sides of the line between the two forms of A_log's and dt_bias's gradients, and more heads than a
    workgroup's lanes past it: the float64 oracle's; and the entry point without scratch, which always takes the pass of
    a workgroup a head: the same db and da bit for bit, its float32 sums within two roundings of the others'."""
    print("case gates parameters", rows, H, ptypes, flush=True)
    gen = torch.Generator().manual_seed(rows + H)
    xs = [_draw((rows, H), torch.bfloat16, gen), _draw((rows, H), torch.bfloat16, gen, 3.0), _draw((H,), ptypes[0], gen),
          _draw((H,), ptypes[1], gen)]
    _compare(gates, P.gates, xs, gen)
    b, a, rate, bias = (x.cuda() for x in xs)
    rate, bias = rate.float(), bias.float()
    db_up, dg_up = (_draw((rows, H), torch.float32, gen).cuda() for _ in range(2))
    f32 = lambda: torch.empty(H, device="cuda")
    n, code, p, st = rows * H, N.BF16, N.ptr, N.stream_of(b)
    part = torch.empty(N.lib().macai_gdr_gates_partials(n, H), dtype=torch.float64, device="cuda")
    got = [[torch.empty_like(b), torch.empty_like(a), f32(), f32()] for _ in range(2)]
    ins = [p(x) for x in (b, a, rate, bias, db_up, dg_up)]
    N.call("macai_gdr_gates_bwd", *ins, *(p(x) for x in got[0]), n, H, code, st)
    d_b, d_a, d_rate, d_bias = (p(x) for x in got[1])
    N.call("macai_gdr_gates_bwd_typed", *ins, d_b, d_a, p(part), d_rate, N.F32, d_bias, N.F32, n, H, code, st)
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    for x, y in zip(got[0][2:], got[1][2:]):   # double sums in two orders: past their roundings to float32 2^-52 a term
        assert rel(x.double().cpu(), y.double().cpu()) < 2.0 ** -23


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_conv_infinities_and_nan(dtype):
    """Infinite and NaN inputs, and ones whose exponential overflows: y and dx are finite, infinite or NaN where plain
    PyTorch's are, of the same sign."""
    print("case conv infinities", dtype, flush=True)
    T, C = 41, 24
    gen = torch.Generator().manual_seed(5)
    x, w = _draw((1, T, C), dtype, gen), _draw((C, 1, 4), dtype, gen, 0.3).abs()
    for i, bad in enumerate((float("inf"), float("-inf"), float("nan"), 3e4, -3e4, 600.0, -600.0)):
        x[0, 6 * i, i::7] = bad
    leaf = x.cuda().requires_grad_(True)
    got = conv_qkv(leaf, w.cuda(), 8, 8, 1, 8, False, dtype)
    ups = [_draw(o.shape, dtype, gen) for o in got]
    dx, = torch.autograd.grad(got, leaf, [u.cuda() for u in ups])
    # in float32 on the CPU, sigmoid as 1 / (1 + exp(-u)); a window holds one such value at most
    x32, w32 = torch.nn.functional.pad(x.float(), (0, 0, 3, 0)), w.float().reshape(C, 4)
    u = sum(w32[:, j] * x32[:, j:j + T] for j in range(4))
    s = 1 / (1 + torch.exp(-u))
    y = u * s
    du = torch.nn.functional.pad(torch.cat(ups, 2).reshape(1, T, C).float() * (s * (1 + u * (1 - s))), (0, 0, 0, 3))
    want = [y.reshape(T, C), sum(w32[:, 3 - j] * du[:, j:j + T] for j in range(4)).reshape(T, C)]
    want = [t.to(dtype) for t in want]
    have = [torch.cat([o.detach().cpu().reshape(T, 8) for o in got], 1), dx.cpu().reshape(T, C)]
    for name, a, b in zip(("y", "dx"), have, want):
        for what, fa, fb in (("nan", a.isnan(), b.isnan()), ("inf", a.isinf(), b.isinf())):
            assert torch.equal(fa, fb), (name, what, (fa != fb).nonzero()[:8].tolist())
        inf = b.isinf()
        assert torch.equal(a[inf] > 0, b[inf] > 0), name


def test_conv_far_negative():
    """u between -88.7 and -87.3, where 1 / (1 + e^-u) is subnormal and u times it is not: y and dx keep their values
    (around -1e-36), in the type's precision and that of the exponential (|u| 2^-24 of its argument's rounding, four
    times over)."""
    print("case conv far negative", flush=True)
    us = torch.tensor([-87.0, -87.5, -88.0, -88.5])
    T, C = us.numel(), 24
    x = us.view(1, T, 1).expand(1, T, C).contiguous()
    w = torch.zeros(C, 1, 4)
    w[..., 3] = 1.0                                   # y[t] = silu(x[t])
    u64 = x.double().requires_grad_(True)
    want = u64 * torch.sigmoid(u64)
    dwant, = torch.autograd.grad(want, u64, torch.ones_like(want))
    for v_dtype in (torch.bfloat16, torch.float32):
        leaf = x.bfloat16().cuda().requires_grad_(True)
        out = conv_qkv(leaf, w.cuda(), 8, 8, 1, 8, False, v_dtype)
        dx, = torch.autograd.grad(out, leaf, [torch.ones_like(o) for o in out])
        parts = want.detach().reshape(T, 3, 8).unbind(1)
        for o, r in [*zip((o.reshape(T, 8) for o in out), parts), (dx.reshape(T, C), dwant.reshape(T, C))]:
            e = ((o.detach().cpu().double() - r) / r).abs().max().item()
            assert e < 2.0 ** -BITS[o.dtype] + 4 * 89 * 2.0 ** -24, (v_dtype, o.dtype, e)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_untyped_convolution_entry_points(dtype):
    """macai_gdr_conv_fwd and macai_gdr_conv_bwd take float32 taps: the bits of the typed ones for every output."""
    print("case conv untyped", dtype, flush=True)
    gen = torch.Generator().manual_seed(3)
    B, T, kd, dk, dv = 2, 70, 24, 8, 8
    C = 2 * kd + 3 * dv
    p, code = N.ptr, N.dtype_code(dtype)
    x, w = _draw((B, T, C), dtype, gen).cuda(), _draw((C, 4), torch.float32, gen, 0.3).cuda()
    ups = [_draw((B, T, 3, d), dtype, gen).cuda() for d in (dk, dk, dv)]
    sizes = (B, T, C, kd, dk, 1, dv, code, code, N.stream_of(x))
    nan = lambda *s, d=dtype: torch.full(s, float("nan"), dtype=d, device="cuda")
    got = []
    for typed in (False, True):
        outs = [nan(B, T, 3, d) for d in (dk, dk, dv)] + [nan(B, T, C), nan(C, 4, d=torch.float32)]
        part = nan(N.lib().macai_gdr_conv_partials(B, T, C), d=torch.float32)
        to, wt = ("_typed", [N.F32]) if typed else ("", [])
        N.call("macai_gdr_conv_fwd" + to, p(x), p(w), *wt, *([None] if typed else []), *map(p, outs[:3]), *sizes)
        N.call("macai_gdr_conv_bwd" + to, p(x), p(w), *map(p, ups), p(outs[3]), p(part), p(outs[4]), *wt, *sizes)
        got.append(outs)
    assert all(a.isfinite().all() and torch.equal(a, b) for a, b in zip(*got))
