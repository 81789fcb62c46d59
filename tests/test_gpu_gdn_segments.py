"""Chunked gated delta rule on batches whose sequences are cut into segments
that run in parallel (few heads, long sequences), against the oracle and
against the same call in a workspace one byte too small for the segments,
which runs whole sequences in order.

The two paths differ only in how the state reaches a segment: its entry state
passes through the segments' transition matrices, to 24 bits, and what each
segment adds is formed from a zero state.  Each of the two paths is within
3.1e-5 (RMS + |value|) of the fp32 reference over the chunked tests (errors of
2^-17 of the state's size per product, over the few chunks for which the delta
rule remembers them), so they may differ by twice that: 6.2e-5 of the RMS and
of the value.
Outputs are sums of products of operands rounded to bf16 (the state's hi part,
v_new); a difference that small can flip the last bit of one operand, which
moves an output by up to 2^-8 of one term of its sum, a term being at most of
the outputs' own size: 2^-7 of their RMS beside one bf16 step (2^-7 of the
value) of the output itself are allowed."""
import pytest
import torch
import torch.nn.functional as F

from oracle import gdn as og
from state_tol import assert_state_close

pytestmark = pytest.mark.gpu

O_TOL = dict(rtol=1.6e-2, atol=1e-2)


def _inputs(lens, H, HV, seed=0, V=128):
    gen = torch.Generator().manual_seed(seed)
    T = sum(lens)
    q = torch.randn(1, T, H, 128, generator=gen).bfloat16()
    k = torch.randn(1, T, H, 128, generator=gen).bfloat16()
    v = torch.randn(1, T, HV, V, generator=gen).bfloat16()
    # Some heads forget within a chunk, some keep their state throughout.
    g = -F.softplus(torch.randn(1, T, HV, generator=gen)) * torch.logspace(-4, 0, HV)
    beta = torch.sigmoid(torch.randn(1, T, HV, generator=gen)).bfloat16()
    h0 = torch.randn(len(lens), HV, 128, V, generator=gen)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    return q, k, v, g, beta, h0, cu


def _run(dev, q, k, v, g, beta, h0, cu, segments=True, l2norm=True, bufs=None):
    from torch_npu_ops_amd import _lib, ops
    _, T, H, K = q.shape
    HV, V, N = v.shape[2], v.shape[3], cu.numel() - 1
    need = _lib.lib().xk_gdn_chunk_workspace_bytes(T, N, HV)
    t = [x.to(dev).contiguous() for x in (q, k, v, g.float(), beta, h0, cu)] if bufs is None else bufs
    o = torch.empty(1, T, HV, V, dtype=torch.bfloat16, device=dev)
    fin = torch.empty(N, HV, K, V, device=dev)
    ws = torch.full((need,), 0xA5, dtype=torch.uint8, device=dev)

    def call():
        st = _lib.lib().xk_gdn_chunk_fwd(
            t[0].data_ptr(), t[1].data_ptr(), t[2].data_ptr(), _lib.XK_BF16, t[3].data_ptr(),
            _lib.XK_F32, t[4].data_ptr(), _lib.XK_BF16, o.data_ptr(), t[5].data_ptr(),
            fin.data_ptr(), t[6].data_ptr(), _lib.XK_I32, N, T, H, HV, K, V, K ** -0.5,
            int(l2norm), ws.data_ptr(), need if segments else need - 1, ops._stream(o))
        _lib.check(st, "xk_gdn_chunk_fwd")
    call()
    torch.cuda.synchronize()
    return o, fin, call


def _same(a, b):
    (o1, f1, _), (o2, f2, _) = a, b
    o1, o2 = o1.float(), o2.float()
    rms = o2[o2.isfinite()].pow(2).mean().sqrt().item()
    torch.testing.assert_close(o1, o2, rtol=2 ** -7, atol=2 ** -7 * rms, equal_nan=True)
    rms = f2[f2.isfinite()].pow(2).mean().sqrt().item()
    torch.testing.assert_close(f1, f2, rtol=6.2e-5, atol=6.2e-5 * rms, equal_nan=True)


# One sequence at its shortest segmented length, odd lengths around chunk and
# segment edges, many segments; ragged batches with empty and one-token
# sequences; one and two 64-column tiles.
@pytest.mark.parametrize("lens,H,HV,V", [
    ([1024], 4, 8, 128), ([1025], 2, 4, 128), ([2111], 1, 2, 128), ([4095], 2, 2, 128),
    ([9000], 1, 2, 128), ([2500], 2, 6, 64), ([64 * 31 + 1, 0, 1, 700], 2, 4, 128),
    ([3000, 200, 1500], 1, 1, 128)])
def test_segments(dev, lens, H, HV, V):
    x = _inputs(lens, H, HV, seed=sum(lens), V=V)
    out = _run(dev, *x)
    _same(out, _run(dev, *x, segments=False))
    q, k, v, g, beta, h0, cu = x
    ro, rs = og.chunk_gdn(q, k, v, g, beta, None, h0, cu, use_qk_l2norm=True)
    torch.testing.assert_close(out[0].float().cpu(), ro, **O_TOL)
    assert_state_close(out[1].cpu(), rs)


def test_segments_in_a_graph(dev):
    x = _inputs([3001], 2, 4, seed=3)
    o, fin, call = _run(dev, *x)
    want = o.clone(), fin.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for _ in range(3):
        o.zero_()
        fin.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, want[0]) and torch.equal(fin, want[1])


def test_growing_transition_runs_in_order(dev):
    """Keys of norm > 1 along one direction: 1 - beta |k|^2 < -1, so the
    transition grows without bound and the head must run in order, bit for
    bit as without segments; the other head stays segmented."""
    q, k, v, g, beta, h0, cu = _inputs([2048], 2, 2, seed=5)
    k = F.normalize(k.float(), dim=-1)
    k[:, :, 0] = F.normalize(k[0, 0, 0], dim=-1) * 1.425  # |k|^2 = 2.03
    x = (q, k.bfloat16(), v, g, beta.masked_fill(torch.arange(2) == 0, 1.0), h0, cu)
    x[3][..., 0] = 0.0
    a, b = _run(dev, *x, l2norm=False), _run(dev, *x, segments=False, l2norm=False)
    assert torch.equal(a[0][:, :, 0], b[0][:, :, 0]) and torch.equal(a[1][:, 0], b[1][:, 0])
    _same((a[0][:, :, 1:], a[1][:, 1:], None), (b[0][:, :, 1:], b[1][:, 1:], None))


def test_nan_value_spreads_no_further(dev):
    """A NaN value reaches the same outputs as in order, and no transition."""
    q, k, v, g, beta, h0, cu = _inputs([3000], 1, 2, seed=7)
    v[0, 1500, 1, 17] = float("nan")
    a, b = _run(dev, q, k, v, g, beta, h0, cu), _run(dev, q, k, v, g, beta, h0, cu, segments=False)
    assert b[1][:, 1, :, 17].isnan().all() and not b[1][:, 1, :, 64:].isnan().any()
    _same(a, b)


def _least_workspace(T, N, HV):
    """Bytes of workspace that a call cannot do without: the chunk and
    sequence tables, the 8 KiB store sink and a record of 19,712 bytes per
    (chunk, v-head).  What a segmented call uses beyond them starts there."""
    def align(n):
        return (n + 255) // 256 * 256
    nt = T // 64 + N
    return align(4 * (N + 1)) + align(4 * N) + align(8 * nt) + 8192 + nt * HV * 19712


def _call(t, fin, h0, ws, ws_bytes, V=128, l2norm=True):
    """One xk_gdn_chunk_fwd on device tensors t = (q, k, v, g, beta, cu)."""
    from torch_npu_ops_amd import _lib, ops
    q, k, v, g, beta, cu = t
    T, H, HV, N = q.shape[1], q.shape[2], v.shape[2], cu.numel() - 1
    o = torch.empty_like(v)
    st = _lib.lib().xk_gdn_chunk_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), _lib.XK_BF16, g.data_ptr(), _lib.XK_F32,
        beta.data_ptr(), _lib.XK_BF16, o.data_ptr(), h0.data_ptr(), fin.data_ptr(), cu.data_ptr(),
        _lib.XK_I32, N, T, H, HV, 128, V, 128 ** -0.5, int(l2norm), ws.data_ptr(), ws_bytes,
        ops._stream(o))
    _lib.check(st, "xk_gdn_chunk_fwd")
    return o


@pytest.mark.parametrize("lens,H,HV", [([2111], 1, 2), ([64 * 63 + 1, 0, 1, 1900], 2, 4)])
def test_state_in_place_runs_in_order(dev, lens, H, HV):
    """final_state == initial_state: the first segment of a sequence reads the
    buffer that its last one writes, so the call must not be segmented (the
    workspace past the least is left alone) and is bit for bit the in-order
    call on separate buffers."""
    from torch_npu_ops_amd import _lib
    q, k, v, g, beta, h0, cu = _inputs(lens, H, HV, seed=11)
    t = [x.to(dev).contiguous() for x in (q, k, v, g, beta, cu)]
    T, N = sum(lens), len(lens)
    need, least = _lib.lib().xk_gdn_chunk_workspace_bytes(T, N, HV), _least_workspace(T, N, HV)
    assert need > least + 256  # room for segments
    start = h0.to(dev)
    fin = torch.empty_like(start)
    ws = torch.full((need,), 0xA5, dtype=torch.uint8, device=dev)
    want = _call(t, fin, start, ws, least)
    state = start.clone()
    got = _call(t, state, state, ws, need)
    assert torch.equal(got, want) and torch.equal(state, fin)
    assert (ws[least:] == 0xA5).all()


def _final64(q, k, v, g, beta, h0, lens):
    """Final states in 64 bits, token by token (keys l2-normalised)."""
    k, v, g, beta = k[0].double(), v[0].double(), g[0].double(), beta[0].double()
    k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    k = k.repeat_interleave(v.size(1) // k.size(1), 1)
    out, at = [], 0
    for n, s in zip(lens, h0.double()):
        s = s.clone()
        for t in range(at, at + n):
            s *= g[t].exp()[:, None, None]
            new = beta[t][:, None] * (v[t] - (s * k[t][..., None]).sum(-2))
            s += k[t][..., None] * new[:, None, :]
        out.append(s)
        at += n
    return torch.stack(out)


@pytest.mark.parametrize("beta_to,decay_to,mean", [
    (1.0, 1e-2, 0.0), (0.1, 1e-3, 2.0), (0.01, 1e-5, 0.0), (0.01, 1e-5, 2.0), (1e-3, 1e-6, 0.0)])
def test_slow_heads_lose_no_precision(dev, beta_to, decay_to, mean):
    """Heads that hardly change their state over a segment (small beta, decays
    near 1; keys in all directions or around a common one): the segmented
    final state is as near to 64 bits as the one in order, whose state is
    scaled in fp32 and rounded only in what is added.  A boundary adds a few
    fp32 roundings of the state, a chunk of the chain as many and the hi/lo
    products', and there are more chunks than boundaries: within a factor of
    two."""
    from torch_npu_ops_amd import _lib
    lens, HV = [4096], 2
    q, k, v, g, beta, h0, cu = _inputs(lens, 2, HV, seed=21)
    k = (k.float() + mean * k[:, :1].float()).bfloat16()
    gen = torch.Generator().manual_seed(22)
    g = -torch.rand(g.shape, generator=gen) * decay_to
    beta = (torch.rand(g.shape, generator=gen) * beta_to).bfloat16()
    t = [x.to(dev).contiguous() for x in (q, k, v, g, beta, cu)]
    h0d = h0.to(dev)
    need, least = _lib.lib().xk_gdn_chunk_workspace_bytes(4096, 1, HV), _least_workspace(4096, 1, HV)
    exact, err = _final64(q, k, v, g, beta, h0, lens), {}
    for name, size in (("order", least), ("segments", need)):
        fin = torch.empty_like(h0d)
        ws = torch.zeros(need, dtype=torch.uint8, device=dev)
        _call(t, fin, h0d, ws, size)
        assert bool(ws[least:least + 4].any()) == (name == "segments")  # chunks per segment
        err[name] = ((fin.cpu().double() - exact).norm() / exact.norm()).item()
    print(err)
    assert err["segments"] <= 2 * err["order"]


# A batch that is offered the segment passes takes them whatever its lengths
# (idle passes would slow it down), from the shortest chains that are offered
# them to many segments; a batch whose equal lengths would gain nothing is not.
@pytest.mark.parametrize("N,HV,T,offered", [
    (1, 8, 1024, True), (1, 24, 2048, True), (2, 16, 4096, True), (4, 8, 8192, True),
    (6, 4, 12288, True), (16, 1, 16384, True), (1, 24, 1024, False), (2, 16, 2048, False),
    (2, 24, 4096, False), (4, 16, 8192, False), (6, 8, 6144, False)])
@pytest.mark.parametrize("kind", ["equal", "ragged", "one_long"])
def test_offered_segments_are_taken(dev, N, HV, T, offered, kind):
    from torch_npu_ops_amd import _lib
    need, least = _lib.lib().xk_gdn_chunk_workspace_bytes(T, N, HV), _least_workspace(T, N, HV)
    if kind == "equal":
        lens = [T // N] * N
    elif kind == "ragged":
        lens = [max(1, 2 * T * (i + 1) // (N * (N + 1))) for i in range(N)]
    else:
        lens = [1] * N
    lens[-1] += T - sum(lens)
    q, k, v, g, beta, h0, cu = _inputs(lens, 1, HV, seed=T)
    t = [x.to(dev).contiguous() for x in (q, k, v, g, beta, cu)]
    h0 = h0.to(dev)
    ws = torch.full((need,), 0xA5, dtype=torch.uint8, device=dev)
    _call(t, torch.empty_like(h0), h0, ws, need)
    if not offered:
        assert (ws[least:] == 0xA5).all()
        return
    per = int(ws[least:least + 4].view(torch.int32))  # chunks per segment
    assert 0 < per < (max(lens) + 63) // 64


@pytest.mark.parametrize("HV,V,T", [(8, 64, 4096), (8, 192, 4096), (4, 256, 4096), (16, 64, 8192),
                                    (24, 64, 16384), (8, 320, 4096)])
def test_every_width_fits_the_advertised_workspace(dev, HV, V, T):
    """The size does not know V: with it, states of every width up to 256 take
    their segments (wider ones run in order, with the in-order bits), and one
    byte less runs in order."""
    from torch_npu_ops_amd import _lib
    q, k, v, g, beta, h0, cu = _inputs([T], 2, HV, seed=V, V=V)
    t = [x.to(dev).contiguous() for x in (q, k, v, g, beta, cu)]
    h0 = h0.to(dev)
    need, least = _lib.lib().xk_gdn_chunk_workspace_bytes(T, 1, HV), _least_workspace(T, 1, HV)
    out = {}
    for size in (need, need - 1, least):
        ws = torch.zeros(need, dtype=torch.uint8, device=dev)
        fin = torch.empty_like(h0)
        o = _call(t, fin, h0, ws, size, V=V)
        segmented = bool(ws[least:least + 4].any())
        assert segmented == (size == need and V <= 256)
        out[size] = (o, fin, None)
    assert torch.equal(out[need - 1][0], out[least][0])
    assert torch.equal(out[need - 1][1], out[least][1])
    _same(out[need], out[least])


def _segmented(dev, x, V=128):
    """The call with and without segments: (o, final) of each, after checking
    that each ran as meant."""
    from torch_npu_ops_amd import _lib
    q, k, v, g, beta, h0, cu = x
    t = [a.to(dev).contiguous() for a in (q, k, v, g, beta, cu)]
    h0 = h0.to(dev)
    T, HV, N = q.shape[1], v.shape[2], cu.numel() - 1
    need, least = _lib.lib().xk_gdn_chunk_workspace_bytes(T, N, HV), _least_workspace(T, N, HV)
    out = []
    for size in (need, least):
        ws = torch.zeros(need, dtype=torch.uint8, device=dev)
        fin = torch.empty_like(h0)
        o = _call(t, fin, h0, ws, size, V=V)
        assert bool(ws[least:least + 4].any()) == (size == need)
        out.append((o, fin, None))
    return out


# Segments (checked to be there) of one to four 64-column tiles; empty and
# one-token sequences beside segmented ones; odd lengths.
@pytest.mark.parametrize("lens,H,HV,V", [
    ([2500], 2, 6, 64), ([64 * 63 + 1, 0, 1, 1900], 2, 4, 128), ([3000, 200, 1500], 1, 1, 128),
    ([5000, 1], 1, 2, 192), ([4097], 2, 4, 192), ([3333], 1, 2, 256)])
def test_segments_and_order_agree(dev, lens, H, HV, V):
    x = _inputs(lens, H, HV, seed=sum(lens) + V, V=V)
    a, b = _segmented(dev, x, V)
    _same(a, b)
    q, k, v, g, beta, h0, cu = x
    ro, rs = og.chunk_gdn(q, k, v, g, beta, None, h0, cu, use_qk_l2norm=True)
    torch.testing.assert_close(a[0].float().cpu(), ro, **O_TOL)
    assert_state_close(a[1].cpu(), rs)


@pytest.mark.parametrize("opt", ["no_initial", "no_final", "bf16_g", "f32_beta", "i64_cu",
                                 "wide_rows", "raw_keys"])
def test_segments_with_other_arguments(dev, opt):
    from torch_npu_ops_amd import _lib, ops
    lens, H, HV = [2111, 1, 3000], 2, 4
    q, k, v, g, beta, h0, cu = _inputs(lens, H, HV, seed=31)
    if opt == "raw_keys":
        q, k = F.normalize(q.float(), dim=-1).bfloat16(), F.normalize(k.float(), dim=-1).bfloat16()
    T, N = q.shape[1], len(lens)
    g = g.bfloat16() if opt == "bf16_g" else g
    beta = beta.float() if opt == "f32_beta" else beta
    cu = cu.long() if opt == "i64_cu" else cu
    t = [a.to(dev).contiguous() for a in (q, k, v, g, beta, cu)]
    sqk, sv = H * 128, HV * 128
    if opt == "wide_rows":  # slices of one row, as the conv's output
        row = torch.cat([a.reshape(T, -1) for a in t[:3]] + [t[0].new_zeros(T, 72)], 1)
        t[0], t[1], t[2] = row, row[:, sqk:], row[:, 2 * sqk:]
        sqk = sv = row.size(1)
    h0d = None if opt == "no_initial" else h0.to(dev)
    need, least = _lib.lib().xk_gdn_chunk_workspace_bytes(T, N, HV), _least_workspace(T, N, HV)
    out = []
    for size in (need, least):
        ws = torch.zeros(need, dtype=torch.uint8, device=dev)
        o = torch.empty(1, T, HV, 128, dtype=torch.bfloat16, device=dev)
        fin = None if opt == "no_final" else torch.empty(N, HV, 128, 128, device=dev)
        st = _lib.lib().xk_gdn_chunk_fwd_strided(
            t[0].data_ptr(), t[1].data_ptr(), sqk, t[2].data_ptr(), sv, _lib.XK_BF16,
            t[3].data_ptr(), ops.xk_dtype(t[3]), t[4].data_ptr(), ops.xk_dtype(t[4]), o.data_ptr(),
            ops._ptr(h0d), ops._ptr(fin), t[5].data_ptr(), ops.xk_dtype(t[5]), N, T, H, HV, 128, 128,
            128 ** -0.5, int(opt != "raw_keys"), ws.data_ptr(), size, ops._stream(o))
        _lib.check(st, "xk_gdn_chunk_fwd_strided")
        assert bool(ws[least:least + 4].any()) == (size == need)
        out.append((o, torch.zeros(1, device=dev) if fin is None else fin, None))
    _same(*out)
    ro, rs = og.chunk_gdn(q, k, v, g.float(), beta.float(), None, None if h0d is None else h0, cu,
                          use_qk_l2norm=opt != "raw_keys")
    torch.testing.assert_close(out[0][0].float().cpu(), ro, **O_TOL)
    if opt != "no_final":
        assert_state_close(out[0][1].cpu(), rs)


def test_segments_through_the_cpp_api_on_views(dev):
    """Slices of a wider row, long enough to be segmented, give bit for bit
    what contiguous copies of them and the C call give."""
    from torch_npu_ops_amd import _xk_torch as xt
    q, k, v, g, beta, h0, cu = [x.to(dev) for x in _inputs([3000, 700], 2, 4, seed=41)]
    T = q.shape[1]
    row = torch.cat([a.reshape(T, -1) for a in (q, k, v)] + [q.new_zeros(T, 64)], 1)
    parts = [p.view(1, T, -1, 128) for p in row[:, :1024].split([256, 256, 512], -1)]
    out = [xt.npu_chunk_gated_delta_rule(*a, g, beta, initial_state=h0, output_final_state=True,
                                         cu_seqlens=cu, use_qk_l2norm_in_kernel=True)
           for a in (parts, (q, k, v))]
    seg, _ = _segmented(dev, [x.cpu() for x in (q, k, v, g, beta, h0, cu)])
    for o, fin in out:
        assert torch.equal(o, seg[0]) and torch.equal(fin, seg[1])


@pytest.mark.parametrize("T,HV", [(3000, 4), (26000, 8)])
def test_segments_without_a_workspace_argument(dev, T, HV):
    """The static buffer holds the segments of the first size (same bits as the
    full workspace) and only the records of the second (bits of the order)."""
    from torch_npu_ops_amd import _lib, ops
    x = _inputs([T], 2, HV, seed=51)
    want = _segmented(dev, x)
    need = _lib.lib().xk_gdn_chunk_workspace_bytes(T, 1, HV)
    q, k, v, g, beta, h0, cu = [a.to(dev).contiguous() for a in x]
    o, fin = torch.empty_like(v), torch.empty_like(h0)
    st = _lib.lib().xk_gdn_chunk_fwd_noalloc(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), _lib.XK_BF16, g.data_ptr(), _lib.XK_F32,
        beta.data_ptr(), _lib.XK_BF16, o.data_ptr(), h0.data_ptr(), fin.data_ptr(), cu.data_ptr(),
        _lib.XK_I32, 1, T, 2, HV, 128, 128, 128 ** -0.5, 1, ops._stream(o))
    _lib.check(st, "xk_gdn_chunk_fwd_noalloc")
    assert (need <= 64 << 20) == (T == 3000)
    o2, fin2, _ = want[0 if need <= 64 << 20 else 1]
    assert torch.equal(o, o2) and torch.equal(fin, fin2)
