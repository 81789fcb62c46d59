"""q, k and v as views (slices of the conv's output and others) give bit for
bit what contiguous copies of them give: slices of a wider row are read in
place, every other form goes through a copy."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

H, HV, D = 2, 4, 128


def _views(form, B, T, gen, dev):
    """(q, k, v) of shapes [B, T, H / HV, 128], bf16, not contiguous."""
    def rn(*shape):
        return torch.randn(*shape, generator=gen).bfloat16().to(dev)
    qk, hv = H * D, HV * D
    if form in ("row", "odd_start", "odd_pitch"):
        width = 2 * qk + hv + (4 if form == "odd_pitch" else 64)
        x = rn(B * T, width)
        at = {"row": 0, "odd_start": 1, "odd_pitch": 0}[form]
        parts = [x[:, at:at + qk], x[:, at + qk:at + 2 * qk], x[:, at + 2 * qk:at + 2 * qk + hv]]
        return [p.view(B, T, -1, D) for p in parts]
    if form == "two_pitches":
        return [rn(B * T, qk + 64)[:, :qk].view(B, T, H, D),
                rn(B * T, qk + 128)[:, :qk].view(B, T, H, D),
                rn(B * T, hv + 8)[:, 8:].view(B, T, HV, D)]
    if form == "head_major":
        return [rn(B, n, T, D).transpose(1, 2) for n in (H, H, HV)]
    if form == "every_other_token":
        return [rn(B, 2 * T, n, D)[:, ::2] for n in (H, H, HV)]
    if form == "one_head_expanded":
        return [rn(B, T, 1, D).expand(B, T, n, D) for n in (H, H, HV)]
    assert form == "padded_batch"  # B rows of T + 3 tokens
    return [rn(B, T + 3, n, D)[:, :T] for n in (H, H, HV)]


FORMS = ["row", "odd_start", "odd_pitch", "two_pitches", "head_major", "every_other_token",
         "one_head_expanded", "padded_batch"]


@pytest.mark.parametrize("B,T", [(1, 2), (1, 200), (2, 65)])
@pytest.mark.parametrize("form", FORMS)
def test_chunk(dev, form, B, T):
    from torch_npu_ops_amd import _xk_torch as xt
    gen = torch.Generator().manual_seed(T)
    q, k, v = _views(form, B, T, gen, dev)
    g = F.logsigmoid(torch.randn(B, T, HV, generator=gen)).to(dev)
    beta = torch.sigmoid(torch.randn(B, T, HV, generator=gen)).bfloat16().to(dev)
    h0 = torch.randn(B, HV, D, D, generator=gen).to(dev)
    kw = dict(initial_state=h0, output_final_state=True, use_qk_l2norm_in_kernel=True)
    a = xt.npu_chunk_gated_delta_rule(q, k, v, g, beta, **kw)
    b = xt.npu_chunk_gated_delta_rule(q.contiguous(), k.contiguous(), v.contiguous(), g, beta, **kw)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.parametrize("B,T", [(1, 1), (1, 7), (2, 5)])
@pytest.mark.parametrize("form", FORMS)
def test_recurrent(dev, form, B, T):
    from torch_npu_ops_amd import _xk_torch as xt
    gen = torch.Generator().manual_seed(T)
    q, k, v = _views(form, B, T, gen, dev)
    g = F.logsigmoid(torch.randn(B, T, HV, generator=gen)).to(dev)
    beta = torch.sigmoid(torch.randn(B, T, HV, generator=gen)).bfloat16().to(dev)
    pool = torch.randn(B, HV, D, D, generator=gen).to(dev)
    cu = torch.arange(0, (B + 1) * T, T, dtype=torch.int32, device=dev)
    idx = torch.arange(B, dtype=torch.int32, device=dev)
    out = []
    for t in ((q, k, v), (q.contiguous(), k.contiguous(), v.contiguous())):
        s = pool.clone()
        o, _ = xt.npu_fused_recurrent_gated_delta_rule(
            *t, g, beta, initial_state=s, cu_seqlens=cu, ssm_state_indices=idx)
        out.append((o, s))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


def test_pitch_checks():
    from torch_npu_ops_amd import _lib
    f = 1 << 20

    def call(sqk, sv):
        return _lib.lib().xk_gdn_chunk_fwd_strided(
            f, f, sqk, f, sv, _lib.XK_BF16, f, _lib.XK_F32, f, _lib.XK_BF16, f, None, None, f,
            _lib.XK_I32, 1, 64, 2, 4, 128, 128, 1.0, 1, None, 0, None)
    assert call(256, 512) == _lib.XK_ERR_WORKSPACE  # accepted up to the workspace
    for sqk, sv in ((248, 512), (256, 504), (260, 512), (256, 516)):
        assert call(sqk, sv) == _lib.XK_ERR_INVALID
