"""Fused block kernels (fdl_rms_norm, fdl_silu_mul) against the unfused PyTorch code they
replace (modeling_llada.py:389-403 RMSLayerNorm; flash_cache_triton.py:618-633).

Both sides round to bf16 at the same points; the sum of squares is accumulated in a
different order, so an element may differ by one bf16 ulp. Bar: at least 99% of the
elements bit-identical and every element within one bf16 ulp (relative 2^-7)."""
import pytest
import torch

from fdl import ops
from fdl.model import RMSLayerNorm

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(got: torch.Tensor, ref: torch.Tensor, what: str):
    g, r = got.float(), ref.float()
    same = (got.view(torch.int16) == ref.view(torch.int16)).float().mean().item()
    assert same >= 0.99, f"{what}: only {same:.4f} of the elements bit-identical"
    bound = r.abs() * 2.0 ** -7 + 1e-30
    assert bool(((g - r).abs() <= bound).all()), f"{what}: difference above one bf16 ulp"


@pytest.mark.parametrize("rows,d", [(1, 4096), (37, 4096), (512, 4096), (300, 512), (64, 8192)])
def test_rms_norm_matches_module(rows, d):
    gen = torch.Generator().manual_seed(rows * 7 + d)
    x = (torch.randn(rows, d, generator=gen) * 3.0).to(torch.bfloat16).to(DEV)
    norm = RMSLayerNorm(d, 1e-5, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        norm.weight.copy_((1.0 + 0.1 * torch.randn(d, generator=gen)).to(torch.bfloat16))
        ref = norm(x)
    got = ops.rms_norm(x, norm.weight.detach(), 1e-5)
    torch.cuda.synchronize()
    _check(got, ref, f"rms_norm {rows}x{d}")


@pytest.mark.parametrize("rows", [5, 512])
def test_add_rms_norm_matches_residual_then_module(rows):
    d = 4096
    gen = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, d, generator=gen).to(torch.bfloat16).to(DEV)
    att = (0.5 * torch.randn(rows, d, generator=gen)).to(torch.bfloat16).to(DEV)
    norm = RMSLayerNorm(d, 1e-5, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        norm.weight.copy_((1.0 + 0.1 * torch.randn(d, generator=gen)).to(torch.bfloat16))
        s_ref = x + att
        ref = norm(s_ref)
    s, got = ops.rms_norm(x, norm.weight.detach(), 1e-5, residual=att)
    torch.cuda.synchronize()
    assert torch.equal(s, s_ref), "residual sum must be bit-exact"
    _check(got, ref, "add+rms_norm")


@pytest.mark.parametrize("n", [8, 4096 * 3, 512 * 12288])
def test_silu_mul_matches_torch(n):
    gen = torch.Generator().manual_seed(n % 1000)
    g = (2.0 * torch.randn(n, generator=gen)).to(torch.bfloat16).to(DEV)
    u = torch.randn(n, generator=gen).to(torch.bfloat16).to(DEV)
    ref = torch.nn.functional.silu(g) * u
    got = ops.silu_mul(g, u)
    torch.cuda.synchronize()
    _check(got, ref, f"silu_mul n={n}")


@pytest.mark.parametrize("rows,width", [(1, 8), (37, 4096), (512, 12288)])
def test_silu_mul_rows_on_gate_up_halves(rows, width):
    """fdl_silu_mul_rows on the two halves of one [rows, 2 * width] product (the fused
    ff_proj / up_proj GEMM) against silu(gate) * up on contiguous copies."""
    gen = torch.Generator().manual_seed(rows + width)
    gu = (2.0 * torch.randn(rows, 2 * width, generator=gen)).to(torch.bfloat16).to(DEV)
    gate, up = gu[:, :width], gu[:, width:]
    ref = torch.nn.functional.silu(gate.contiguous()) * up.contiguous()
    got = ops.silu_mul(gate, up)
    torch.cuda.synchronize()
    assert got.is_contiguous() and got.shape == (rows, width)
    _check(got, ref, f"silu_mul_rows {rows}x{width}")


def test_block_mlp_tail_fused_gate_up_matches_two_gemms():
    """The block epilogue with adjacent ff_proj / up_proj weights (one GEMM) against the
    same block with the weights in separate buffers (two GEMMs)."""
    import flash_cache_hip as fch
    from fdl.model import LLaDAConfig, LLaDALlamaBlock, random_init_
    cfg = LLaDAConfig.llada_8b()
    cfg.d_model, cfg.n_heads, cfg.mlp_hidden_size = 512, 4, 1536
    blk = LLaDALlamaBlock(cfg, 0, fch.flash_fused_elastic_cache, device=DEV, dtype=torch.bfloat16)
    gen = torch.Generator(device=DEV).manual_seed(0)
    with torch.no_grad():
        for p in blk.parameters():
            p.normal_(0.0, 0.05, generator=gen)
    assert fch._adjacent_gate_up(blk) is not None
    x = torch.randn(40, 512, generator=gen, device=DEV).to(torch.bfloat16)
    att = torch.randn(40, 512, generator=gen, device=DEV).to(torch.bfloat16)
    fused = fch.block_mlp_tail(blk, x, att)
    blk.up_proj.weight = torch.nn.Parameter(blk.up_proj.weight.detach().clone())
    assert fch._adjacent_gate_up(blk) is None
    split = fch.block_mlp_tail(blk, x, att)
    torch.cuda.synchronize()
    # the GEMM library may order the reduction differently for the wider product
    torch.testing.assert_close(fused.float(), split.float(), atol=2e-2, rtol=1e-2)


@pytest.mark.parametrize("rows,width,chunks", [(5, 64, 2), (512, 12288, 4)])
def test_silu_mul_rows_chunked_output(rows, width, chunks):
    """out_chunks = S writes the same values as S column chunks [S, rows, width / S]."""
    gen = torch.Generator().manual_seed(rows)
    gu = (2.0 * torch.randn(rows, 2 * width, generator=gen)).to(torch.bfloat16).to(DEV)
    gate, up = gu[:, :width], gu[:, width:]
    plain = ops.silu_mul(gate, up)
    chunked = ops.silu_mul(gate, up, out_chunks=chunks)
    torch.cuda.synchronize()
    assert chunked.shape == (chunks, rows, width // chunks)
    assert torch.equal(chunked, plain.view(rows, chunks, width // chunks).transpose(0, 1))


@pytest.mark.parametrize("S,rows,cols", [(1, 3, 8), (4, 512, 4096), (3, 17, 72)])
def test_split_reduce_residual_bit_exact(S, rows, cols):
    """residual = bf16(residual + ((p0 + p1) + p2 ...)) in place, the same float32 order."""
    gen = torch.Generator().manual_seed(S * rows + cols)
    part = torch.randn(S, rows, cols, generator=gen).to(DEV)
    res = torch.randn(rows, cols, generator=gen).to(torch.bfloat16).to(DEV)
    acc = part[0].clone()
    for s in range(1, S):
        acc = acc + part[s]
    ref = (res.float() + acc).to(torch.bfloat16)
    out = ops.split_reduce_residual(part, res)
    torch.cuda.synchronize()
    assert out.data_ptr() == res.data_ptr() and torch.equal(out, ref)


def test_block_mlp_tail_split_k_ff_out_matches_single_product():
    """The epilogue with ff_out stored transposed (split-K: chunked SiLU output, batched
    float32-output product, partials + residual in one pass) against the same weights in
    the plain layout (one product accumulating into the residual), and against float32."""
    import flash_cache_hip as fch
    from fdl.model import LLaDAConfig, LLaDALlamaBlock
    cfg = LLaDAConfig.llada_8b()
    cfg.d_model, cfg.n_heads, cfg.mlp_hidden_size = 512, 4, 1536
    blk = LLaDALlamaBlock(cfg, 0, fch.flash_fused_elastic_cache, device=DEV, dtype=torch.bfloat16)
    gen = torch.Generator(device=DEV).manual_seed(1)
    with torch.no_grad():
        for p in blk.parameters():
            p.normal_(0.0, 0.05, generator=gen)
    x = torch.randn(96, 512, generator=gen, device=DEV).to(torch.bfloat16)
    att = torch.randn(96, 512, generator=gen, device=DEV).to(torch.bfloat16)
    assert fch._split_k_ff_out(blk, 96) is not None
    split = fch.block_mlp_tail(blk, x, att)
    blk.ff_out.weight = torch.nn.Parameter(blk.ff_out.weight.detach().contiguous())
    assert fch._split_k_ff_out(blk, 96) is None
    single = fch.block_mlp_tail(blk, x, att)
    # float32 reference of the same epilogue from the bf16 intermediates
    og = x + (att.float() @ blk.attn_out.weight.float().t()).to(torch.bfloat16)
    xn = blk.ff_norm(og)
    g = torch.nn.functional.silu(xn.float() @ blk.ff_proj.weight.float().t()).to(torch.bfloat16)
    u = (xn.float() @ blk.up_proj.weight.float().t()).to(torch.bfloat16)
    hidden = (g.float() * u.float()).to(torch.bfloat16)
    ref = og.float() + hidden.float() @ blk.ff_out.weight.float().t()
    torch.cuda.synchronize()
    torch.testing.assert_close(split.squeeze(0).float(), single.squeeze(0).float(), atol=2e-2, rtol=1e-2)
    torch.testing.assert_close(split.squeeze(0).float(), ref, atol=5e-2, rtol=2e-2)


@pytest.mark.parametrize("chunks", [1, 4])
@pytest.mark.parametrize("rows,k,width", [
    # weight-streaming tiles of 24 (width up to 6144) and of 48 pairs
    (1, 256, 96), (64, 4096, 12288), (65, 384, 12288), (17, 640, 192), (100, 256, 6144), (33, 256, 6240),
    (128, 256, 192), (129, 256, 96), (256, 512, 12288),                 # 128-row tiles
    (257, 256, 12288), (300, 384, 12384), (600, 512, 12288),            # 256-row tiles
])
def test_gate_up_silu_matches_unfused(rows, k, width, chunks):
    """Both products in float32 rounded to bf16, then silu and the product as torch rounds them.
    A float32 sum of k bf16 products may round to the reference's bf16 neighbour, 2^-8 of the
    value at most, in g and in u. silu(g) = g sigmoid(g) changes by (1 + |g|) times g's relative
    change at most (its logarithmic derivative is 1 + g sigmoid(-g)), and two more roundings add
    2^-9 each on both sides: 2^-8 (1 + |g|) + 2^-8 + 2^-7 of the value, and where g or u
    crosses zero the sums' own error (1e-5 of unit-scale sums) through the other factor, 1e-3."""
    gen = torch.Generator().manual_seed(rows + k)
    x = torch.randn(rows, k, generator=gen).to(torch.bfloat16).to(DEV)
    wg, wu = ((torch.randn(width, k, generator=gen) * 0.05).to(torch.bfloat16).to(DEV)
              for _ in range(2))
    g = (x.float() @ wg.float().t()).to(torch.bfloat16)
    u = (x.float() @ wu.float().t()).to(torch.bfloat16)
    ref = torch.nn.functional.silu(g) * u
    got = ops.gate_up_silu(x, wg, wu, out_chunks=chunks)
    if chunks > 1:
        assert got.shape == (chunks, rows, width // chunks)
        got = got.transpose(0, 1).reshape(rows, width)
    tol = ref.float().abs() * (2.0**-8 * (2 + g.float().abs()) + 2.0**-7) + 1e-3
    assert bool(((got.float() - ref.float()).abs() <= tol).all())
    assert (got != ref).float().mean() < 0.02


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("rows,k,n_out", [(1, 64, 128), (64, 512, 256), (65, 192, 128), (128, 4096, 384),
                                          (129, 576, 256), (40, 12288, 4096), (200, 1024, 4096)])
def test_linear_partials_and_the_passes_that_add_them(rows, k, n_out, transposed):
    """Partial sums against float64 (fp32 sums of k terms: 2^-24 sqrt(k) of the terms' 2-norm,
    with a factor 8), and the norm over them bit for bit the norm over their bf16 sum."""
    gen = torch.Generator().manual_seed(rows + k)
    x = torch.randn(rows, k, generator=gen).to(torch.bfloat16).to(DEV)
    w = (torch.randn(n_out, k, generator=gen) * 0.05).to(torch.bfloat16).to(DEV)
    part = ops.linear_partials(x, w.t().contiguous() if transposed else w, transposed=transposed)
    assert part.dtype == torch.float32 and tuple(part.shape[1:]) == (rows, n_out)
    ref = x.double().cpu() @ w.double().cpu().t()
    scale = (x.double().cpu() ** 2) @ (w.double().cpu() ** 2).t()
    err = (part.double().cpu().sum(0) - ref).abs()
    assert bool((err <= 8 * 2.0**-24 * k**0.5 * scale.sqrt() + 1e-12).all())
    h = torch.randn(rows, n_out, generator=gen).to(torch.bfloat16).to(DEV)
    nw = torch.randn(n_out, generator=gen).to(torch.bfloat16).to(DEV)
    total = part[0].clone()
    for p in part[1:]:
        total += p
    ref_s, ref_y = ops.rms_norm(h, nw, 1e-5, residual=total.to(torch.bfloat16))
    got_s, got_y = ops.rms_norm_partials(h, nw, 1e-5, part)
    assert torch.equal(got_s, ref_s) and torch.equal(got_y, ref_y)


def test_attn_out_with_hooks_is_called_as_a_module():
    """A module with a hook, a bias or another class is called; a plain one runs in parts."""
    import flash_cache_hip as fch
    m = torch.nn.Linear(256, 256, bias=False, device=DEV, dtype=torch.bfloat16)
    x = torch.randn(8, 256, device=DEV).to(torch.bfloat16)
    assert fch._attn_out_in_parts(m, x, x)
    hook = m.register_forward_hook(lambda *a: None)
    assert not fch._attn_out_in_parts(m, x, x)
    hook.remove()
    assert not fch._attn_out_in_parts(torch.nn.Linear(256, 256, device=DEV, dtype=torch.bfloat16), x, x)
    assert not fch._attn_out_in_parts(m, x, x.t().contiguous().t())
    assert not fch._attn_out_in_parts(m, x[:, :128], x)
    many = torch.randn(200, 256, device=DEV).to(torch.bfloat16)
    assert not fch._attn_out_in_parts(m, many, many)  # a small weight's rows
    assert not fch._attn_out_in_parts(torch.nn.Identity(), many, many)


@pytest.mark.parametrize("rows", [1, 64, 65, 128])
@torch.no_grad()
def test_block_mlp_tail_with_every_product_of_few_rows(rows):
    """The epilogue of few rows at a width whose ff_out (2^25 elements) runs in parts, beside
    attn_out in parts and the fused gate and up product, against float32 products of the same
    bf16 intermediates. The output is a bf16 residual stream of size ~1 plus an MLP term of about
    that size: the roundings of g, u and their product (2^-9 of each of 18432 terms, in random
    directions) stay far below the result's own, 2^-9 of values up to 8, and a changed rounding of
    the residual, 2^-8 of it: 2^-7 of the value, bounded here by 2e-2."""
    import flash_cache_hip as fch
    from fdl.model import LLaDAConfig, LLaDALlamaBlock
    cfg = LLaDAConfig(d_model=2048, n_heads=16, mlp_hidden_size=18432)
    blk = LLaDALlamaBlock(cfg, 0, fch.flash_fused_elastic_cache, device=DEV, dtype=torch.bfloat16)
    gen = torch.Generator(device=DEV).manual_seed(rows)
    for p in blk.parameters():
        p.normal_(0.0, 0.02, generator=gen) if p.dim() == 2 else p.normal_(1.0, 0.1, generator=gen)
    x, att = (torch.randn(rows, 2048, generator=gen, device=DEV).to(torch.bfloat16) for _ in range(2))
    assert fch._attn_out_in_parts(blk.attn_out, x, att)
    assert fch._ff_out_in_parts(blk.ff_out.weight, rows) and fch._split_k_ff_out(blk, rows) is not None
    assert fch._fused_gate_up(x, fch._adjacent_gate_up(blk))
    x0 = x.clone()
    got = fch.block_mlp_tail(blk, x, att)
    assert torch.equal(x, x0) and got.shape == (1, rows, 2048)
    og = x + (att.float() @ blk.attn_out.weight.float().t()).to(torch.bfloat16)
    xn = blk.ff_norm(og)
    g = torch.nn.functional.silu((xn.float() @ blk.ff_proj.weight.float().t()).to(torch.bfloat16))
    u = (xn.float() @ blk.up_proj.weight.float().t()).to(torch.bfloat16)
    ref = og.float() + (g * u).float() @ blk.ff_out.weight.float().t()
    torch.testing.assert_close(got[0].float(), ref, atol=5e-2, rtol=2e-2)


@pytest.mark.parametrize("rows", [1, 37])
def test_final_norm_matches_module(rows):
    """The model's final norm in one kernel against the module (the bounds of the norm kernel's
    own test), and the module itself under autograd."""
    from fdl.model import _final_norm
    norm = RMSLayerNorm(512, 1e-5, DEV, torch.bfloat16)
    x = torch.randn(1, rows, 512, device=DEV).to(torch.bfloat16)
    with torch.no_grad():
        norm.weight.normal_()
        got = _final_norm(norm, x)
        assert got.shape == x.shape
        _check(got, norm(x), f"final norm {rows}")
    assert _final_norm(norm, x).requires_grad


def _elsewhere(case, m, x):
    """A forward of `m` that must not be bypassed: sets it up, returns (calls so far, undo)."""
    calls = []
    if case == "forward":  # as an offload or adapter wrapper replaces it
        own = m.forward
        m.forward = lambda *a: (calls.append(1), own(*a))[1]
        return calls, lambda: m.__dict__.pop("forward")
    if case == "global hook":
        h = torch.nn.modules.module.register_module_forward_hook(
            lambda mod, a, out: calls.append(1) if mod is m else None)
        return calls, h.remove
    h = m.register_forward_pre_hook(lambda mod, a: calls.append(1))
    return calls, h.remove


@pytest.mark.parametrize("case", ["forward", "global hook", "hook"])
@torch.no_grad()
def test_modules_that_do_more_than_their_forward_are_called(case):
    """attn_out in a block's tail and the final norm run their modules where a call does more
    than the class's forward, and in kernels of their own again afterwards, with like results."""
    import flash_cache_hip as fch
    from fdl.model import LLaDAConfig, LLaDALlamaBlock, _final_norm
    cfg = LLaDAConfig(d_model=512, n_heads=4, mlp_hidden_size=1536)
    blk = LLaDALlamaBlock(cfg, 0, fch.flash_fused_elastic_cache, device=DEV, dtype=torch.bfloat16)
    for p in blk.parameters():
        p.normal_(0.0, 0.05)
    norm = RMSLayerNorm(512, 1e-5, DEV, torch.bfloat16)
    x, att = (torch.randn(8, 512, device=DEV).to(torch.bfloat16) for _ in range(2))
    want = fch.block_mlp_tail(blk, x, att), _final_norm(norm, x)
    for m, run, ref in ((blk.attn_out, lambda: fch.block_mlp_tail(blk, x, att), want[0]),
                        (norm, lambda: _final_norm(norm, x), want[1])):
        calls, undo = _elsewhere(case, m, x)
        got = run()
        undo()
        assert len(calls) == 1
        torch.testing.assert_close(got.float(), ref.float(), atol=2e-2, rtol=1e-2)
        run()
        assert len(calls) == 1


def test_final_norm_keeps_forward_mode_derivatives_and_autocast_products():
    """A tangent passes through the final norm as through its module; attn_out under autocast is
    the module's product in autocast's type."""
    import torch.autograd.forward_ad as fwd
    import flash_cache_hip as fch
    from fdl.model import _final_norm
    norm = RMSLayerNorm(64, 1e-5, DEV, torch.bfloat16).requires_grad_(False)
    x, t = (torch.randn(5, 64, device=DEV).to(torch.bfloat16) for _ in range(2))
    with fwd.dual_level():
        got = fwd.unpack_dual(_final_norm(norm, fwd.make_dual(x, t))).tangent
        ref = fwd.unpack_dual(norm(fwd.make_dual(x, t))).tangent
        assert got is not None and torch.equal(got, ref)
    got = torch.func.vmap(lambda r: _final_norm(norm, r))(x)
    torch.testing.assert_close(got.float(), norm(x).float(), atol=2e-2, rtol=1e-2)
    m = torch.nn.Linear(256, 256, bias=False, device=DEV, dtype=torch.bfloat16)
    a = torch.randn(8, 256, device=DEV).to(torch.bfloat16)
    assert fch._attn_out_in_parts(m, a, a)
    with torch.autocast("cuda", torch.float16):
        assert not fch._attn_out_in_parts(m, a, a)
