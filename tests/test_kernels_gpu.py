"""Each HIP kernel alone against its plain PyTorch reference (tests/torch_ops.py), in float32 and
bfloat16, at sizes other than the engine's tiny models: widths and vocabularies that are no power
of two, head sizes 16 .. 256, groups of 1, 3, 7, page sizes 4 .. 64."""
import itertools
import math
import threading

import numpy as np
import pytest
import torch

from torch_ops import TorchOps, exponential_noise
from velox_amd.engine.runner import collection_held

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]


@pytest.fixture(scope="module")
def ops():
    from velox_amd.kernels import load_ops

    return load_ops("cuda")


@pytest.fixture(scope="module")
def ref():
    return TorchOps()


def tol(dtype):
    return dict(rtol=2e-5, atol=2e-6) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-3)


def rand(shape, dtype, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype).cuda()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hidden,vocab", [(96, 320), (3584, 1000), (50, 77)])
def test_embed(ops, ref, dtype, hidden, vocab):
    table = rand((vocab, hidden), dtype, 0)
    ids = torch.randint(0, vocab, (37,), generator=torch.Generator().manual_seed(1)).to(torch.int32).cuda()
    torch.testing.assert_close(ops.embed(ids, table), ref.embed(ids, table), rtol=0, atol=0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hidden", [64, 96, 3584, 1000])
def test_add_rmsnorm(ops, ref, dtype, hidden):
    tokens = 19
    residual = rand((tokens, hidden), torch.float32, 2)
    delta = rand((tokens, hidden), dtype, 3)
    weight = 1 + rand((hidden,), torch.float32, 4, 0.02)
    r_hip, r_ref = residual.clone(), residual.clone()
    got = ops.add_rmsnorm(r_hip, delta, weight, 1e-5, dtype)
    want = ref.add_rmsnorm(r_ref, delta, weight, 1e-5, dtype)
    torch.testing.assert_close(r_hip, r_ref, rtol=0, atol=0)
    torch.testing.assert_close(got.float(), want.float(), **tol(dtype))
    # no delta: the residual is untouched
    before = r_hip.clone()
    got = ops.add_rmsnorm(r_hip, None, weight, 1e-6, dtype)
    torch.testing.assert_close(r_hip, before, rtol=0, atol=0)
    torch.testing.assert_close(got.float(), ref.add_rmsnorm(r_ref, None, weight, 1e-6, dtype).float(), **tol(dtype))
    # chosen rows: nothing is written
    rows = torch.tensor([18, 0, 7, 7], dtype=torch.int32).cuda()
    got = ops.add_rmsnorm_rows(r_hip, delta, rows, weight, 1e-6, dtype)
    torch.testing.assert_close(r_hip, before, rtol=0, atol=0)
    torch.testing.assert_close(got.float(), ref.add_rmsnorm_rows(r_ref, delta, rows, weight, 1e-6, dtype).float(), **tol(dtype))


def test_rmsnorm_eps_is_inside_the_root(ops):
    # tiny inputs: rsqrt(ms + eps) and 1 / (sqrt(ms) + eps) differ by orders of magnitude
    hidden = 128
    x = torch.full((1, hidden), 1e-4, device="cuda")
    w = torch.ones(hidden, device="cuda")
    got = ops.add_rmsnorm(x.clone(), None, w, 1e-6, torch.float32)
    want = 1e-4 / math.sqrt(1e-8 + 1e-6)
    torch.testing.assert_close(got, torch.full_like(got, want), rtol=1e-5, atol=0)


@pytest.mark.parametrize("a_dtype,w_dtype,out_dtype", [
    (torch.float32, torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16, torch.bfloat16),
    (torch.bfloat16, torch.float32, torch.bfloat16), (torch.bfloat16, torch.bfloat16, torch.float32),
])
@pytest.mark.parametrize("m,n,k", [(1, 320, 96), (7, 263, 80), (65, 130, 150), (130, 64, 224), (3, 70, 37), (16, 1001, 3584), (9, 3584, 18944), (2, 13, 260)])
def test_gemm_fma(ops, ref, a_dtype, w_dtype, out_dtype, m, n, k):
    x = rand((m, k), a_dtype, 5)
    w = rand((n, k), w_dtype, 6, 0.05)
    bias = rand((n,), torch.float32, 7)
    for b in (None, bias):
        got = ops.gemm_fma(x, w, b, out_dtype)
        want = ref.linear(x, w, b, out_dtype)
        if k >= 1024 and out_dtype == torch.float32:
            # sums of thousands of terms round differently in every order of adding: the yardstick is the exact product
            # (float64), and the kernel has to be as close to it as the library's float32 product is, within a factor of two
            exact = x.double() @ w.double().T + (b.double() if b is not None else 0)
            library = (x.float() @ w.float().T + (b if b is not None else 0)).double()
            assert float((got.double() - exact).abs().max()) <= 2 * float((library - exact).abs().max()) + 1e-7
            continue
        torch.testing.assert_close(got.float(), want.float(), **tol(out_dtype))
    if m <= 16 and m > 1:
        # few rows take a kernel of their own: a row's sum depends on that row alone, to the bit, whatever else is in the batch
        alone = ops.gemm_fma(x[m - 1:].contiguous(), w, None, out_dtype)
        assert torch.equal(alone[0], ops.gemm_fma(x, w, None, out_dtype)[m - 1])


@pytest.mark.parametrize("m,n,k", [(1, 320, 96), (8, 152064 // 8, 512), (64, 1000, 3584), (300, 4608, 3584)])
def test_linear_bf16_library_path(ops, ref, m, n, k):
    x = rand((m, k), torch.bfloat16, 8)
    w = rand((n, k), torch.bfloat16, 9, 0.02)
    got = ops.linear(x, w, None, torch.bfloat16)
    want = ref.linear(x, w, None, torch.bfloat16)
    torch.testing.assert_close(got.float(), want.float(), rtol=2e-2, atol=2e-2)
    got32 = ops.linear(x, w, None, torch.float32)
    torch.testing.assert_close(got32, ref.linear(x, w, None, torch.float32), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("inter", [128, 224, 150, 18944])
def test_silu_mul(ops, ref, dtype, inter):
    gate_up = rand((11, 2 * inter), dtype, 10, 2.0)
    torch.testing.assert_close(ops.silu_mul(gate_up).float(), ref.silu_mul(gate_up).float(), **tol(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,d,half,page", [(4, 2, 16, 8, 4), (3, 1, 32, 16, 8), (6, 2, 48, 24, 16), (28, 4, 128, 64, 16), (2, 2, 64, 16, 32), (5, 5, 16, 0, 4)])
def test_rope_kv_write(ops, ref, dtype, nh, nkv, d, half, page):
    tokens, pages = 23, 12
    width = (nh + 2 * nkv) * d
    qkv = rand((tokens, width), dtype, 11)
    bias = rand((width,), torch.float32, 12, 0.1)
    positions = torch.randint(0, 500, (tokens,), generator=torch.Generator().manual_seed(13)).to(torch.int32).cuda()
    slots = (torch.randperm((pages - 1) * page, generator=torch.Generator().manual_seed(14))[:tokens] + page).to(torch.int32).cuda()
    if half:
        angles = torch.outer(torch.arange(512, dtype=torch.float32), 1.0 / (10000.0 ** (torch.arange(half, dtype=torch.float32) / half)))
        cos, sin = angles.cos().cuda(), angles.sin().cuda()
    else:
        cos = sin = None
    for use_bias in (bias, None):
        caches = []
        for impl in (ops, ref):
            k_cache = torch.zeros((pages, nkv, page, d), dtype=dtype, device="cuda")
            v_cache = torch.zeros((pages, nkv, d, page), dtype=dtype, device="cuda")
            buf = qkv.clone()
            impl.rope_kv_write(buf, nh, nkv, d, positions, cos, sin, slots, k_cache, v_cache, page, write_kv=True, bias=use_bias)
            caches.append((buf[:, : nh * d].float(), k_cache.float(), v_cache.float()))
        for got, want in zip(*caches):
            torch.testing.assert_close(got, want, **tol(dtype))
    # write_kv=False leaves the cache alone
    k_cache = torch.zeros((pages, nkv, page, d), dtype=dtype, device="cuda")
    v_cache = torch.zeros((pages, nkv, d, page), dtype=dtype, device="cuda")
    ops.rope_kv_write(qkv.clone(), nh, nkv, d, positions, cos, sin, slots, k_cache, v_cache, page, write_kv=False, bias=bias)
    assert not k_cache.any() and not v_cache.any()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,d,page", [(28, 4, 128, 16), (4, 2, 16, 8), (3, 1, 32, 32), (6, 2, 48, 4)])
def test_rope_kv_write_for_consecutive_tokens_of_prompts(ops, ref, dtype, nh, nkv, d, page):
    """Prompt portions: consecutive tokens in consecutive slots (runs of eight are written as whole vectors), starting
    anywhere in a page, pages in any order, a single decoded token between two portions."""
    half = d // 2
    width = (nh + 2 * nkv) * d
    pages = 40
    order = (torch.randperm(pages - 1, generator=torch.Generator().manual_seed(15)) + 1).tolist()
    slots, positions = [], []
    for start, count in ((5, 37), (0, 1), (16, 70), (3, 9)):  # (first position, tokens) of each sequence's portion
        table = [order.pop() for _ in range((start + count + page - 1) // page)]
        for p in range(start, start + count):
            slots.append(table[p // page] * page + p % page)
            positions.append(p)
    tokens = len(slots)
    qkv = rand((tokens, width), dtype, 16)
    bias = rand((width,), torch.float32, 17, 0.1)
    slots = torch.tensor(slots, dtype=torch.int32).cuda()
    positions = torch.tensor(positions, dtype=torch.int32).cuda()
    angles = torch.outer(torch.arange(512, dtype=torch.float32), 1.0 / (10000.0 ** (torch.arange(half, dtype=torch.float32) / half)))
    cos, sin = angles.cos().cuda(), angles.sin().cuda()
    results = []
    for impl in (ops, ref):
        k_cache = torch.full((pages, nkv, page, d), 3.0, dtype=dtype, device="cuda")
        v_cache = torch.full((pages, nkv, d, page), 3.0, dtype=dtype, device="cuda")
        buf = qkv.clone()
        impl.rope_kv_write(buf, nh, nkv, d, positions, cos, sin, slots, k_cache, v_cache, page, write_kv=True, bias=bias)
        results.append((buf[:, : nh * d].float(), k_cache.float(), v_cache.float()))
    for got, want in zip(*results):
        torch.testing.assert_close(got, want, **tol(dtype))


@pytest.mark.parametrize("m", [1, 5, 16])
@pytest.mark.parametrize("nh,nkv,d,k,page", [(4, 2, 64, 128, 4), (28, 4, 128, 3584, 16), (3, 1, 32, 192, 1), (2, 2, 96, 64, 8), (5, 5, 160, 320, 32)])
def test_qkv_projection_with_rotation_and_cache_write_in_one_kernel(ops, ref, m, nh, nkv, d, k, page):
    """The fused decode kernel against product -> bias -> rotation -> cache write done one after the other in float32,
    and against the unfused kernels; untouched cache entries stay untouched."""
    pages = 24
    width = (nh + 2 * nkv) * d
    half = d // 2
    x = rand((m, k), torch.bfloat16, 70)
    w = rand((width, k), torch.bfloat16, 71, 0.05)
    bias = rand((width,), torch.float32, 72, 0.3)
    positions = torch.randint(0, 500, (m,), generator=torch.Generator().manual_seed(73)).to(torch.int32).cuda()
    slots = (torch.randperm((pages - 1) * page, generator=torch.Generator().manual_seed(74))[:m] + page).to(torch.int32).cuda()
    angles = torch.outer(torch.arange(512, dtype=torch.float32), 1.0 / (10000.0 ** (torch.arange(half, dtype=torch.float32) / half)))
    cos, sin = angles.cos().cuda(), angles.sin().cuda()
    pw = ops.prepare_weight(w, rotary_heads=(nh, nkv, d))
    assert pw.copy("rotary") is not None
    for use_bias in (bias, None):
        # float32 reference: exact product of the bfloat16 operands, then everything in float32
        k32 = torch.full((pages, nkv, page, d), 7.0, dtype=torch.float32, device="cuda")
        v32 = torch.full((pages, nkv, d, page), 7.0, dtype=torch.float32, device="cuda")
        wide = ref.linear(x, w, None, torch.float32)
        ref.rope_kv_write(wide, nh, nkv, d, positions, cos, sin, slots, k32, v32, page, write_kv=True, bias=use_bias)
        results = {}
        for fused in (True, False):
            k_cache = torch.full((pages, nkv, page, d), 7.0, dtype=torch.bfloat16, device="cuda")
            v_cache = torch.full((pages, nkv, d, page), 7.0, dtype=torch.bfloat16, device="cuda")
            for waves in ((8, 16) if fused else (None,)):
                q = ops.qkv_rope_write(x, pw, use_bias, nh, nkv, d, positions, cos, sin, slots, k_cache, v_cache, page, waves=waves, fused=fused)
                results[(fused, waves)] = (q[:, : nh * d].float(), k_cache.float(), v_cache.float())
        scale = float(wide.abs().max())
        for key, (q, kc, vc) in results.items():
            fused = key[0]
            # the unfused route rounds the product to bfloat16 before the rotation: one more rounding
            bound = dict(rtol=1e-2, atol=(1e-2 if fused else 2e-2) * scale)
            torch.testing.assert_close(q, wide[:, : nh * d], msg=lambda t: f"{key} q: {t}", **bound)
            torch.testing.assert_close(kc, k32, msg=lambda t: f"{key} k: {t}", **bound)
            torch.testing.assert_close(vc, v32, msg=lambda t: f"{key} v: {t}", **bound)
        torch.testing.assert_close(results[(True, 8)][0], results[(False, None)][0], rtol=2e-2, atol=2e-2 * scale)
    # a layer that reads another layer's cache writes nothing: not a case for the fused kernel
    with pytest.raises(Exception):
        ops.qkv_rope_write(x, pw, bias, nh, nkv, d, positions, cos, sin, slots, k_cache, v_cache, page, write_kv=False, fused=True)
    before = k_cache.clone()
    ops.qkv_rope_write(x, pw, bias, nh, nkv, d, positions, cos, sin, slots, k_cache, v_cache, page, write_kv=False)
    assert torch.equal(before, k_cache)


@pytest.mark.parametrize("m", [17, 40, 64])
@pytest.mark.parametrize("nh,nkv,d,k,page,rotate", [(4, 2, 64, 128, 4, True), (28, 4, 128, 3584, 16, True), (3, 1, 32, 192, 1, True), (2, 2, 96, 1024, 8, False),
                                                    (5, 5, 48, 320, 32, True)])
def test_qkv_projection_at_17_to_64_rows_with_partial_sums_added_by_the_rotation(ops, ref, m, nh, nkv, d, k, page, rotate):
    """Split-K partial sums -> (sum, bias, rotation, cache write) in one kernel, against the same steps in float32; slots
    in runs of consecutive tokens (a prompt's portion) and scattered (decoding requests)."""
    pages = 80
    width = (nh + 2 * nkv) * d
    half = d // 2
    x = rand((m, k), torch.bfloat16, 90)
    w = rand((width, k), torch.bfloat16, 91, 0.05)
    bias = rand((width,), torch.float32, 92, 0.3)
    positions = torch.randint(0, 500, (m,), generator=torch.Generator().manual_seed(93)).to(torch.int32).cuda()
    scattered = torch.randperm((pages - 1) * page, generator=torch.Generator().manual_seed(94))[:m] + page
    consecutive = torch.arange(m) + page + 3
    angles = torch.outer(torch.arange(512, dtype=torch.float32), 1.0 / (10000.0 ** (torch.arange(half, dtype=torch.float32) / half)))
    cos, sin = (angles.cos().cuda(), angles.sin().cuda()) if rotate else (None, None)
    pw = ops.prepare_weight(w, rotary_heads=(nh, nkv, d))
    scale = float(ref.linear(x, w, None, torch.float32).abs().max())
    for slots in (scattered, consecutive):
        slots = slots.to(torch.int32).cuda()
        for use_bias in (bias, None):
            k32 = torch.full((pages, nkv, page, d), 7.0, dtype=torch.float32, device="cuda")
            v32 = torch.full((pages, nkv, d, page), 7.0, dtype=torch.float32, device="cuda")
            wide = ref.linear(x, w, None, torch.float32)
            ref.rope_kv_write(wide, nh, nkv, d, positions, cos, sin, slots, k32, v32, page, write_kv=True, bias=use_bias)
            k_cache = torch.full((pages, nkv, page, d), 7.0, dtype=torch.bfloat16, device="cuda")
            v_cache = torch.full((pages, nkv, d, page), 7.0, dtype=torch.bfloat16, device="cuda")
            for splits in (None, 1, 3):
                partial = ops.skinny_gemm_splitk(x, w, splits=splits, packed=pw.copy(1))
                q = ops.rope_kv_write_partial(partial, nh, nkv, d, positions, cos, sin, slots, k_cache, v_cache, page, bias=use_bias)
                bound = dict(rtol=1e-2, atol=1e-2 * scale)
                torch.testing.assert_close(q[:, : nh * d].float(), wide[:, : nh * d], **bound)
                torch.testing.assert_close(k_cache.float(), k32, **bound)
                torch.testing.assert_close(v_cache.float(), v32, **bound)
            # the route the engine takes for this many rows is this one
            k2, v2 = torch.full_like(k_cache, 7.0), torch.full_like(v_cache, 7.0)
            q2 = ops.qkv_rope_write(x, pw, use_bias, nh, nkv, d, positions, cos, sin, slots, k2, v2, page)
            torch.testing.assert_close(q2[:, : nh * d].float(), wide[:, : nh * d], rtol=1e-2, atol=1e-2 * scale)
            torch.testing.assert_close(k2.float(), k32, rtol=1e-2, atol=1e-2 * scale)
    # a layer that reads another layer's cache writes nothing
    before = k_cache.clone()
    ops.qkv_rope_write(x, pw, bias, nh, nkv, d, positions, cos, sin, slots, k_cache, v_cache, page, write_kv=False)
    assert torch.equal(before, k_cache)


@pytest.mark.parametrize("m", [1, 7, 16])
@pytest.mark.parametrize("hidden,inner", [(64, 128), (3584, 3584), (200, 320), (96, 18944), (5120, 192), (8192, 64)])
def test_residual_add_and_norm_split_between_two_products(ops, ref, m, hidden, inner):
    """The decode fusion: a product adds itself to the residual and applies the norm weight (DeferredNorm); the next
    product (plain, gate/up + SiLU, or q/k/v with rotation) scales its rows.  Against residual add -> RMSNorm -> product
    done one after the other."""
    from velox_amd.parts.base import DeferredNorm, ResidualSink
    from velox_amd.parts.norms import RMSNorm

    x = rand((m, inner), torch.bfloat16, 80)
    w_out = rand((hidden, inner), torch.bfloat16, 81, 0.05)
    residual0 = rand((m, hidden), torch.float32, 82, 2.0)
    norm = RMSNorm("", hidden, 1e-5)
    norm.weight = (1.0 + rand((hidden,), torch.float32, 83, 0.1))
    p_out = ops.prepare_weight(w_out)
    if hidden % 64 != 0:
        # the next product cannot stream this width: it gets the materialised rows
        pass
    # reference: product in float32 from the bfloat16 operands, add, norm
    delta = ref.linear(x, w_out, None, torch.float32)
    want_residual = residual0 + delta
    want_normed = ref.add_rmsnorm(residual0.clone(), delta, norm.weight, norm.eps, torch.float32)
    residual = residual0.clone()
    deferred = ops.linear(x, p_out, None, torch.bfloat16, partials_ok=True, residual_norm=ResidualSink(residual, norm))
    assert isinstance(deferred, DeferredNorm) and deferred.norm is norm
    torch.testing.assert_close(residual, want_residual, rtol=1e-5, atol=1e-4 * float(want_residual.abs().max()))
    torch.testing.assert_close(ops.materialize(deferred).float(), want_normed, rtol=2e-2, atol=2e-2)
    assert norm.forward(residual, deferred, None) is deferred
    for row_tiles in (1, 2, 0):  # tiles of the weight per workgroup (0: half a tile): the same sums in the same order
        again = residual0.clone()
        other = ops._linear_into_residual(x, p_out, ResidualSink(again, norm), row_tiles=row_tiles)
        assert torch.equal(again, residual) and torch.equal(other.x, deferred.x)
        blocks = (hidden + 15) // 16
        assert other.sums.shape[1] == (2 * blocks if row_tiles == 0 else blocks)
        torch.testing.assert_close(other.sums[:m].sum(1), deferred.sums[:m].sum(1), rtol=1e-5, atol=0)
        torch.testing.assert_close(ops.materialize(other).float(), ops.materialize(deferred).float(), rtol=1e-2, atol=1e-2)
    with pytest.raises(ValueError):
        RMSNorm("", hidden, 1e-5).forward(residual, deferred, None)
    if hidden % 64 != 0:
        return
    # consumers
    normed_bf16 = want_normed.to(torch.bfloat16)
    w_next = rand((320, hidden), torch.bfloat16, 84, 0.05)
    bias = rand((320,), torch.float32, 85)
    scale = float(ref.linear(normed_bf16, w_next, None, torch.float32).abs().max())
    tol = dict(rtol=2e-2, atol=2e-2 * scale)
    torch.testing.assert_close(ops.linear(deferred, w_next, bias, torch.float32), ref.linear(normed_bf16, w_next, bias, torch.float32), **tol)  # unregistered: materialised
    p_next = ops.prepare_weight(w_next)
    torch.testing.assert_close(ops.linear(deferred, p_next, bias, torch.float32), ref.linear(normed_bf16, w_next, bias, torch.float32), **tol)
    # 64 rows of the weight per wave (the variant for very tall weights), four and eight waves
    for waves in (4, 8):
        if hidden // 16 <= 64 * waves:
            got = ops.skinny_gemm(deferred.x, w_next, bias, torch.float32, waves=waves, row_tiles=4, packed=p_next.copy(1), row_scale=deferred)
            torch.testing.assert_close(got, ref.linear(normed_bf16, w_next, bias, torch.float32), **tol)
    p_next = ops.prepare_weight(w_next, stacked=2, handle=p_next)
    want_glu = ref.linear_silu_mul(normed_bf16, w_next, torch.bfloat16).float()
    torch.testing.assert_close(ops.linear_silu_mul(deferred, p_next, torch.bfloat16).float(), want_glu, rtol=3e-2, atol=3e-2 * float(want_glu.abs().max()))
    # q/k/v with rotation: 2 heads, 1 kv head, head size 80 -> 320 rows
    nh, nkv, d, page, pages = 2, 1, 80, 8, 12
    p_next = ops.prepare_weight(w_next, rotary_heads=(nh, nkv, d), handle=p_next)
    positions = torch.randint(0, 300, (m,), generator=torch.Generator().manual_seed(86)).to(torch.int32).cuda()
    slots = (torch.randperm((pages - 1) * page, generator=torch.Generator().manual_seed(87))[:m] + page).to(torch.int32).cuda()
    angles = torch.outer(torch.arange(512, dtype=torch.float32), 1.0 / (10000.0 ** (torch.arange(d // 2, dtype=torch.float32) / (d // 2))))
    cos, sin = angles.cos().cuda(), angles.sin().cuda()
    outs = []
    for source in (deferred, normed_bf16):
        k_cache = torch.zeros((pages, nkv, page, d), dtype=torch.bfloat16, device="cuda")
        v_cache = torch.zeros((pages, nkv, d, page), dtype=torch.bfloat16, device="cuda")
        q = ops.qkv_rope_write(source, p_next, bias, nh, nkv, d, positions, cos, sin, slots, k_cache, v_cache, page)
        outs.append((q[:, : nh * d].float(), k_cache.float(), v_cache.float()))
    for got, want in zip(*outs):
        torch.testing.assert_close(got, want, rtol=3e-2, atol=3e-2 * max(1.0, float(want.abs().max())))


def _rows_from_lanes_order(twin, k):
    """[k / 64 * 1024] in the order the skinny kernels' lanes read activations -> [16, k]."""
    return twin.view(k // 64, 2, 4, 16, 8).permute(3, 0, 2, 1, 4).reshape(16, k)


@pytest.mark.parametrize("m", [1, 5, 13, 16])
def test_decode_activations_handed_on_in_the_lanes_order(ops, ref, m, monkeypatch):
    """The gate/up kernel and the residual-add kernel leave their result a second time in the order the next product's
    lanes read it; a product gives the same bits whether it reads that copy or the row-major one."""
    from velox_amd.parts.base import DeferredNorm, ResidualSink
    from velox_amd.parts.norms import RMSNorm

    # (the engine asks for the copy from 13 rows on, where it pays; the kernels take any number up to 16)
    monkeypatch.setattr(ops, "_room_for_packed_rows", lambda rows, n: torch.empty(n // 64 * 1024, dtype=torch.bfloat16, device="cuda") if rows <= 16 and n % 64 == 0 else None)
    hidden, inner = 256, 448
    x = rand((m, hidden), torch.bfloat16, 90)
    w_gu = rand((2 * inner, hidden), torch.bfloat16, 91, 0.05)
    w_down = rand((hidden, inner), torch.bfloat16, 92, 0.05)
    p_gu = ops.prepare_weight(w_gu, stacked=2)
    p_down = ops.prepare_weight(w_down)
    act = ops.linear_silu_mul(x, p_gu, torch.bfloat16)
    twin, version = act._velox_packed_rows
    assert version == act._version and torch.equal(_rows_from_lanes_order(twin, inner)[:m], act)
    norm = RMSNorm("", hidden, 1e-6)
    norm.weight = 1.0 + rand((hidden,), torch.float32, 93, 0.1)
    results = []
    for use_twin in (True, False):
        source = act if use_twin else act.clone()  # (a clone is another tensor object: no copy hangs on it)
        assert (ops._packed_rows_of(source, inner) is not None) == use_twin
        residual = rand((m, hidden), torch.float32, 94)
        deferred = ops.linear(source, p_down, None, torch.bfloat16, partials_ok=True, residual_norm=ResidualSink(residual, norm))
        assert isinstance(deferred, DeferredNorm)
        next_twin = ops._packed_rows_of(deferred.x, hidden)
        assert torch.equal(_rows_from_lanes_order(next_twin, hidden)[:m], deferred.x)
        results.append((residual, deferred.x.clone(), deferred.sums[:m].clone(), deferred))
    for a, b in zip(results[0][:3], results[1][:3]):
        assert torch.equal(a, b)
    # the consumers of a DeferredNorm, with and without its copy
    deferred = results[0][3]
    plain = DeferredNorm(deferred.x.clone(), deferred.sums, deferred.width, deferred.eps, deferred.norm)
    bias = rand((2 * inner,), torch.float32, 95)
    assert torch.equal(ops.linear(deferred, p_gu, bias, torch.float32), ops.linear(plain, p_gu, bias, torch.float32))
    assert torch.equal(ops.linear_silu_mul(deferred, p_gu, torch.bfloat16), ops.linear_silu_mul(plain, p_gu, torch.bfloat16))
    nh, nkv, d, page, pages = 3, 2, 128, 16, 6  # (3 + 2 * 2) * 128 = 896 = 2 * inner rows
    p_gu = ops.prepare_weight(w_gu, rotary_heads=(nh, nkv, d), handle=p_gu)
    positions = torch.arange(m, dtype=torch.int32, device="cuda") * 7
    slots = (torch.randperm((pages - 1) * page, generator=torch.Generator().manual_seed(96))[:m] + page).to(torch.int32).cuda()
    angles = torch.outer(torch.arange(128, dtype=torch.float32), 1.0 / (10000.0 ** (torch.arange(d // 2, dtype=torch.float32) / (d // 2))))
    cos, sin = angles.cos().cuda(), angles.sin().cuda()
    outs = []
    for source in (deferred, plain):
        k_cache = torch.zeros((pages, nkv, page, d), dtype=torch.bfloat16, device="cuda")
        v_cache = torch.zeros((pages, nkv, d, page), dtype=torch.bfloat16, device="cuda")
        q = ops.qkv_rope_write(source, p_gu, bias, nh, nkv, d, positions, cos, sin, slots, k_cache, v_cache, page, fused=True)
        outs.append((q, k_cache, v_cache))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    # a copy goes stale with its tensor
    act.add_(1)
    assert ops._packed_rows_of(act, inner) is None


def _attention_case(dtype, nh, nkv, d, page, seqs, seed, garbage=False):
    """seqs: list of (q_len, kv_len).  Builds a paged cache with shuffled pages and a flat qkv."""
    g = torch.Generator().manual_seed(seed)
    total_pages = sum((kv + page - 1) // page for _, kv in seqs) + 3
    perm = (torch.randperm(total_pages - 1, generator=g) + 1).tolist()
    k_cache = torch.zeros((total_pages, nkv, page, d), dtype=dtype)
    v_cache = torch.zeros((total_pages, nkv, d, page), dtype=dtype)
    if garbage:
        k_cache.normal_(0, 50.0, generator=g)
        v_cache.normal_(0, 50.0, generator=g)
    width = max((kv + page - 1) // page for _, kv in seqs)
    tables = torch.zeros((len(seqs), width), dtype=torch.int32)
    tokens = sum(q for q, _ in seqs)
    qkv = (torch.randn((tokens, (nh + 2 * nkv) * d), generator=g)).to(dtype)
    cu = [0]
    for b, (q_len, kv_len) in enumerate(seqs):
        n_pages = (kv_len + page - 1) // page
        mine = [perm.pop() for _ in range(n_pages)]
        tables[b, :n_pages] = torch.tensor(mine, dtype=torch.int32)
        keys = torch.randn((kv_len, nkv, d), generator=g).to(dtype)
        values = torch.randn((kv_len, nkv, d), generator=g).to(dtype)
        for n in range(kv_len):
            k_cache[mine[n // page], :, n % page, :] = keys[n]
            v_cache[mine[n // page], :, :, n % page] = values[n]
        cu.append(cu[-1] + q_len)
    return dict(
        qkv=qkv.cuda(), k_cache=k_cache.cuda(), v_cache=v_cache.cuda(), tables=tables.cuda(),
        cu=torch.tensor(cu, dtype=torch.int32).cuda(), kv=torch.tensor([kv for _, kv in seqs], dtype=torch.int32).cuda(),
        max_q=max(q for q, _ in seqs), max_kv=max(kv for _, kv in seqs),
    )


def _run_attention(impl, case, nh, nkv, d, page, window=None, splits=None, all_decode=False, workspace=None):
    return impl.paged_attention(
        case["qkv"], nh, nkv, d, case["k_cache"], case["v_cache"], page, case["tables"], case["cu"], case["kv"],
        case["max_q"], case["max_kv"], 1.0 / math.sqrt(d), window, all_decode, workspace, splits=splits,
    ).float()


ATTN_SHAPES = [(4, 2, 16, 4), (3, 1, 32, 8), (6, 2, 48, 16), (28, 4, 128, 16), (8, 8, 64, 64), (7, 1, 96, 32), (2, 1, 256, 16), (40, 8, 128, 2), (5, 1, 80, 8),
               (6, 2, 192, 16)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,d,page", ATTN_SHAPES)
def test_paged_attention_mixed_batch(ops, ref, dtype, nh, nkv, d, page):
    # whole prompts, a portion with earlier context, single decoded tokens, a two-token portion
    seqs = [(70, 70), (33, 141), (1, 97), (2, 66), (1, 1), (130, 130)]
    case = _attention_case(dtype, nh, nkv, d, page, seqs, seed=d + nh)
    got = _run_attention(ops, case, nh, nkv, d, page)
    want = _run_attention(ref, case, nh, nkv, d, page)
    torch.testing.assert_close(got, want, **(dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,d,page", ATTN_SHAPES)
@pytest.mark.parametrize("window", [None, 200])
def test_paged_attention_decoded_tokens_before_portions(ops, ref, dtype, nh, nkv, d, page, window):
    """A mixed step as the engine lays it out: single decoded tokens first (one of them behind a long context), then
    portions of prompts.  Told how many sequences lead with one token, the wrapper sends those through the streaming
    kernel with split keys and the rest through the general kernel; every row agrees with the plain reference, and
    the decoded rows with the same rows in a step of their own, to the bit."""
    from velox_amd.engine.batch import Workspace

    seqs = [(1, 2300), (1, 97), (1, 1), (1, 640), (33, 141), (2, 66), (70, 70), (1, 30)]
    case = _attention_case(dtype, nh, nkv, d, page, seqs, seed=d + nh + 2)
    workspace = Workspace(torch.device("cuda"))
    tolerance = dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)
    want = _run_attention(ref, case, nh, nkv, d, page, window=window)
    one_launch = _run_attention(ops, case, nh, nkv, d, page, window=window, workspace=workspace)
    got = ops.paged_attention(case["qkv"], nh, nkv, d, case["k_cache"], case["v_cache"], page, case["tables"], case["cu"], case["kv"],
                              case["max_q"], case["max_kv"], 1.0 / math.sqrt(d), window, False, workspace, decode_prefix=4).float()
    torch.testing.assert_close(got, want, **tolerance)
    torch.testing.assert_close(one_launch, want, **tolerance)
    assert torch.equal(got[4:], one_launch[4:])  # the general kernel's rows do not depend on who else is in the launch
    alone = dict(case)
    alone["qkv"], alone["tables"], alone["kv"] = case["qkv"][:4].contiguous(), case["tables"][:4].contiguous(), case["kv"][:4].contiguous()
    alone["cu"] = torch.arange(5, dtype=torch.int32, device="cuda")
    alone["max_q"] = 1
    decoded = _run_attention(ops, alone, nh, nkv, d, page, window=window, all_decode=True, workspace=workspace)
    assert torch.equal(got[:4], decoded)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,d,page", [(28, 4, 128, 16), (4, 2, 16, 4), (2, 1, 256, 16), (12, 2, 128, 32)])
def test_paged_attention_portions_behind_many_keys_split_them(ops, ref, dtype, nh, nkv, d, page):
    """Few prompt tokens behind thousands of keys: the wrapper splits the keys over workgroups (and merges), alone and
    behind decoded tokens that lead the step (whose rows the second launch's merge must leave alone)."""
    from velox_amd.engine.batch import Workspace

    seqs = [(1, 4500), (1, 10), (150, 4400), (40, 40), (2, 4200)]
    case = _attention_case(dtype, nh, nkv, d, page, seqs, seed=d + nh + 3)
    workspace = Workspace(torch.device("cuda"))
    tolerance = dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)
    assert ops.choose_portion_splits(192, nh // nkv, nkv, 4500) > 1
    want = _run_attention(ref, case, nh, nkv, d, page)
    for prefix in (0, 2):
        got = ops.paged_attention(case["qkv"], nh, nkv, d, case["k_cache"], case["v_cache"], page, case["tables"], case["cu"], case["kv"],
                                  case["max_q"], case["max_kv"], 1.0 / math.sqrt(d), None, False, workspace, decode_prefix=prefix).float()
        torch.testing.assert_close(got, want, **tolerance)
    one_pass = _run_attention(ops, case, nh, nkv, d, page, splits=1, workspace=workspace)
    torch.testing.assert_close(one_pass, want, **tolerance)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,d,page", [(28, 4, 128, 16), (32, 16, 64, 64), (16, 8, 32, 8), (24, 12, 48, 4)])
@pytest.mark.parametrize("window", [None, 300])
def test_paged_attention_long_portions(ops, ref, dtype, nh, nkv, d, page, window):
    """Steps with thousands of rows take the 128-row workgroups in bfloat16: long whole prompts, a long portion behind
    a longer context, and short entries beside them.  A row's result is the same as in a small step, to rounding (the
    large workgroups add a row's keys in another order) and to the bit in float32, which has one kind of workgroup."""
    seqs = [(1100, 1100), (700, 1300), (1, 97), (300, 300), (2, 40)]
    case = _attention_case(dtype, nh, nkv, d, page, seqs, seed=d + nh + 1)
    got = _run_attention(ops, case, nh, nkv, d, page, window=window)
    want = _run_attention(ref, case, nh, nkv, d, page, window=window)
    torch.testing.assert_close(got, want, **(dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)))
    # the 300-token prompt again, in a step of its own (64-row workgroups): its rows must not have changed
    first = sum(q for q, _ in seqs[:3])
    alone = dict(case)
    alone["qkv"] = case["qkv"][first:first + 300].contiguous()
    alone["tables"] = case["tables"][3:4].contiguous()
    alone["cu"] = torch.tensor([0, 300], dtype=torch.int32, device="cuda")
    alone["kv"] = case["kv"][3:4].contiguous()
    alone["max_q"], alone["max_kv"] = 300, 300
    same = dict(rtol=0, atol=0) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(_run_attention(ops, alone, nh, nkv, d, page, window=window), got[first:first + 300], **same)


@pytest.mark.parametrize("nh,nkv,d,page", [(4, 2, 16, 4), (6, 2, 48, 16), (5, 1, 80, 8), (7, 1, 96, 32), (28, 4, 128, 16), (40, 8, 128, 2)])
@pytest.mark.parametrize("window,splits", [(None, None), (90, None), (None, 3)])
def test_float32_row_tiles_that_waves_share_keep_their_bits(ops, ref, nh, nkv, d, page, window, splits):
    """Float32 portions of few rows: waves that share a row tile (each a part of the keys, then a part of the channels) give the
    bits of one wave per row tile, in workgroups of 16, 32 and 64 rows (1 row, one short of a row tile, one beyond it, several
    workgroups; key tiles that only some of a workgroup's rows read), and with them whatever the launcher picks."""
    from velox_amd.engine.batch import Workspace

    seqs = [(1, 97), (15, 15), (17, 145), (64, 64), (65, 193), (130, 130), (2, 66)]
    case = _attention_case(torch.float32, nh, nkv, d, page, seqs, seed=d + nh + 4)
    workspace = Workspace(torch.device("cuda"))
    lib = ops.attention_library(d)
    got = {}
    try:
        for choice in (1, 2, 3, 4, 0):
            lib.velox_attention_portion_kernel(choice)
            got[choice] = _run_attention(ops, case, nh, nkv, d, page, window=window, splits=splits, workspace=workspace)
    finally:
        lib.velox_attention_portion_kernel(0)
    torch.testing.assert_close(got[1], _run_attention(ref, case, nh, nkv, d, page, window=window), rtol=1e-4, atol=1e-5)
    for choice in (2, 3, 4, 0):
        assert torch.equal(got[choice], got[1]), choice


@pytest.mark.parametrize("nh,nkv,d,seqs,window", [(32, 8, 16, [(300, 2000)], None), (12, 12, 48, [(2048, 2048)], None), (16, 16, 80, [(1024, 1024)], 256), (28, 4, 128, [(64, 64)] * 16, None),
                                                  (12, 2, 128, [(850, 850)], 128), (12, 2, 128, [(1024, 1024)], 256), (32, 8, 96, [(1024, 1024)], 256)])
def test_float32_row_tiles_are_shared_only_where_that_is_no_slower(ops, nh, nkv, d, seqs, window):
    """Steps where waves that share row tiles would take 1.1 to 1.4 times as long as a row tile per wave: the launcher's choice is within 6%, what
    two timings of the same kernels may differ by."""
    from velox_amd.kernels.measure import time_in_graph

    case, lib = _attention_case(torch.float32, nh, nkv, d, 16, seqs, seed=d), ops.attention_library(d)
    times = {}
    try:
        for choice in (1, 0, 1, 0):
            lib.velox_attention_portion_kernel(choice)
            times[choice] = min(times.get(choice, 1e9), time_in_graph(lambda: _run_attention(ops, case, nh, nkv, d, 16, window=window)))
    finally:
        lib.velox_attention_portion_kernel(0)
    assert times[0] <= 1.06 * times[1], times


@pytest.mark.parametrize("dtype,nh,nkv,d,page,long_context,choices", [
    (torch.bfloat16, 14, 2, 128, 8, 17000, (1, 2, 3)), (torch.bfloat16, 6, 3, 64, 8, 16500, (2, 3)), (torch.float32, 4, 2, 32, 4, 9000, (0,))])
@pytest.mark.parametrize("window", [None, 5000])
def test_paged_attention_behind_more_pages_than_the_kernels_keep_ids_of(ops, ref, dtype, nh, nkv, d, page, long_context, choices, window):
    """A workgroup keeps the page ids of the keys it visits in LDS, 2,048 at a time, and fetches the next lot when its
    tiles leave the window: portions behind contexts of more than 2,048 pages in one pass over the keys (no split), in
    every kernel for portions, with a short sequence and a single token behind the long context beside them."""
    from velox_amd.engine.batch import Workspace

    assert long_context // page > 2048
    seqs = [(200, long_context), (64, 64), (1, long_context - 300)]
    case = _attention_case(dtype, nh, nkv, d, page, seqs, seed=d + nh + 5)
    want = _run_attention(ref, case, nh, nkv, d, page, window=window)
    tolerance = dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)
    lib = ops.attention_library(d)
    workspace = Workspace(torch.device("cuda"))
    try:
        for choice in choices:
            lib.velox_attention_portion_kernel(choice)
            got = _run_attention(ops, case, nh, nkv, d, page, window=window, splits=1, workspace=workspace)
            torch.testing.assert_close(got, want, **tolerance)
    finally:
        lib.velox_attention_portion_kernel(0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,d,page", [(28, 4, 128, 16), (4, 2, 16, 4), (6, 2, 96, 8), (8, 8, 64, 1)])
@pytest.mark.parametrize("window", [None, 200])
def test_paged_attention_few_rows_many_keys(ops, ref, dtype, nh, nkv, d, page, window):
    """Short portions behind long contexts: few workgroups, each with many key tiles (in bfloat16 two sets of waves
    then share a workgroup's tiles, an odd number of tiles included)."""
    seqs = [(40, 900), (3, 705), (1, 520), (17, 64 * 9 + 17)]
    case = _attention_case(dtype, nh, nkv, d, page, seqs, seed=d + nh + 2)
    got = _run_attention(ops, case, nh, nkv, d, page, window=window)
    want = _run_attention(ref, case, nh, nkv, d, page, window=window)
    torch.testing.assert_close(got, want, **(dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,d,page", [(4, 2, 16, 4), (28, 4, 128, 16), (3, 1, 32, 8)])
def test_paged_attention_garbage_in_unused_slots_and_null_page(ops, ref, dtype, nh, nkv, d, page):
    seqs = [(5, 37), (1, 64), (9, 9)]
    clean = _attention_case(dtype, nh, nkv, d, page, seqs, seed=3)
    dirty = _attention_case(dtype, nh, nkv, d, page, seqs, seed=3, garbage=True)
    # same seed: same real keys, values and queries? the garbage draw shifts the stream, so copy them over
    dirty["qkv"] = clean["qkv"]
    tables = clean["tables"].cpu()
    for b, (_, kv_len) in enumerate(seqs):
        for n in range(kv_len):
            p, o = int(tables[b, n // page]), n % page
            dirty["k_cache"][p, :, o, :] = clean["k_cache"][p, :, o, :]
            dirty["v_cache"][p, :, :, o] = clean["v_cache"][p, :, :, o]
    dirty["tables"] = clean["tables"]
    got_clean = _run_attention(ops, clean, nh, nkv, d, page)
    got_dirty = _run_attention(ops, dirty, nh, nkv, d, page)
    torch.testing.assert_close(got_dirty, got_clean, rtol=0, atol=0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,d,page", [(4, 2, 16, 4), (28, 4, 128, 16), (7, 1, 96, 32)])
@pytest.mark.parametrize("window", [1, 5, 64, 100])
def test_paged_attention_window(ops, ref, dtype, nh, nkv, d, page, window):
    seqs = [(70, 70), (33, 141), (1, 197), (2, 66)]
    case = _attention_case(dtype, nh, nkv, d, page, seqs, seed=11)
    got = _run_attention(ops, case, nh, nkv, d, page, window=window)
    want = _run_attention(ref, case, nh, nkv, d, page, window=window)
    torch.testing.assert_close(got, want, **(dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)))


@pytest.mark.parametrize("nh,nkv,d,page", [(28, 4, 128, 16), (12, 2, 128, 8), (8, 8, 64, 64), (6, 3, 64, 16), (5, 1, 128, 32)])
@pytest.mark.parametrize("window", [None, 300])
def test_paged_attention_with_tiles_loaded_straight_into_lds(ops, ref, nh, nkv, d, page, window):
    """The kernel for portions of prompts whose tiles of keys and values reach LDS by direct loads (bfloat16, head sizes 64
    and 128, pages of 8 tokens and more), made to run wherever it can, beside the kernel it stands in for: whole prompts
    whose lengths are no multiple of a tile or of a piece of eight keys, portions behind longer contexts, short
    entries beside them, pages in no order, and loud garbage in every slot beyond the sequences' ends (values there must
    not reach the output, not even multiplied with a probability of zero) and on the null page."""
    from velox_amd.engine.batch import Workspace

    lib = ops.attention_library(d)
    seqs = [(1100, 1100), (700, 1301), (1, 97), (300, 300), (2, 40), (67, 67), (130, 1003)]
    case = _attention_case(torch.bfloat16, nh, nkv, d, page, seqs, seed=d + nh + 7)
    dirty = _attention_case(torch.bfloat16, nh, nkv, d, page, seqs, seed=d + nh + 7, garbage=True)
    dirty["qkv"], dirty["tables"] = case["qkv"], case["tables"]
    tables = case["tables"].cpu()
    used = torch.zeros(dirty["k_cache"].shape[0], page, dtype=torch.bool)
    for b, (_, kv_len) in enumerate(seqs):
        for n in range(kv_len):
            used[int(tables[b, n // page]), n % page] = True
    keep = used.cuda()
    dirty["k_cache"] = torch.where(keep[:, None, :, None], case["k_cache"], dirty["k_cache"] * float("inf"))  # +-inf where no key lives
    dirty["v_cache"] = torch.where(keep[:, None, None, :], case["v_cache"], dirty["v_cache"] * float("inf"))
    tolerance = dict(rtol=2e-2, atol=2e-2)
    want = _run_attention(ref, case, nh, nkv, d, page, window=window)
    try:
        results = {}
        for choice in (1, 2, 3):  # (the kernels it stands in for; direct loads; direct loads with two sets of waves)
            lib.velox_attention_portion_kernel(choice)
            results[choice] = _run_attention(ops, case, nh, nkv, d, page, window=window)
            torch.testing.assert_close(results[choice], want, **tolerance)
            assert torch.equal(_run_attention(ops, dirty, nh, nkv, d, page, window=window), results[choice])
        # three kernels did run (they add a row's keys in different orders)
        assert not torch.equal(results[1], results[2]) and not torch.equal(results[2], results[3])
        # split keys (few tokens behind many keys) through the same kernels, and the partial results merged
        far = _attention_case(torch.bfloat16, nh, nkv, d, page, [(150, 4400), (90, 90), (2, 4200)], seed=d + nh + 8)
        workspace = Workspace(torch.device("cuda"))
        for choice in (2, 3):
            lib.velox_attention_portion_kernel(choice)
            for splits in (1, 3, 4):
                got = _run_attention(ops, far, nh, nkv, d, page, window=window, splits=splits, workspace=workspace)
                torch.testing.assert_close(got, _run_attention(ref, far, nh, nkv, d, page, window=window), **tolerance)
        # Scores that climb along the sequence, slowly (a row's best score moves up a little with every tile, so the
        # reference of its exponents lags behind and catches up every few tiles) and in jumps (far above everything seen):
        # the kernels with direct loads keep a reference that need not be the maximum
        climbing = _attention_case(torch.bfloat16, nh, nkv, d, page, [(900, 900), (400, 1100)], seed=d + nh + 9)
        direction = torch.randn(d, generator=torch.Generator().manual_seed(3))
        direction = direction / direction.norm()
        tables = climbing["tables"].cpu()
        for b, kv_len in enumerate((900, 1100)):
            for n in range(kv_len):
                height = 0.07 * n + (40.0 if n in (300, 301, 777) else 0.0)
                climbing["k_cache"][int(tables[b, n // page]), :, n % page, :] += (height * direction).to(torch.bfloat16).cuda()
        climbing["qkv"][:, : nh * d] = (climbing["qkv"][:, : nh * d].float() * 0.3 + (direction * math.sqrt(d)).repeat(nh).cuda()).to(torch.bfloat16)
        want = _run_attention(ref, climbing, nh, nkv, d, page, window=window)
        for choice in (1, 2, 3):
            lib.velox_attention_portion_kernel(choice)
            torch.testing.assert_close(_run_attention(ops, climbing, nh, nkv, d, page, window=window), want, **tolerance)
    finally:
        lib.velox_attention_portion_kernel(0)


@pytest.mark.parametrize("seed", [0, 1, 2, 3])
def test_paged_attention_random_steps_agree_with_the_reference(ops, ref, seed):
    """Steps drawn at random: head size, heads and groups, page size, data type, window, splits of the keys, which kernel
    takes the portions, and one to six sequences that are single tokens, short portions or long ones, from an empty
    cache or behind up to 5,000 keys."""
    import random

    from velox_amd.engine.batch import Workspace

    rng = random.Random(seed)
    workspace = Workspace(torch.device("cuda"))
    for case_no in range(12):
        d = rng.choice([16, 48, 64, 80, 96, 128, 192, 256])
        page = rng.choice([1, 2, 4, 8, 16, 32, 64, 128])
        dtype = rng.choice(DTYPES)
        nkv = rng.choice([1, 2, 4, 8])
        nh = nkv * rng.choice([1, 2, 3, 5, 7])
        seqs = []
        for _ in range(rng.randint(1, 6)):
            kind = rng.random()
            q = 1 if kind < 0.25 else rng.randint(2, 70) if kind < 0.5 else rng.randint(71, 900)
            seqs.append((q, q + rng.choice([0, 0, rng.randint(1, 300), rng.randint(300, 5000)])))
        window = rng.choice([None, None, rng.randint(1, 3000)])
        choice = rng.choice([0, 0, 1, 2, 3])
        splits = rng.choice([None, None, 1, 2, 3])
        case = _attention_case(dtype, nh, nkv, d, page, seqs, seed=100 * seed + case_no)
        lib = ops.attention_library(d)
        lib.velox_attention_portion_kernel(choice)
        try:
            got = _run_attention(ops, case, nh, nkv, d, page, window=window, splits=splits, workspace=workspace)
        finally:
            lib.velox_attention_portion_kernel(0)
        want = _run_attention(ref, case, nh, nkv, d, page, window=window)
        said = f"seed {seed} case {case_no}: {dtype} d={d} page={page} heads {nh}/{nkv} {seqs} window={window} kernel {choice} splits={splits}"
        torch.testing.assert_close(got, want, msg=lambda m: f"{said}: {m}", **(dict(rtol=2e-2, atol=2e-2) if dtype == torch.bfloat16 else dict(rtol=1e-4, atol=2e-5)))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,d,page", [(4, 2, 16, 4), (28, 4, 128, 16), (3, 1, 32, 8), (2, 1, 256, 16)])
def test_decode_split_keys_equals_one_pass(ops, ref, dtype, nh, nkv, d, page):
    from velox_amd.engine.batch import Workspace

    seqs = [(1, 700), (1, 3), (1, 129), (1, 64), (1, 1)]
    case = _attention_case(dtype, nh, nkv, d, page, seqs, seed=21)
    workspace = Workspace(torch.device("cuda"))
    one = _run_attention(ops, case, nh, nkv, d, page, splits=1, all_decode=True, workspace=workspace)
    want = _run_attention(ref, case, nh, nkv, d, page)
    t = dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(one, want, **t)
    for splits in (2, 3, 8, 32):  # 32 splits leave most of them empty for the short sequences
        got = _run_attention(ops, case, nh, nkv, d, page, splits=splits, all_decode=True, workspace=workspace)
        torch.testing.assert_close(got, want, **t)


@pytest.mark.parametrize("dtype", DTYPES)
def test_decode_behind_more_pages_than_the_streaming_kernel_keeps_ids_of(ops, ref, dtype):
    """The streaming kernel keeps the page ids of a split's keys in LDS; a split of more pages than it has room for
    (2,048) goes through the kernel for portions instead, with the same result; with more splits the streaming kernel
    takes it again."""
    from velox_amd.engine.batch import Workspace

    nh, nkv, d, page = 6, 2, 64, 4
    seqs = [(1, 9000), (1, 77), (1, 8300)]
    case = _attention_case(dtype, nh, nkv, d, page, seqs, seed=31)
    workspace = Workspace(torch.device("cuda"))
    want = _run_attention(ref, case, nh, nkv, d, page)
    t = dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)
    for splits in (1, 2, 8):  # 1 and 2: 2,250 and 1,125 + 2 pages per split, beyond and within the room for ids
        got = _run_attention(ops, case, nh, nkv, d, page, splits=splits, all_decode=True, workspace=workspace)
        torch.testing.assert_close(got, want, **t)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,d,page,lens,window", [
    (28, 4, 128, 16, [1500, 65, 130, 300, 1, 700, 16, 17], None),  # some in several parts, some in one
    (28, 4, 128, 16, [3000] + [20] * 70, None),  # more sequences than a wave has lanes, one far longer
    (6, 2, 64, 4, [9000, 77, 8300, 5, 500, 31, 32, 33] * 2, None),  # more page ids than a part has room for
    (4, 2, 16, 4, [900, 1, 1, 1, 250, 128, 129, 127] * 2, 200),  # a window bounds what a sequence's share is
    (32, 8, 64, 64, [640] * 9, None),  # all alike
    (3, 1, 256, 8, [2000 - 60 * b for b in range(32)], None),
])
def test_decoded_tokens_whose_keys_are_shared_out(ops, ref, dtype, nh, nkv, d, page, lens, window):
    """Single tokens behind unequal contexts, their keys shared out over the workgroups by how many each sequence has: the
    reference's results, the same bits again (the counters of arrivals are left at zero), and those of the sequences in another
    order as far as the parts they are cut in are the same."""
    from velox_amd.engine.batch import Workspace

    assert d * (4 if dtype == torch.float32 else 2) > 512 or ops.shares_keys(len(lens), nkv)
    case = _attention_case(dtype, nh, nkv, d, page, [(1, n) for n in lens], seed=d + len(lens))
    workspace = Workspace(torch.device("cuda"))

    def run(case, **more):
        return ops.paged_attention(case["qkv"], nh, nkv, d, case["k_cache"], case["v_cache"], page, case["tables"], case["cu"], case["kv"], 1, case["max_kv"],
                                   1.0 / math.sqrt(d), window, True, workspace, uneven=True, **more).float()

    got = run(case)
    want = _run_attention(ref, case, nh, nkv, d, page, window=window)
    torch.testing.assert_close(got, want, **(dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)))
    if "attention_arrivals" in workspace.addresses():
        assert not workspace.get("attention_arrivals", len(lens) * nkv).any()
    assert torch.equal(run(case), got)
    order = torch.randperm(len(lens), generator=torch.Generator().manual_seed(1)).cuda()
    moved = dict(case, qkv=case["qkv"][order].contiguous(), tables=case["tables"][order].contiguous(), kv=case["kv"][order].contiguous())
    assert torch.equal(run(moved), got[order])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("sinks", [False, True])
@pytest.mark.parametrize("nh,nkv,d,page", [(28, 4, 128, 16), (4, 4, 64, 4)])
def test_a_captured_step_shares_its_keys_out_by_the_lengths_of_each_replay(ops, ref, dtype, sinks, nh, nkv, d, page):
    """One launch captured for up to 4,096 keys (9,000 with pages of four tokens, more page ids than a share has room for) and a workspace that is as
    large as was asked for: its replays cut the sequences by their lengths, and leave the counters of arrivals at zero."""
    from velox_amd.engine.batch import Workspace

    most = 4096 if page == 16 else 9000
    case = _attention_case(dtype, nh, nkv, d, page, [(1, most - 7 * b) for b in range(16)], seed=7)
    out_elems, lse_elems = ops.attention_scratch_elems(nh, nkv, d, 16, 16, most, block_size=page)
    workspace = Workspace(torch.device("cuda"))
    for name, elems in (("attention_partial_out", out_elems), ("attention_partial_lse", lse_elems), ("attention_arrivals", 16 * nkv)):
        workspace.reserve(name, elems)
    workspace.fix()
    sink = rand((nh,), torch.float32, 8, 2.0) if sinks else None

    def run():
        return ops.paged_attention(case["qkv"], nh, nkv, d, case["k_cache"], case["v_cache"], page, case["tables"], case["cu"], case["kv"], 1, most, 1.0 / math.sqrt(d),
                                   None, True, workspace, uneven=True, sinks=sink)

    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with collection_held(), torch.cuda.graph(graph):
        captured = run()
    full = case["kv"].tolist()
    for lens in ([30 + b for b in range(16)], full, [1] * 15 + [full[15]], full[:1] + [17] * 15, [500, 1, 2000, 64, 65, 300, 1500, 16] * 2, [1] * 16):
        case["kv"].copy_(torch.tensor(lens, dtype=torch.int32))
        for _ in range(2):
            graph.replay()
            got = captured.clone()
            torch.cuda.synchronize()
            assert not workspace.get("attention_arrivals", 16 * nkv).any()
            assert torch.equal(got, run())
        want = ref.paged_attention(case["qkv"], nh, nkv, d, case["k_cache"], case["v_cache"], page, case["tables"], case["cu"], case["kv"], 1, max(lens), 1.0 / math.sqrt(d),
                                   None, True, None, sinks=sink).float()
        torch.testing.assert_close(got.float(), want, **(dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)))


@pytest.mark.parametrize("dtype", DTYPES)
def test_an_infinite_value_stays_infinite_whatever_merges_the_splits(ops, dtype):
    """A value of infinity behind a key that counts makes its channel infinite, not a number that is none, also where a merge asks for more parts
    than there are."""
    from velox_amd.engine.batch import Workspace
    from velox_amd.parts.base import ResidualSink
    from velox_amd.parts.norms import RMSNorm

    nh, nkv, d, page = 8, 4, 64, 16
    case = _attention_case(dtype, nh, nkv, d, page, [(1, 700 + b) for b in range(8)], seed=12)
    for b in range(8):  # the last key of every sequence, in the last split
        case["v_cache"][case["tables"][b, (699 + b) // page].long(), 0, 5 + b, (699 + b) % page] = float("inf")
    workspace = Workspace(torch.device("cuda"))
    assert ops.shares_keys(8, nkv)
    want = _run_attention(ops, case, nh, nkv, d, page, all_decode=True, splits=1, workspace=workspace)
    assert int(want.isinf().sum()) == 8 * nh // nkv and not want.isnan().any()
    for more in ({"uneven": True}, {"splits": 3}):
        got = ops.paged_attention(case["qkv"], nh, nkv, d, case["k_cache"], case["v_cache"], page, case["tables"], case["cu"], case["kv"], 1, case["max_kv"], 1.0 / math.sqrt(d), None,
                                  True, workspace, **more).float()
        torch.testing.assert_close(got, want, **(dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)))
    if dtype == torch.bfloat16:
        weight, norm, results = ops.prepare_weight(rand((512, nh * d), dtype, 13, 0.05)), RMSNorm("", 512, 1e-5), []
        norm.weight = torch.ones(512, device="cuda")
        for more in ({"splits": 1}, {"parts": 2}, {"parts": 3}, {"parts": 8}):
            residual = torch.zeros((2, 512), device="cuda")
            attention = ops.paged_attention(case["qkv"][:2], nh, nkv, d, case["k_cache"], case["v_cache"], page, case["tables"][:2], case["cu"][:3], case["kv"][:2], 1, case["max_kv"],
                                            1.0 / math.sqrt(d), None, True, workspace, **more)
            ops.linear(attention, weight, None, dtype, residual_norm=ResidualSink(residual, norm))
            results.append(residual)
        for got in results[1:]:
            assert results[0].isinf().any() and torch.equal(got.isnan(), results[0].isnan()) and torch.equal(got.isinf(), results[0].isinf())


@pytest.mark.parametrize("dtype", DTYPES)
def test_keys_shared_out_in_front_of_portions(ops, ref, dtype):
    """A mixed step: its single tokens' shares and its portions' splits use the same scratch, one after the other."""
    from velox_amd.engine.batch import Workspace

    nh, nkv, d, page = 16, 4, 64, 16
    lens = [900, 3, 250, 64, 1, 2000, 128, 129, 17, 16]
    case = _attention_case(dtype, nh, nkv, d, page, [(1, n) for n in lens] + [(70, 4500), (3, 3)], seed=9)
    workspace = Workspace(torch.device("cuda"))
    assert ops.shares_keys(len(lens), nkv)

    def run(**more):
        return ops.paged_attention(case["qkv"], nh, nkv, d, case["k_cache"], case["v_cache"], page, case["tables"], case["cu"], case["kv"], 70, 4500, 1.0 / math.sqrt(d), None,
                                   False, workspace, decode_prefix=len(lens), portions_max_kv_len=4500, **more).float()

    got = run(uneven=True)
    want = _run_attention(ref, case, nh, nkv, d, page)
    torch.testing.assert_close(got, want, **(dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)))
    assert not workspace.get("attention_arrivals", len(lens) * nkv).any()
    assert torch.equal(run(uneven=True), got) and torch.equal(run()[len(lens):], got[len(lens):])


@pytest.mark.parametrize("count,items", [(65280, None), (65535, None), (100, 65536), (100, 65535)])
def test_more_decoded_tokens_or_shares_than_a_grid_has_room_for(ops, monkeypatch, count, items):
    """Single tokens up to 65,535 were always taken, and so are a hundred whose contexts may be so long that there could be more shares of keys
    than the grid's second dimension has room for: their keys are then split equally."""
    from velox_amd.engine.batch import Workspace

    d, page = 16, 16
    k_cache, v_cache = rand((2, 1, page, d), torch.float32, 81), rand((2, 1, d, page), torch.float32, 82)
    q = rand((count, d), torch.float32, 83)
    kv = torch.arange(count, dtype=torch.int32).remainder(page).add(1).cuda()
    tables = torch.ones((count, 1), dtype=torch.int32, device="cuda")
    if items is not None:
        monkeypatch.setattr(ops, "_shared_items", lambda *sizes: items)
    workspace = Workspace(torch.device("cuda"))
    got = ops.paged_attention(q, 1, 1, d, k_cache, v_cache, page, tables, torch.arange(count + 1, dtype=torch.int32, device="cuda"), kv, 1, page, 0.25, None, True, workspace,
                              uneven=True)
    assert ("attention_arrivals" in workspace.addresses()) == (items == 65535)
    scores = (0.25 * q @ k_cache[1, 0].T).masked_fill(torch.arange(page, device="cuda") >= kv[:, None], float("-inf"))
    torch.testing.assert_close(got, scores.softmax(-1) @ v_cache[1, 0].T, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("m,n,k", [(17, 16384, 64), (32, 16388, 448), (33, 24580, 256), (64, 32700, 192)])
def test_a_head_of_some_rows_streams_its_packed_copy(ops, m, n, k):
    """Float32 results of 17 to 64 rows of a registered weight: products of bfloat16 numbers, exact in float32, and k additions."""
    x, w = rand((m, k), torch.bfloat16, 63), rand((n, k), torch.bfloat16, 64)
    got = ops.linear(x, ops.prepare_weight(w), None, torch.float32)
    assert got.shape == (m, n) and got.dtype == torch.float32 and got.is_contiguous()
    want = x.double() @ w.double().T
    assert torch.all((got.double() - want).abs() <= k * 2.0 ** -23 * (x.double().abs() @ w.double().abs().T) + 1e-30)
    assert torch.equal(got, ops.skinny_gemm_splitk(x, w, splits=1, packed=ops.pack_rows(w))[0])


@pytest.mark.parametrize("n,k", [(7, 260), (4094, 36), (4099, 512), (120001, 8), (30002, 300)])
def test_gemm_fma_of_few_rows_in_every_shape(ops, n, k):
    """Two, four and eight rows of W a wave, numbers of rows of A between those that are built: a product's bits are those of each of its rows
    alone, whose sums are k products and additions in float32."""
    x, w, bias = rand((16, k), torch.float32, 60), rand((n, k), torch.float32, 61), rand((n,), torch.float32, 62)
    whole = ops.gemm_fma(x, w, bias, torch.float32)
    bound = (k + 8) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T + bias.double().abs())
    assert torch.all((whole.double() - (x.double() @ w.double().T + bias.double())).abs() <= bound)
    for m in (1, 2, 3, 4, 5, 7, 8, 9, 12, 13):
        assert torch.equal(ops.gemm_fma(x[:m].contiguous(), w, bias, torch.float32), whole[:m])


@pytest.mark.parametrize("m,n,k", [(1, 512, 64), (1, 520, 8960), (4, 1536, 1536), (2, 1540, 8960), (3, 2048, 192), (1, 2048, 20480), (4, 512, 5120), (1, 768, 11008)])
def test_a_few_rows_into_the_residual(ops, ref, m, n, k):
    """The product of up to four rows with a narrow weight: the smallest and longest sums it takes, odd numbers of blocks of 64 indices, waves
    without any, outputs that end inside a tile."""
    from velox_amd.parts.base import ResidualSink
    from velox_amd.parts.norms import RMSNorm

    assert ops._few_rows_pieces(m, k) <= 10
    x, w = rand((m, k), torch.bfloat16, 40), rand((n, k), torch.bfloat16, 41, 0.05)
    norm = RMSNorm("", n, 1e-5)
    norm.weight = 1.0 + rand((n,), torch.float32, 42, 0.1)
    residual0 = rand((m, n), torch.float32, 43)
    residual, other = residual0.clone(), residual0.clone()
    deferred = ops.linear(x, ops.prepare_weight(w), None, torch.bfloat16, partials_ok=True, residual_norm=ResidualSink(residual, norm))
    assert deferred.sums.shape == (16, 2 * ((n + 15) // 16))
    want = residual0.double() + x.double() @ w.double().T
    # products of bfloat16 numbers are exact in float32; k additions, rounded down or to nearest
    assert torch.all((residual.double() - want).abs() <= k * 2.0 ** -23 * (x.double().abs() @ w.double().abs().T + residual0.abs()))
    assert torch.equal(deferred.x, (residual * norm.weight).to(torch.bfloat16))
    torch.testing.assert_close(deferred.sums[:m].sum(1), (residual * residual).sum(1), rtol=1e-5, atol=0)
    ops._linear_into_residual(x, ops.prepare_weight(w), ResidualSink(other, norm), row_tiles=1)
    torch.testing.assert_close(residual, other, rtol=1e-5, atol=1e-5 * float(want.abs().max()))


@pytest.mark.parametrize("m", [1, 2, 3, 4])
@pytest.mark.parametrize("nh,nkv,d,k,page", [(4, 2, 64, 128, 4), (12, 2, 128, 1536, 16), (5, 2, 96, 192, 1), (28, 2, 128, 1088, 8), (16, 4, 32, 64, 16)])
@pytest.mark.parametrize("use_bias", [True, False])
def test_qkv_projection_of_a_few_rows_in_halves_of_its_tiles(ops, m, nh, nkv, d, k, page, use_bias):
    """Against the kernel for up to 16 rows (``waves=8`` asks for it), with plain rows and with rows whose norm is still to be taken: the same
    sums of exact products in another order of additions, rounded to bfloat16 once."""
    from velox_amd.parts.base import ResidualSink
    from velox_amd.parts.norms import RMSNorm

    width, half = (nh + 2 * nkv) * d, d // 2
    assert 512 <= width <= 16 * ops.num_cus and (ops._few_rows_pieces(m, k) <= 2 or m > 2)  # (three and four rows of the longer sums stay)
    w, bias = ops.prepare_weight(rand((width, k), torch.bfloat16, 71, 0.05), rotary_heads=(nh, nkv, d)), rand((width,), torch.float32, 72) if use_bias else None
    angles = torch.outer(torch.arange(64, dtype=torch.float32), 1.0 / (10000.0 ** (torch.arange(half, dtype=torch.float32) / half)))
    cos, sin = angles.cos().cuda(), angles.sin().cuda()
    positions, slots = torch.tensor([9, 0, 63, 5][:m], dtype=torch.int32).cuda(), torch.tensor([page, 3 * page - 1, 4 * page, 2 * page][:m], dtype=torch.int32).cuda()
    norm = RMSNorm("", k, 1e-6)
    norm.weight = 1.0 + rand((k,), torch.float32, 73, 0.1)
    rows = rand((m, k), torch.bfloat16, 74)
    deferred = ops.linear(rand((m, 256), torch.bfloat16, 75), ops.prepare_weight(rand((k, 256), torch.bfloat16, 76, 0.1)), None, torch.bfloat16,
                          residual_norm=ResidualSink(rand((m, k), torch.float32, 77), norm))
    for x in (rows, deferred):
        results = []
        for more in ({}, {"waves": 8}):
            k_cache, v_cache = torch.full((5, nkv, page, d), 7.0, dtype=torch.bfloat16, device="cuda"), torch.full((5, nkv, d, page), 7.0, dtype=torch.bfloat16, device="cuda")
            results.append((ops.qkv_rope_write(x, w, bias, nh, nkv, d, positions, cos, sin, slots, k_cache, v_cache, page, **more), k_cache, v_cache))
        for got, want in zip(*results):
            scale = float(want.float().abs().max())
            torch.testing.assert_close(got.float(), want.float(), rtol=2.0 ** -7, atol=k * 2.0 ** -22 * scale)


@pytest.mark.parametrize("nh,nkv,d,n,lens", [(12, 2, 128, 1536, [391]), (12, 2, 128, 1536, [1000, 3]), (28, 4, 128, 3584, [2048]), (14, 2, 64, 896, [100, 70, 128, 1]), (12, 2, 48, 512, [65])])
def test_parts_of_an_attention_that_the_output_product_merges(ops, ref, nh, nkv, d, n, lens):
    from velox_amd.engine.batch import Workspace
    from velox_amd.kernels.hip_ops import KernelError
    from velox_amd.parts.base import AttentionParts, ResidualSink
    from velox_amd.parts.norms import RMSNorm

    case = _attention_case(torch.bfloat16, nh, nkv, d, 16, [(1, length) for length in lens], seed=3)
    weight = ops.prepare_weight(rand((n, nh * d), torch.bfloat16, 44, 0.05))
    norm = RMSNorm("", n, 1e-5)
    norm.weight = torch.ones(n, device="cuda")
    workspace, m = Workspace(torch.device("cuda")), len(lens)

    def product(**more):
        residual = torch.zeros((m, n), device="cuda")
        sink = ResidualSink(residual, norm)
        parts = ops.attention_parts(m, nh, nkv, d, weight, sink, max(lens)) or 8  # (two pieces also where one pass is quicker)
        attention = ops.paged_attention(case["qkv"], nh, nkv, d, case["k_cache"], case["v_cache"], 16, case["tables"], case["cu"], case["kv"], 1, max(lens),
                                        1.0 / math.sqrt(d), None, True, workspace, **(more or {"parts": parts}))
        assert parts in (2, 4, 8) and isinstance(attention, AttentionParts) == (not more)
        ops.linear(attention, weight, None, torch.bfloat16, residual_norm=sink)
        return residual

    got, whole = product(), product(splits=1)
    # (either rounds the attention's output to bfloat16 once; a wave's running maximum takes other steps)
    assert float((got - whole).norm() / whole.norm()) < 2.0 ** -8
    case["kv"].fill_(1)  # behind one key the other parts are empty
    assert float((product() - product(splits=1)).norm()) <= 1e-4 * float(whole.norm())
    with pytest.raises(KernelError):
        ops.linear(AttentionParts(torch.zeros(8, device="cuda"), torch.zeros(8, device="cuda"), 1, m, nh, d), weight, None, torch.bfloat16)


def test_far_key_among_hundreds_is_found(ops):
    # one key far back matches the query strongly: the output must be (nearly) that key's value
    nh, nkv, d, page = 4, 2, 64, 16
    seqs = [(1, 900)]
    case = _attention_case(torch.float32, nh, nkv, d, page, seqs, seed=5)
    target = 37
    tables = case["tables"].cpu()
    q = case["qkv"][0, : nh * d].view(nh, d)
    p, o = int(tables[0, target // page]), target % page
    for h in range(nh):
        case["k_cache"][p, h // 2, o, :] = 0
    case["k_cache"][p, 0, o, :] = 4.0 * (q[0] + q[1]) / 2
    case["k_cache"][p, 1, o, :] = 4.0 * (q[2] + q[3]) / 2
    out = _run_attention(ops, case, nh, nkv, d, page).view(nh, d)
    want = _run_attention(TorchOps(), case, nh, nkv, d, page).view(nh, d)
    torch.testing.assert_close(out, want, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("rows,vocab", [(1, 152064), (8, 151936), (64, 32003), (3, 5000), (300, 4099), (2, 2047)])
def test_argmax_over_chunks_of_the_vocabulary(ops, ref, rows, vocab):
    logits = rand((rows, vocab), torch.float32, 31, 3.0)
    torch.testing.assert_close(ops.argmax(logits), ref.argmax(logits))
    # ties across chunks: the first index wins; a maximum in the last, shorter chunk is found
    logits[0, vocab // 3] = logits[0, vocab - 5] = 60.0
    logits[rows - 1, vocab - 1] = 70.0
    got = ops.argmax(logits)
    assert int(got[rows - 1]) == vocab - 1 and (rows == 1 or int(got[0]) == vocab // 3)
    # an unaligned row start (a slice of a wider tensor)
    wide = rand((rows, vocab + 3), torch.float32, 32, 3.0)
    if (vocab + 3) % 4 == 0:
        torch.testing.assert_close(ops.argmax(wide[:, :vocab].contiguous()), ref.argmax(wide[:, :vocab]))


def test_argmax_and_sampling(ops, ref):
    vocab = 1003
    logits = rand((6, vocab), torch.float32, 30, 3.0)
    logits[2, 77] = logits[2, 900] = 50.0  # a tie: the first index wins
    torch.testing.assert_close(ops.argmax(logits), ref.argmax(logits))
    assert int(ops.argmax(logits)[2]) == 77

    options = np.zeros((6, 6), dtype=np.int32)
    f = options.view(np.float32)
    rows = [(0.0, 1.0, 0), (0.8, 1.0, 0), (1.0, 0.9, 0), (1.3, 1.0, 5), (0.7, 0.5, 50), (1.0, 1.0, 1)]
    for r, (temp, top_p, top_k) in enumerate(rows):
        f[r, 0], f[r, 1] = temp, top_p
        options[r, 2:] = (top_k, 1234 + r, 99, r)
    got = ops.sample(logits, torch.from_numpy(options).cuda()).cpu().numpy()
    for r in range(6):
        token, scores = TorchOps.sample_row(logits[r].cpu().numpy(), options[r])
        assert np.isfinite(scores[got[r]]), f"row {r}: token {got[r]} was filtered out"
        assert scores[got[r]] >= scores.max() - 1e-3, f"row {r}: token {got[r]} score {scores[got[r]]} vs best {scores.max()} ({token})"
    assert got[0] == int(logits[0].argmax())
    assert got[5] == int(logits[5].argmax())  # top_k = 1 is greedy


@pytest.mark.parametrize("vocab,spread", [(152064, 1.2), (151936 + 3, 4.0), (320, 2.0), (4099, 0.3)])
def test_sampling_keeps_exactly_the_tokens_the_filters_allow(ops, vocab, spread):
    """The threshold of top-k / top-p at the real vocabulary size, flat and peaked rows, ties across the threshold: over many
    draws per row, every drawn token is one the plain filter keeps, and the tokens at the filter's edge (the last kept ones)
    are drawn as well, so the kept set is neither too small nor too large.  A row's draw does not depend on its place."""
    settings = [(0.8, 0.9, 0), (1.0, 1.0, 7), (0.7, 0.5, 50), (1.3, 0.95, 1000), (1.0, 0.999, 0), (0.5, 0.3, 3), (1.0, 1.0, 0), (2.0, 0.6, 20000),
                (1.0, 1e-20, 0), (1.0, 1.0, 2)]  # a share of the mass so small that it rounds to nothing: the best token is still kept
    base = rand((len(settings), vocab), torch.float32, 77, spread)
    base[2, 5] = base[2, 11] = base[2, vocab - 1] = float(base[2].max()) + 0.5  # three equal tokens at the top
    base[5, :40] = float(base[5].max())  # forty equal tokens: rank 0 for all of them, so top_k = 3 keeps all forty
    base[9, 3], base[9, 8], base[9, 100], base[9, vocab - 2] = (float(base[9].max()) + x for x in (1.0, 0.5, 0.5, 0.5))  # top_k = 2 with three tokens tied at the cut
    draws = 300
    logits = base.repeat_interleave(draws, 0).contiguous()
    options = np.zeros((len(settings) * draws, 6), dtype=np.int32)
    f = options.view(np.float32)
    for r, (temp, top_p, top_k) in enumerate(settings):
        rows = slice(r * draws, (r + 1) * draws)
        f[rows, 0], f[rows, 1] = temp, top_p
        options[rows, 2] = top_k if 0 < top_k < vocab else 0
        options[rows, 3], options[rows, 4] = 4242 + r, 17
        options[rows, 5] = np.arange(draws)
    got = ops.sample(logits, torch.from_numpy(options).cuda()).cpu().numpy()
    for r, (temp, top_p, top_k) in enumerate(settings):
        _, scores = TorchOps.sample_row(base[r].cpu().numpy(), options[r * draws])
        kept = np.isfinite(scores)
        drawn = got[r * draws:(r + 1) * draws]
        assert kept[drawn].all(), f"row {r}: tokens {sorted(set(drawn[~kept[drawn]]))} were drawn but are filtered out"
        if kept.sum() <= 50:
            # few tokens are kept: 300 draws at these temperatures reach every one of them, the edge of the filter included
            x = base[r].cpu().numpy().astype(np.float64)
            share = np.where(kept, np.exp((x - x.max()) / temp), 0.0)
            probable = share / share.sum() > 0.04  # (missed by 300 draws with probability below 1e-5)
            assert set(np.flatnonzero(probable)) <= set(drawn), f"row {r}: kept tokens {sorted(set(np.flatnonzero(probable)) - set(drawn))} never drawn"
        # each draw is the best score among the kept tokens, with the generator's noise for its own counter
        for j in (0, 1, draws - 1):
            token, scores = TorchOps.sample_row(base[r].cpu().numpy(), options[r * draws + j])
            assert scores[drawn[j]] >= scores.max() - 1e-3, (r, j, int(drawn[j]), token)
    # stated without the plain filter: a share of the mass of nothing keeps the one best token, and a cut of top-k that falls
    # into a run of equal logits keeps the whole run (the reference keeps exactly k by sorted position, engine/sampler.py:218-221)
    assert set(got[8 * draws:9 * draws]) == {int(base[8].argmax())}
    assert set(got[9 * draws:10 * draws]) == {3, 8, 100, vocab - 2}
    # the same rows in another order and beside other rows: the same tokens
    order = torch.randperm(len(settings) * draws, generator=torch.Generator().manual_seed(5))[:97]
    again = ops.sample(logits[order.cuda()].contiguous(), torch.from_numpy(options[order.numpy()]).cuda()).cpu().numpy()
    assert (again == got[order.numpy()]).all()


@pytest.mark.parametrize("vocab,spread", [(152064, 1.2), (151936 + 3, 4.0), (321, 2.0), (4099, 0.3)])
def test_sampling_with_rows_cut_into_chunks_gives_the_same_tokens(ops, vocab, spread):
    """Few rows are sampled with several workgroups per row, one kernel per pass, the tables of the threshold's digits
    added up in global memory: the tokens are those of the one-workgroup kernel, bit for bit, for every number of chunks
    (chunks that end inside the last quad, chunks beyond the row's end, rows that start off a 16-byte boundary), for
    greedy rows, rows without a filter and rows with one, side by side."""
    settings = [(0.8, 0.9, 0), (1.0, 1.0, 7), (0.0, 1.0, 0), (0.7, 0.5, 50), (1.3, 0.95, 1000), (1.0, 0.999, 0), (0.5, 0.3, 3), (1.0, 1.0, 0), (2.0, 0.6, 20000),
                (1.0, 1e-20, 0)]
    base = rand((len(settings), vocab), torch.float32, 78, spread)
    base[3, 5] = base[3, 11] = base[3, vocab - 1] = float(base[3].max()) + 0.5
    base[6, :40] = float(base[6].max())
    base[2, 17] = base[2, vocab - 2] = float(base[2].max()) + 1.0  # a tie in the greedy row, in different chunks: the first wins
    draws = 5
    logits = base.repeat_interleave(draws, 0).contiguous()
    options = np.zeros((len(settings) * draws, 6), dtype=np.int32)
    f = options.view(np.float32)
    for r, (temp, top_p, top_k) in enumerate(settings):
        rows = slice(r * draws, (r + 1) * draws)
        f[rows, 0], f[rows, 1] = temp, top_p
        options[rows, 2] = top_k if 0 < top_k < vocab else 0
        options[rows, 3], options[rows, 4] = 999 + r, 3
        options[rows, 5] = np.arange(draws)
    device_options = torch.from_numpy(options).cuda()
    whole = ops.sample(logits, device_options, chunks=1).cpu().numpy()
    assert whole[2 * draws] == 17
    assert set(whole[9 * draws:10 * draws]) == {int(base[9].argmax())}  # top_p of nothing: the best token, not an id outside the vocabulary
    for chunks in (None, 2, 3, 7, 16, 64):
        got = ops.sample(logits, device_options, chunks=chunks).cpu().numpy()
        assert (got == whole).all(), (chunks, np.flatnonzero(got != whole)[:10], got[got != whole][:10], whole[got != whole][:10])
    # no row with a filter: the kernels of the digits are left out
    plain = [r for r, (temp, top_p, top_k) in enumerate(settings) if temp == 0.0 or (top_p >= 1.0 and top_k == 0)]
    pick = torch.tensor([r * draws + j for r in plain for j in range(draws)])
    got = ops.sample(logits[pick.cuda()].contiguous(), device_options[pick.cuda()].contiguous(), with_filter=False, chunks=5).cpu().numpy()
    assert (got == whole[pick.numpy()]).all()
    # a broken promise gives no token rather than one from the wrong set
    broken = ops.sample(logits, device_options, with_filter=False, chunks=5).cpu().numpy()
    has_filter = np.array([temp != 0.0 and (top_p < 1.0 or 0 < top_k < vocab) for temp, top_p, top_k in settings]).repeat(draws)
    assert (broken[has_filter] == -1).all() and (broken[~has_filter] == whole[~has_filter]).all()


@pytest.mark.parametrize("vocab", [16384, 16389, 40000])
@pytest.mark.parametrize("top_p, top_k", [(0.9, 0), (1.0, 40), (0.8, 300)])
def test_sampling_with_as_many_tokens_left_as_a_list_holds(ops, vocab, top_p, top_k):
    """Two chunks of 2,048 quads and more hand the tokens that the first digit leaves over from kernel to kernel, at most 256 a wave: rows
    that leave a wave (quads 0 .. 63, then 1,024 .. 1,087 of the first chunk) one less, as many and one more, or none.  The one-workgroup
    kernel has no lists: the same tokens, bit for bit."""
    wave = [i for i in range(vocab // 2 - 8) if i // 4 % 1024 < 64]
    logits = rand((4 * 6, vocab), torch.float32, 5, 0.5) - 30.0
    for r in range(logits.shape[0]):
        left = wave[:(255, 256, 257, 0)[r % 4]]
        logits[r, left] = 4.0 + 0.9 * torch.rand(len(left), generator=torch.Generator().manual_seed(r)).to(logits)
        logits[r, vocab - 1 - r] = 4.5
    options = np.zeros((logits.shape[0], 6), dtype=np.int32)
    options.view(np.float32)[:, 0], options.view(np.float32)[:, 1] = 1.0, top_p
    options[:, 2], options[:, 3] = top_k, np.arange(logits.shape[0])
    options = torch.from_numpy(options).cuda()
    assert torch.equal(ops.sample(logits, options, chunks=2), ops.sample(logits, options, chunks=1))


@pytest.mark.parametrize("vocab, chunks", [(40000, 3), (152064, 4), (9001, 32)])
@pytest.mark.parametrize("top_p, top_k", [(0.9, 0), (1.0, 900), (0.3, 0), (1.0, 15000)])
def test_sampling_with_lists_and_open_tokens_beyond_their_room(ops, vocab, chunks, top_p, top_k):
    """Rows with more listed tokens (6,144) and more kept ones (3,072) than LDS holds, rows of which only some chunks are listed, and, in rows
    that are not listed, 1,023 to 1,025 and far more equal logits around the threshold: the tokens of the one-workgroup kernel, bit for bit."""
    g = torch.Generator().manual_seed(9)
    logits = torch.full((8, vocab), -30.0) - torch.rand((8, vocab), generator=g)
    logits[0, torch.randperm(vocab, generator=g)[:vocab // 10]] = 4.2
    spread = torch.randperm(vocab, generator=g)[:vocab // 10]
    logits[1, spread] = 4.0 + 0.9 * torch.rand(len(spread), generator=g)
    for r, equal in enumerate((1023, 1024, 1025, 16000, vocab), start=2):
        if r < 6:
            logits[r, :vocab // 2] = 3.6 + 0.3 * torch.rand(vocab // 2, generator=g)  # (the other half's chunks are listed)
        logits[r, torch.randperm(vocab, generator=g)[:equal]] = 3.75
    logits[7] = 1.0 + 0.2 * torch.rand(vocab, generator=g)
    logits = logits.repeat_interleave(3, 0).cuda()
    options = np.zeros((logits.shape[0], 6), dtype=np.int32)
    options.view(np.float32)[:, 0], options.view(np.float32)[:, 1] = 1.0, top_p
    options[:, 2], options[:, 3] = top_k if top_k < vocab else 0, np.arange(logits.shape[0])
    options = torch.from_numpy(options).cuda()
    whole = ops.sample(logits, options, chunks=1)
    for _ in range(2):
        assert torch.equal(ops.sample(logits, options, chunks=chunks), whole)


@pytest.mark.parametrize("vocab, chunks", [(40000, 2), (40000, 3), (152064, 18), (9001, 32)])
@pytest.mark.parametrize("top_p, top_k", [(0.9, 0), (1.0, 40), (1.0, 6000)])
def test_sampling_with_as_many_tokens_left_as_one_workgroup_takes(ops, vocab, chunks, top_p, top_k):
    """A chunk's share of the 6,144 tokens that one workgroup finishes a row with: chunks that leave one less, as many and one more, in one chunk of
    the row and in all; spread over a chunk's waves, or in one wave's quads alone; scores of zero with either sign.  The tokens of the
    one-workgroup kernel, bit for bit."""
    g = torch.Generator().manual_seed(vocab + chunks)
    share, per_chunk = 6144 // chunks, 4 * (((vocab + 3) // 4 + chunks - 1) // chunks)
    logits = torch.full((16, vocab), -30.0) - torch.rand((16, vocab), generator=g)
    for r, (more, everywhere) in enumerate(itertools.product((-1, 0, 1, 40, 4000), (False, True))):
        for c in range(chunks if everywhere else 1):
            room = torch.arange(c * per_chunk, min((c + 1) * per_chunk, vocab))
            left = room[torch.randperm(len(room), generator=g)[:share + more]] if r % 4 else room[:share + more]
            logits[r, left] = 4.0 + 0.9 * torch.rand(len(left), generator=g)
    logits[10], logits[11], logits[12] = 0.0, -0.0, torch.where(torch.rand(vocab, generator=g) < 0.5, 0.0, -0.0)
    logits[13, ::2], logits[14], logits[15] = float("-inf"), 1.2 * torch.randn(vocab, generator=g), 0.3 * torch.randn(vocab, generator=g).bfloat16().float()
    logits = logits.repeat_interleave(2, 0).cuda()
    options = np.zeros((logits.shape[0], 6), dtype=np.int32)
    options.view(np.float32)[:, 0], options.view(np.float32)[:, 1] = 1.0, top_p
    options[:, 2], options[:, 3] = top_k, np.arange(logits.shape[0])
    options = torch.from_numpy(options).cuda()
    assert torch.equal(ops.sample(logits, options, chunks=chunks), ops.sample(logits, options, chunks=1))


@pytest.mark.parametrize("kind, top_p, top_k", [("equal", 1.0, 2000), ("masked", 1.0, 2000), ("wide", 0.9, 0), ("wide", 1.0, 20000)])
def test_rows_in_chunks_are_worked_on_by_all_of_their_workgroups(ops, kind, top_p, top_k):
    """Eight rows of 152,064 whose threshold many tokens share (equal logits; all but 100 masked to -inf and a larger top-k) or that leave tens of thousands
    over: 18 workgroups a row take well below half of one workgroup's time (a tenth to a third; one of the 18 alone would take two thirds and more)."""
    from velox_amd.kernels.measure import time_in_graph

    g = torch.Generator().manual_seed(2)
    rows, vocab = 8, 152064
    logits = {"equal": torch.ones((rows, vocab)), "wide": 1.5 * torch.randn((rows, vocab), generator=g), "masked": torch.full((rows, vocab), float("-inf"))}[kind]
    if kind == "masked":
        logits[:, torch.randperm(vocab, generator=g)[:100]] = torch.randn((rows, 100), generator=g)
    logits = logits.cuda()
    options = np.zeros((rows, 6), dtype=np.int32)
    options.view(np.float32)[:, 0], options.view(np.float32)[:, 1] = 0.8, top_p
    options[:, 2], options[:, 3] = top_k, np.arange(rows)
    options = torch.from_numpy(options).cuda()
    one, many = (time_in_graph(lambda: ops.sample(logits, options, chunks=chunks)) for chunks in (1, 18))
    assert many < 0.5 * one, (many, one)


def test_penalties_over_long_histories_and_a_large_vocabulary(ops, ref):
    vocab, rows, width = 152064, 4, 6000
    logits = rand((rows, vocab), torch.float32, 34, 2.0)
    g = torch.Generator().manual_seed(35)
    tokens = torch.randint(0, vocab, (rows, width), generator=g).to(torch.int32)
    tokens[1, :3000] = torch.randint(8000, 8200, (3000,), generator=g).to(torch.int32)  # many repeats inside one range of the table
    tokens[2, :] = 151000  # one token, 6000 times
    tokens = tokens.cuda()
    lengths = torch.tensor([6000, 3500, 6000, 1], dtype=torch.int32).cuda()
    coeffs = torch.tensor([[1.3, 0.5, 0.2], [2.0, 1.0, 0.01], [0.8, 0.0, 0.001], [1.1, 0.2, 0.3]], dtype=torch.float32).cuda()
    got, want = logits.clone(), logits.clone()
    ops.apply_penalties(got, tokens, lengths, coeffs)
    ref.apply_penalties(want, tokens, lengths, coeffs)
    torch.testing.assert_close(got, want, rtol=1e-6, atol=1e-6)
    assert int((got != logits).sum()) > 5000
    again = logits.clone()
    ops.apply_penalties(again, tokens, lengths, coeffs)
    assert torch.equal(again, got)


def test_penalties_from_a_table_of_counts_kept_on_the_device(ops, ref):
    """The table of counts is built from a request's tokens, grows by the sampler's tokens, and penalises the rows that
    point into it exactly as the history-walking kernel does with the same tokens; rows that point nowhere keep their logits."""
    vocab, rows = 152064, 5
    logits = rand((rows, vocab), torch.float32, 36, 2.0)
    g = torch.Generator().manual_seed(37)
    histories = [torch.randint(0, vocab, (n,), generator=g).to(torch.int32) for n in (6000, 1, 3500, 0, 777)]
    histories[2][:3000] = torch.randint(8000, 8200, (3000,), generator=g).to(torch.int32)
    histories[0][:500] = 151000
    counts = torch.zeros((8, vocab), dtype=torch.int32, device="cuda")
    place = [6, 0, 3, -1, 2]  # row 3 has no penalties; the table's rows are in no particular order
    for h, at in zip(histories, place):
        if at >= 0 and h.numel():
            ops.count_tokens(counts[at], h.cuda())
    new_tokens = torch.tensor([151000, 17, 8100, 5, vocab - 1], dtype=torch.int32)
    row_of = torch.tensor(place, dtype=torch.int32).cuda()
    ops.count_sampled(counts, row_of, new_tokens.cuda())
    coeffs = torch.tensor([[1.3, 0.5, 0.2], [2.0, 1.0, 0.01], [0.8, 0.0, 0.001], [1.7, 0.3, 0.3], [1.1, 0.2, 0.3]], dtype=torch.float32).cuda()
    got = logits.clone()
    ops.apply_penalties_from_counts(got, counts, row_of, coeffs)
    # the same through the history-walking kernel and through the plain formula
    width = 6001
    tokens = torch.zeros((rows, width), dtype=torch.int32)
    lengths = torch.zeros(rows, dtype=torch.int32)
    for r, (h, at) in enumerate(zip(histories, place)):
        if at < 0:
            continue
        whole = torch.cat([h, new_tokens[r:r + 1]])
        tokens[r, : whole.numel()] = whole
        lengths[r] = whole.numel()
    walked, want = logits.clone(), logits.clone()
    ops.apply_penalties(walked, tokens.cuda(), lengths.cuda(), coeffs)
    ref.apply_penalties(want, tokens.cuda(), lengths.cuda(), coeffs)
    assert torch.equal(got, walked)
    torch.testing.assert_close(got, want, rtol=1e-6, atol=1e-6)
    assert torch.equal(got[3], logits[3]) and int((got != logits).sum()) > 6000
    assert int(counts[6, 151000]) == 501 + int((histories[0][500:] == 151000).sum()) and int(counts.sum()) == sum(h.numel() for h, at in zip(histories, place) if at >= 0) + 4


def test_sampling_follows_the_distribution(ops):
    vocab = 50
    logits = rand((1, vocab), torch.float32, 31, 1.5).repeat(4000, 1).contiguous()
    options = np.zeros((4000, 6), dtype=np.int32)
    options.view(np.float32)[:, 0] = 0.9
    options.view(np.float32)[:, 1] = 1.0
    options[:, 3] = 7
    options[:, 5] = np.arange(4000)
    got = ops.sample(logits, torch.from_numpy(options).cuda()).cpu().numpy()
    probs = torch.softmax(logits[0].cpu() / 0.9, -1).numpy()
    counts = np.bincount(got, minlength=vocab)
    expected = probs * 4000
    keep = expected > 5
    chi2 = (((counts - expected) ** 2) / expected)[keep].sum()
    assert chi2 < 2.0 * keep.sum() + 30, f"chi-square {chi2} over {keep.sum()} bins"


def test_penalties(ops, ref):
    vocab, rows, width = 333, 3, 40
    logits = rand((rows, vocab), torch.float32, 32, 2.0)
    tokens = torch.randint(0, 60, (rows, width), generator=torch.Generator().manual_seed(33)).to(torch.int32).cuda()
    lengths = torch.tensor([40, 0, 17], dtype=torch.int32).cuda()
    coeffs = torch.tensor([[1.3, 0.5, 0.2], [2.0, 1.0, 1.0], [0.8, 0.0, 0.7]], dtype=torch.float32).cuda()
    got, want = logits.clone(), logits.clone()
    ops.apply_penalties(got, tokens, lengths, coeffs)
    ref.apply_penalties(want, tokens, lengths, coeffs)
    torch.testing.assert_close(got, want, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k", [(1, 320, 64), (8, 3584, 3584), (16, 263, 128), (7, 4608, 3584), (17, 100, 192), (32, 1000, 256), (33, 70, 64), (64, 3584, 18944), (50, 152064 // 16, 448)])
def test_skinny_gemm(ops, ref, out_dtype, m, n, k):
    x = rand((m, k), torch.bfloat16, 40)
    w = rand((n, k), torch.bfloat16, 41, 0.05)
    bias = rand((n,), torch.float32, 42)
    want = ref.linear(x, w, None, torch.float32)
    scale = float(want.abs().max())
    for waves, row_tiles in ((None, None), (4, 1), (8, 1), (16, 1), (4, 4), (8, 4)):
        for b in (None, bias):
            got = ops.skinny_gemm(x, w, b, out_dtype, waves=waves, row_tiles=row_tiles).float()
            expect = want + (b if b is not None else 0)
            atol = 1e-4 * scale if out_dtype == torch.float32 else 1e-2 * scale
            torch.testing.assert_close(got, expect, rtol=1e-2 if out_dtype == torch.bfloat16 else 1e-4, atol=atol)
    # the weight in the order the lanes read it gives the same bits as the row-major weight
    packed = ops.pack_rows(w)
    got = ops.skinny_gemm(x, None, bias, out_dtype, packed=packed, n=n).float()  # with its own choice of waves and tiles
    torch.testing.assert_close(got, want + bias, rtol=1e-2 if out_dtype == torch.bfloat16 else 1e-4, atol=atol)
    for waves, row_tiles in ((4, 1), (16, 1), (4, 4)):
        torch.testing.assert_close(ops.skinny_gemm(x, None, bias, out_dtype, waves=waves, row_tiles=row_tiles, packed=packed, n=n),
                                   ops.skinny_gemm(x, w, bias, out_dtype, waves=waves, row_tiles=row_tiles), rtol=0, atol=0)
    # the same rows give the same bits whatever else is in the batch, as long as the batch stays in one size class
    # (up to 16, up to 32, up to 64 rows: the classes split K differently, which changes the order of the sums)
    fewer = 1 if m <= 16 else 17 if m <= 32 else 33
    if m > fewer:
        part = ops.skinny_gemm(x[:fewer].contiguous(), w, None, out_dtype)
        torch.testing.assert_close(ops.skinny_gemm(x, w, None, out_dtype)[:fewer], part, rtol=0, atol=0)


def test_prepared_copies_belong_to_one_weight_and_one_version(ops, ref):
    """What ``prepare_weight`` returns is held by the caller and stands in the weight's place; a plain tensor is multiplied
    as it is (no copy is ever found through an address), and a weight changed in place behind its copies is an error, not a
    product with stale values."""
    from velox_amd.kernels.hip_ops import KernelError

    x = rand((4, 128), torch.bfloat16, 60)
    first = rand((96, 128), torch.bfloat16, 61, 0.05)
    prepared = ops.prepare_weight(first)
    assert prepared.weight is first and prepared.copy(1) is not None and prepared.copy(2) is None
    want = ref.linear(x, first, None, torch.float32)
    torch.testing.assert_close(ops.linear(x, prepared, None, torch.float32), want, rtol=1e-4, atol=1e-4)
    torch.testing.assert_close(ops.linear(x, first, None, torch.float32), want, rtol=1e-4, atol=1e-4)
    other = rand((96, 128), torch.bfloat16, 62, 0.05)
    assert ops.prepare_weight(other, stacked=2, handle=prepared).weight is other  # another weight: a new handle, not an extended one
    first.mul_(2.0)
    with pytest.raises(KernelError, match="changed in place"):
        ops.linear(x, prepared, None, torch.float32)
    again = ops.prepare_weight(first, handle=prepared)
    assert again is not prepared
    torch.testing.assert_close(ops.linear(x, again, None, torch.float32), 2 * want, rtol=1e-4, atol=1e-4)
    stacked = ops.prepare_weight(other, stacked=2)
    assert stacked.copy(2) is not None and stacked.copy(1) is None
    # what the kernels cannot read in their lanes' order stays as it is
    assert ops.prepare_weight(rand((96, 100), torch.bfloat16, 63)) is None
    assert ops.prepare_weight(rand((96, 128), torch.float32, 64)) is None


def test_a_part_refuses_a_weight_bound_again_behind_prepared_copies(ops):
    from velox_amd.parts import make_part

    ff = make_part("feed_forward", "gated_mlp", prefix="m.", hidden_size=128, intermediate_size=192)
    ff.gate_up_weight = rand((384, 128), torch.bfloat16, 65, 0.05)
    ff.down_weight = rand((128, 192), torch.bfloat16, 66, 0.05)
    assert ff.operand("down_weight") is ff.down_weight  # nothing prepared yet: the tensor itself
    ff.prepare_kernels(ops)
    assert ff.operand("down_weight").weight is ff.down_weight and ff.operand("gate_up_weight").copy(2) is not None
    ff.down_weight = ff.down_weight.clone()
    with pytest.raises(RuntimeError, match="bound again"):
        ff.operand("down_weight")
    ff.prepare_kernels(ops)
    assert ff.operand("down_weight").weight is ff.down_weight


@pytest.mark.parametrize("m,inter,k", [(1, 128, 64), (8, 18944, 3584), (16, 150, 128), (7, 1000, 192), (3, 16, 64)])
def test_skinny_gemm_with_silu_epilogue(ops, ref, m, inter, k):
    x = rand((m, k), torch.bfloat16, 50)
    w = rand((2 * inter, k), torch.bfloat16, 51, 0.05)
    gate_up = ref.linear(x, w, None, torch.float32)
    want = (torch.nn.functional.silu(gate_up[:, :inter]) * gate_up[:, inter:])
    scale = float(want.abs().max())
    for waves, pairs in ((None, None), (4, 1), (8, 1), (4, 2), (8, 2)):
        got = ops.linear_silu_mul(x, w, torch.bfloat16, waves=waves, pairs=pairs).float()
        torch.testing.assert_close(got, want, rtol=1e-2, atol=1e-2 * scale)
    packed = ops.pack_rows(w, matrices=2)
    for waves, pairs in ((None, None), (4, 1), (8, 2)):
        torch.testing.assert_close(ops.linear_silu_mul(x, w, torch.bfloat16, waves=waves, pairs=pairs, packed=packed),
                                   ops.linear_silu_mul(x, w, torch.bfloat16, waves=waves, pairs=pairs), rtol=0, atol=0)
    # larger batches take the unfused route and agree with it
    big = rand((40, k), torch.bfloat16, 52)
    torch.testing.assert_close(ops.linear_silu_mul(big, w, torch.bfloat16).float(), ref.linear_silu_mul(big, w, torch.bfloat16).float(), rtol=3e-2, atol=3e-2 * scale)


@pytest.mark.parametrize("m,inter,k", [(17, 18944, 3584), (64, 18944, 3584), (32, 150, 128), (33, 1000, 192), (40, 16, 64), (64, 81, 1600), (24, 400, 320)])
def test_gate_up_product_with_silu_epilogue_at_17_to_64_rows(ops, ref, m, inter, k):
    """A registered [Wgate; Wup] at 17 .. 64 rows: one kernel (ten waves per workgroup, five pairs of gate and up tiles)
    against the product in float32 followed by silu(gate) * up; widths that are no multiple of 16 or of 80, a K that
    is no multiple of a chunk of 256."""
    x = rand((m, k), torch.bfloat16, 53)
    w = rand((2 * inter, k), torch.bfloat16, 54, 0.05)
    gate_up = ref.linear(x, w, None, torch.float32)
    want = (torch.nn.functional.silu(gate_up[:, :inter]) * gate_up[:, inter:])
    scale = float(want.abs().max())
    unregistered = ops.linear_silu_mul(x, w, torch.bfloat16).float()  # (product + SiLU kernel)
    pw = ops.prepare_weight(w, stacked=2)
    got = ops.linear_silu_mul(x, pw, torch.bfloat16).float()
    torch.testing.assert_close(got, want, rtol=1e-2, atol=1e-2 * scale)
    torch.testing.assert_close(got, unregistered, rtol=2e-2, atol=2e-2 * scale)
    # rows of a batch do not depend on one another: the first rows alone give the same bits
    few = ops.linear_silu_mul(x[:17].contiguous(), pw, torch.bfloat16).float()
    assert torch.equal(few, got[:17])


@pytest.mark.parametrize("m,n,k", [(17, 3584, 18944), (64, 3584, 3584), (33, 100, 640), (64, 4608, 3584), (40, 260, 128), (64, 72, 1600)])
def test_skinny_gemm_splitk_and_norm_that_adds_the_partials(ops, ref, m, n, k):
    x = rand((m, k), torch.bfloat16, 60)
    w = rand((n, k), torch.bfloat16, 61, 0.05)
    want = ref.linear(x, w, None, torch.float32)
    scale = float(want.abs().max())
    for splits in (None, 1, 2, 5):
        part = ops.skinny_gemm_splitk(x, w, splits=splits)
        assert part.dim() == 3 and part.shape[1:] == (m, n) and part.dtype == torch.float32
        torch.testing.assert_close(part.sum(0), want, rtol=1e-4, atol=1e-4 * scale)
        # the weight in the order the lanes read it: the same products in the same order
        torch.testing.assert_close(ops.skinny_gemm_splitk(x, w, splits=splits, packed=ops.pack_rows(w)), part, rtol=0, atol=0)
    part = ops.skinny_gemm_splitk(x, w)
    if n % 4 == 0:
        residual = rand((m, n), torch.float32, 62)
        weight = 1 + rand((n,), torch.float32, 63, 0.02)
        r_hip, r_ref = residual.clone(), residual.clone()
        got = ops.add_rmsnorm(r_hip, part, weight, 1e-6, torch.bfloat16)
        ref_out = ref.add_rmsnorm(r_ref, part, weight, 1e-6, torch.bfloat16)
        torch.testing.assert_close(r_hip, r_ref, rtol=1e-5, atol=1e-5 * scale)
        torch.testing.assert_close(got.float(), ref_out.float(), rtol=2e-2, atol=2e-2)
        rows = torch.tensor([m - 1, 0, 3], dtype=torch.int32).cuda()
        torch.testing.assert_close(ops.add_rmsnorm_rows(r_hip, part, rows, weight, 1e-6, torch.float32),
                                   ref.add_rmsnorm_rows(r_ref, part, rows, weight, 1e-6, torch.float32), rtol=1e-4, atol=1e-4)


def test_probes_report_rates_in_the_band_of_this_card(ops):
    """The two probes that bench.py reports its fractions against: a read of 2 GiB (far more than the caches hold) streams
    at more than half and less than all of the published 8 TB/s; independent bfloat16 matrix instructions run at more than
    half and no more than the published 2.5 PFLOP/s.  A probe that measured nothing (a loop the compiler removed, a
    launch that failed) or counted its work wrongly would fall out of these bands."""
    read = ops.probe_read_bandwidth(num_bytes=(2 << 30) + 48, repeats=3)
    mfma = ops.probe_mfma_rate(iterations=20000, repeats=3)
    assert 4000.0 < read < 8000.0, read
    assert 1250.0 < mfma <= 2600.0, mfma


def test_grid_barrier_probe_ends_and_counts_every_round(ops):
    """The probe of a barrier across one workgroup per compute unit runs all its rounds (nobody gives up waiting: that
    would raise) in both forms, takes between 0.2 and 200 us per barrier, and the fenced form is the dearer one."""
    relaxed = ops.probe_grid_barrier(False, rounds=200, repeats=2)
    fenced = ops.probe_grid_barrier(True, rounds=200, repeats=2)
    assert 0.2 < relaxed < 200.0 and 0.2 < fenced < 200.0, (relaxed, fenced)
    assert fenced > relaxed, (relaxed, fenced)


def test_kernel_timer_times_a_launch_inside_a_graph(ops):
    """`velox_amd.kernels.measure` (the timings that the launch rules quote): a case of scattered pages has the shapes
    the attention entry point checks, and the timer replays a graph of launches and returns a plausible time per call."""
    import math

    from velox_amd.engine.batch import Workspace
    from velox_amd.kernels.measure import attention_case, time_in_graph

    qkv, k, v, tables, cu_q, kv_lens = attention_case(2, 96, 160, 4, 2, 64, 16)
    assert tables.shape == (2, 10) and int(tables.min()) >= 1 and len(set(tables.flatten().tolist())) == 20
    workspace = Workspace(torch.device("cuda"))
    each = time_in_graph(lambda: ops.paged_attention(qkv, 4, 2, 64, k, v, 16, tables, cu_q, kv_lens, 96, 160, 1 / math.sqrt(64), None, False, workspace),
                         launches=2, rounds=2)
    assert 1.0 < each < 5000.0, each


def test_place_tokens_puts_sampled_ids_into_a_steps_rows(ops, ref):
    from velox_amd.kernels.hip_ops import KernelError

    ids = torch.arange(100, 140, dtype=torch.int32).cuda()
    tokens = torch.tensor([7, 8, 9, 10, 11], dtype=torch.int32).cuda()
    dest = torch.tensor([3, 39, 0, 17, 99, 5], dtype=torch.int32).cuda()   # (the fifth pair points outside ids: skipped)
    source = torch.tensor([4, 0, 2, 2, 1, 77], dtype=torch.int32).cuda()   # (the sixth outside tokens: skipped)
    want = ids.clone()
    ref.place_tokens(want, dest, source, tokens, 4)
    got = ids.clone()
    ops.place_tokens(got, dest, source, tokens, 6)
    assert torch.equal(got, want) and got[3] == 11 and got[39] == 7 and got[0] == 9 and got[17] == 9 and got[5] == 105
    untouched = ids.clone()
    ops.place_tokens(untouched, dest, source, tokens, 0)
    assert torch.equal(untouched, ids)
    with pytest.raises(KernelError):
        ops.place_tokens(got, dest, source, tokens, 7)


# -- routed experts on the matrix cores: tiles of 128 or 192 rows x 256 rows of W, steps of 64 indices -------------------------
@pytest.mark.parametrize("rows, hidden, inter, top, scale_input, unit", [
    ((65,), 64, 64, 1, False, "glu"),  # one row beyond a half tile, one step
    ((64, 1, 0, 129, 127), 200, 136, 1, True, "glu"),  # a last step of fewer indices, columns beyond a tile, groups of every size
    ((128, 128, 1), 256, 264, 1, True, "relu2"),
    ((300, 70), 136, 72, 2, False, "relu2"),
    ((40, 33, 20, 200, 90), 328, 520, 2, True, "glu"),
])
def test_grouped_products_at_the_edges_of_their_tiles(ops, rows, hidden, inter, top, scale_input, unit):
    experts_against_float64(ops, rows, hidden, inter, top, scale_input, unit)


@pytest.mark.parametrize("rows, hidden, inter, top", [((700, 0, 1, 193, 192, 1153), 64, 128, 1), ((191, 2100, 385), 192, 320, 2), ((97,), 128, 64, 1)])
@pytest.mark.parametrize("scale_input", [False, True])
@pytest.mark.parametrize("unit", ["glu", "clamped", "relu2"])
def test_grouped_products_in_tiles_of_128_and_192_rows(ops, monkeypatch, rows, hidden, inter, top, scale_input, unit):
    """Empty experts, last tiles of one row and of all, more than the five tiles that are dealt out together; rows gathered through the plan and
    copied.  Each output is one chain of sums: the same bits either way."""
    monkeypatch.setattr(ops._core, "velox_routed_tile_rows", lambda *sizes: 128)
    first = experts_against_float64(ops, rows, hidden, inter, top, scale_input, unit)
    monkeypatch.setattr(ops._core, "velox_routed_tile_rows", lambda *sizes: 192)
    assert torch.equal(experts_against_float64(ops, rows, hidden, inter, top, scale_input, unit), first)


@pytest.mark.parametrize("hidden, inter", [(64, 64), (128, 24), (192, 136), (320, 64), (1088, 200)])
@pytest.mark.parametrize("scale_input, unit", [(False, "glu"), (True, "relu2")])
def test_grouped_products_of_few_rows_that_read_whole_lines(ops, hidden, inter, scale_input, unit):
    """At most 64 pairs: sums that are a multiple of 64 terms read W in whole lines, in quarters that end inside a round and with waves without
    any; outputs that end among the first or the second eight rows of a tile; one, two and four tiles of rows."""
    for rows in ((1, 0, 16), (30, 2, 1), (40, 24)):
        experts_against_float64(ops, rows, hidden, inter, 1, scale_input, unit)


@pytest.mark.parametrize("hidden, inter", [(64, 2432), (64, 3200), (64, 5120), (4864, 64), (6400, 64), (10240, 64)])
@pytest.mark.parametrize("scale_input, unit", [(False, "glu"), (True, "relu2")])
def test_grouped_products_in_tiles_of_192_and_256_columns(ops, monkeypatch, hidden, inter, scale_input, unit):
    """As many tiles as make 192 or 256 columns take fewer rounds than narrower ones, in the one product or in the other (the sizes
    above all have 128); outputs that end inside a tile, the same bits with tiles of 128 rows, which are other widths."""
    rows = (150, 200, 90, 130, 170, 100)
    monkeypatch.setattr(ops._core, "velox_routed_tile_rows", lambda *sizes: 128)
    first = experts_against_float64(ops, rows, hidden, inter, 1, scale_input, unit)
    monkeypatch.setattr(ops._core, "velox_routed_tile_rows", lambda *sizes: 192)
    assert torch.equal(experts_against_float64(ops, rows, hidden, inter, 1, scale_input, unit), first)


@pytest.mark.parametrize("rows", [(0, 700, 0, 0, 1, 0), (0, 0, 0, 0, 0, 129), (400, 1, 193, 0, 2, 64), (1, 1, 1, 1, 1, 60)])
@pytest.mark.parametrize("hidden, inter, scale_input, unit", [(64, 2432, False, "glu"), (192, 128, True, "glu"), (4864, 64, True, "relu2")])
def test_grouped_products_of_experts_that_get_very_unlike_numbers_of_rows(ops, monkeypatch, rows, hidden, inter, scale_input, unit):
    """The width of the tiles is chosen by the rows that the experts were given, not by those that they could expect."""
    monkeypatch.setattr(ops._core, "velox_routed_tile_rows", lambda *sizes: 128)
    first = experts_against_float64(ops, rows, hidden, inter, 1, scale_input, unit)
    monkeypatch.setattr(ops._core, "velox_routed_tile_rows", lambda *sizes: 192)
    assert torch.equal(experts_against_float64(ops, rows, hidden, inter, 1, scale_input, unit), first)


def experts_against_float64(ops, rows, hidden, inter, top, scale_input, unit):
    """Against float64.  Two roundings to bfloat16 (8 bits), each off by at most 2^-8 of its value: the units' middles, which the second
    product adds up (at most 2^-8 sum |W_down| |middle|), and the result.  Float32 sums of a few hundred terms add less than
    1e-5 of the same sums."""
    generator = torch.Generator(device="cuda").manual_seed(sum(rows) + hidden)
    experts, tokens = len(rows), max(sum(rows) // top, max(rows))
    drawn = lambda *shape: torch.randn(*shape, generator=generator, device="cuda")  # noqa: E731
    x = drawn(tokens, hidden).bfloat16()
    branches = 1 if unit == "relu2" else 2
    alpha, limit, shift = (1.702, 2.0, 1.0) if unit == "clamped" else (1.0, float("inf"), 0.0)
    first = (drawn(experts * branches * inter, hidden) * hidden ** -0.5).bfloat16()
    down = (drawn(experts * hidden, inter) * inter ** -0.5).bfloat16()
    weight = torch.rand(tokens, top, generator=generator, device="cuda") + 0.5
    choice = torch.full((tokens, top), experts, dtype=torch.int32, device="cuda")  # (no expert: such a pair has no row)
    at = [(t, k) for k in range(top) for t in range(tokens)]
    for e, count in enumerate(rows):
        for t, k in at[:count]:
            choice[t, k] = e
        at = at[count:]
    got = ops.routed_experts(x, choice, weight, first, down, experts, scale_input, None, torch.bfloat16, identity_experts=1, **({"ungated": unit} if unit == "relu2" else {"unit": (alpha, limit, shift)}))
    want = torch.zeros(tokens, hidden, dtype=torch.float64, device="cuda")
    spread = torch.zeros_like(want)
    for e in range(experts):
        w1, w2 = first.view(experts, -1, hidden)[e].double(), down.view(experts, hidden, inter)[e].double()
        t, k = (choice == e).nonzero(as_tuple=True)
        share = weight[t, k].double()[:, None]
        both = ((x[t].float() * share.float()).bfloat16() if scale_input else x[t]).double() @ w1.T  # (a scaled row is a bfloat16 row, as in the reference)
        if unit == "relu2":
            middle = torch.relu(both).square()
        else:
            gate, up = both[:, :inter].clamp(max=limit), both[:, inter:].clamp(-limit, limit)
            middle = gate * torch.sigmoid(alpha * gate) * (up + shift)
        want.index_add_(0, t, middle @ w2.T * (1.0 if scale_input else share))
        spread.index_add_(0, t, middle.abs() @ w2.abs().T * (1.0 if scale_input else share))
    none = choice == experts
    want += (x.double()[:, None, :] * (weight.double() * none)[:, :, None]).sum(1)
    bound = (2.0 ** -8 + 2e-5) * spread + 2.0 ** -8 * 1.01 * want.abs() + 1e-6
    assert torch.all((got.double() - want).abs() <= bound), float(((got.double() - want).abs() / bound).max())
    return got


@pytest.mark.parametrize("tokens, top, hidden, inter, unit", [(1, 2, 64, 72, "glu"), (7, 3, 328, 64, "glu"), (16, 4, 200, 136, "relu2"), (21, 3, 264, 40, "glu"), (22, 3, 264, 40, "glu"),
                                                              (90, 2, 136, 264, "relu2"), (300, 4, 520, 72, "glu")])
def test_rows_that_their_pairs_weight_scales_are_rounded_once_on_every_path(ops, tokens, top, hidden, inter, unit):
    """Up to 64 pairs are scaled where they are loaded, more are copied: the same bits as rows that were scaled beforehand (a float32
    product, one rounding).  Each token has one pair with an expert, so nothing is added up behind the products."""
    experts, branches = 6, 2 if unit == "glu" else 1
    generator = torch.Generator().manual_seed(tokens)
    x, weight = rand((tokens, hidden), torch.bfloat16, tokens), torch.rand(tokens, top, generator=generator).cuda() + 0.3
    first = rand((experts * branches * inter, hidden), torch.bfloat16, 1, hidden ** -0.5)
    down = rand((experts * hidden, inter), torch.bfloat16, 2, inter ** -0.5)
    at = torch.arange(tokens, device="cuda")
    choice = torch.full((tokens, top), experts, dtype=torch.int32, device="cuda")  # (no expert: such a pair has no row)
    choice[at, at % top] = torch.randint(0, experts, (tokens,), generator=generator).to(torch.int32).cuda()
    more = {"ungated": unit} if unit != "glu" else {}
    got = ops.routed_experts(x, choice, weight, first, down, experts, True, None, torch.bfloat16, **more)
    rows = (x.float() * weight[at, at % top][:, None]).bfloat16()
    want = ops.routed_experts(rows, choice, torch.ones_like(weight), first, down, experts, False, None, torch.bfloat16, **more)
    assert torch.equal(got, want)


@pytest.mark.parametrize("m, n, k, tile", [(17, 64, 128, "32 x 32, 2"), (33, 65, 36, None), (64, 100, 256, "32 x 32, 2"), (70, 333, 260, "32 x 32, 2"), (65, 2048, 1540, "32 x 32, 2"),
                                           (200, 2048, 516, "32 x 64, 2"), (300, 6500, 132, "32 x 64, 2"), (610, 1536, 288, "64 x 64, 2"), (1025, 4100, 196, "64 x 64, 1"),
                                           (1020, 4100, 260, "128 x 64, 1"), (616, 7004, 1540, "128 x 64, 1"), (1024, 4096, 128, "128 x 64, 1"), (640, 6565, 132, "128 x 64, 1")])
def test_float32_products_on_the_matrix_instructions(ops, m, n, k, tile):
    """Every tile and both numbers of sets of waves, remainders in all three sizes (and one sum too short for them).  A sum of at most GEMM_FOLD = 128 terms, then of as many
    such sums, all float32: off by at most (128 + k / 128 + 2) 2^-24 of the sum of the terms' sizes.  The same row in a batch of
    another size, which takes another tile, has the same bits."""
    if tile is not None:
        code = ops._core.velox_gemm_f32_tile(m, n)
        assert f"{code // 10000} x {code // 10 % 1000}, {code % 10}" == tile
    generator = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w, bias = (torch.randn(*shape, generator=generator, device="cuda") for shape in ((m, k), (n, k), (n,)))
    got = ops.gemm_fma(a, w, bias, torch.float32)
    want = a.double() @ w.double().T + bias.double()
    bound = (128 + k / 128 + 2) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T + bias.double().abs())
    assert torch.all((got.double() - want).abs() <= bound)
    assert torch.equal(ops.gemm_fma(a[-17:].contiguous(), w, bias, torch.float32), got[-17:])


@pytest.mark.parametrize("nh, nkv, page", [(32, 1, 16), (6, 2, 8), (65, 1, 32)])
@pytest.mark.parametrize("window", [None, 90])
def test_portions_of_heads_of_256_channels(ops, ref, nh, nkv, page, window):
    """Rows and keys at the edges of the 128-row and 64-key tiles, portions behind contexts, single tokens beside them."""
    seqs = [(1, 129), (4, 4), (64, 64), (5, 69), (43, 107), (130, 200), (2, 63), (33, 33)]
    case = _attention_case(torch.bfloat16, nh, nkv, 256, page, seqs, seed=nh + page)
    got = _run_attention(ops, case, nh, nkv, 256, page, window=window)
    want = _run_attention(ref, case, nh, nkv, 256, page, window=window)
    torch.testing.assert_close(got, want, rtol=2e-2, atol=2e-2)  # (the tolerance of the other bfloat16 attention tests above)


@pytest.mark.parametrize("nh, nkv, page", [(32, 1, 16), (6, 2, 8), (65, 1, 32)])
@pytest.mark.parametrize("window", [None, 90])
@pytest.mark.parametrize("splits", [1, 3])
def test_portions_of_heads_of_256_channels_have_the_general_kernels_bits(ops, nh, nkv, page, window, splits):
    """Direct loads change how keys and values reach LDS and not what is added in which order: a latent's outputs reach a router, and a
    token that stands near a tie there must not go to another expert because of the kernel its step has run."""
    from velox_amd.engine.batch import Workspace

    seqs = [(1, 129), (4, 4), (64, 64), (5, 69), (43, 107), (130, 200), (2, 63), (33, 330), (300, 777)]
    case = _attention_case(torch.bfloat16, nh, nkv, 256, page, seqs, seed=nh + page)
    case["qkv"] *= 2  # (scores that move a row's maximum now and then)
    lib = ops.attention_library(256)
    try:
        results = []
        for choice in (1, 0):
            lib.velox_attention_portion_kernel(choice)
            results.append(_run_attention(ops, case, nh, nkv, 256, page, window=window, splits=splits, workspace=Workspace(torch.device("cuda"))))
    finally:
        lib.velox_attention_portion_kernel(0)
    assert torch.equal(results[0], results[1])


@pytest.mark.parametrize("n, k", [(128, 224), (100, 96), (4, 8), (260, 72)])
@pytest.mark.parametrize("gated", [None, "output", "head"])
def test_per_head_products_in_pieces_of_four_and_one_by_one(ops, n, k, gated):
    """Rows laid out for 8-byte stores and gate loads, and the same rows two columns further on, which are written one by one: the same
    bits, nothing beside them touched, and the float32 product within one rounding of the result and, with a gate, its exponential."""
    rows, heads = 130, 5
    x, maps = rand((rows, heads * k), torch.bfloat16, n), rand((heads, n, k), torch.bfloat16, k, k ** -0.5)
    wide = n + 4
    want = torch.stack([x.float()[:, h * k:(h + 1) * k] @ maps[h].float().T for h in range(heads)], 1)
    gate = None
    if gated is not None:
        gate = rand((rows, 8 + (heads * n if gated == "output" else heads)), torch.bfloat16, 3)
        z = gate[:, 4:4 + (heads * n if gated == "output" else heads)].float().reshape(rows, heads, -1)
        want = want * torch.sigmoid(z)
    results = []
    for offset in (0, 2):
        out = torch.full((rows, heads * wide), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.head_linear(x, k, 0, maps, out, wide, offset, gate, 4 if gate is not None else 0, gated == "head")
        out = out.view(rows, heads, wide)
        results.append(out[:, :, offset:offset + n])
        assert torch.all(out[:, :, :offset] == 7.0) and torch.all(out[:, :, offset + n:] == 7.0)
    assert torch.equal(results[0], results[1])
    # bfloat16's unit roundoff is 2^-8; float32 sums of k terms of size about k^-1/2 are off by far less than 1e-4
    assert torch.all((results[0].float() - want).abs() <= 2.0 ** -8 * 1.01 * want.abs() + 1e-4)


@pytest.mark.parametrize("rows, heads, n, k", [(2049, 8, 224, 96), (513, 32, 132, 72), (130, 128, 512, 128), (8193, 2, 260, 104)])
@pytest.mark.parametrize("gated", [None, "output", "head"])
def test_per_head_products_whose_maps_stay_in_registers(ops, rows, heads, n, k, gated):
    """Remainders of the 16 rows, of a workgroup's rows, of 64 columns a wave and 32 indices: the bits of the same products in two launches of
    half of the rows and fewer, which the kernel with the rows in LDS takes."""
    x, maps = rand((rows, heads * k), torch.bfloat16, n), rand((heads, n, k), torch.bfloat16, k, k ** -0.5)
    gate = None if gated is None else rand((rows, 8 + (heads * n if gated == "output" else heads)), torch.bfloat16, 3)
    wide, few = n + 4, 16383 // heads

    def run(first, last):
        out = torch.full((last - first, heads * wide), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.head_linear(x[first:last], k, 0, maps, out, wide, 0, gate[first:last] if gate is not None else None, 4 if gate is not None else 0, gated == "head")
        return out

    whole = run(0, rows)
    assert torch.all(whole.view(rows, heads, wide)[:, :, n:] == 7.0)
    assert torch.equal(whole, torch.cat([run(at, min(rows, at + few)) for at in range(0, rows, few)]))


@pytest.mark.parametrize("tokens", [65, 512, 513, 3072, 3073])
@pytest.mark.parametrize("kv_heads, dim, heads, columns", [(3, 40, 6, 6), (8, 64, 8, 520)])
def test_what_a_recurrence_reads_does_not_depend_on_how_tokens_are_spread(ops, tokens, kv_heads, dim, heads, columns):
    """One, two and eight workgroups a token: the same bits as 40 tokens at a time."""
    main, decay = rand((tokens, 2 * kv_heads * dim + 8), torch.bfloat16, tokens), rand((tokens, columns), torch.float32, 2)
    rate, bias, beta = rand((heads,), torch.float32, 3).abs(), rand((columns,), torch.float32, 4), rand((tokens, heads), torch.bfloat16, 5)

    def prepare(rows):
        return ops.recurrence_prepare(main[rows].contiguous(), 0, kv_heads * dim, kv_heads, dim, True, 0.3, decay[rows].contiguous(), 0, heads, columns, rate, bias, 1.0, beta[rows].contiguous(), 0)

    whole = prepare(slice(0, tokens))
    for first in (0, tokens // 2, tokens - 40):
        rows = slice(first, first + 40)
        for got, want in zip(whole, prepare(rows)):
            assert torch.equal(got[rows], want)


@pytest.mark.parametrize("m, n, k, splits", [(65, 100, 5128, 1), (128, 256, 64, 1), (129, 260, 200, 2), (300, 516, 1096, 3), (1100, 300, 520, 5), (70, 1024, 72, 8)])
def test_products_in_tiles_with_a_cut_sum(ops, m, n, k, splits):
    """Against float64: remainders in all sizes, more than one block of row tiles, a last part that is short or empty.  Float32 sums of at
    most k terms in one part (an error below k 2^-24 of the sum of the terms' sizes), one rounding to bfloat16 (2^-8) for one part."""
    generator = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w = (torch.randn(*shape, generator=generator, device="cuda").bfloat16() for shape in ((m, k), (n, k)))
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    whole = ops.gemm_tiles(a, w)
    assert torch.all((whole.double() - want).abs() <= k * 2.0 ** -24 * size + 2.0 ** -8 * 1.01 * want.abs() + 1e-6)
    parts = ops.gemm_tiles(a, w, splits, torch.float32)
    assert parts.shape == (splits, m, n) and torch.all((parts.double().sum(0) - want).abs() <= k * 2.0 ** -24 * size + 1e-6)


TILES = (128128, 128192, 128256, 192192, 192256, 256192, 256256)


@pytest.mark.parametrize("m, n, k", [(1, 8, 8), (129, 260, 200), (65, 64, 64), (193, 264, 128), (257, 520, 192), (1030, 1544, 448), (3000, 6152, 320)])
def test_products_in_every_tile(ops, m, n, k):
    """Remainders in all sizes, odd numbers of steps, sums shorter than the loads are ahead, more tiles than workgroups.  Against float64 as
    above, the bias one more float32 addition; every tile has the same bits and writes nothing else."""
    generator = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w, bias = (torch.randn(*shape, generator=generator, device="cuda") for shape in ((m, k), (n, k), (n,)))
    a, w = a.bfloat16(), w.bfloat16()
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    first = None
    for tile in TILES if k % 64 == 0 else (128256, 0):
        plain = ops.gemm_tiles(a, w, tile=tile)
        biased = ops.gemm_tiles(a, w, bias=bias, tile=tile)
        parts = ops.gemm_tiles(a, w, 3, torch.float32, tile=tile)
        assert torch.all((plain.double() - want).abs() <= k * 2.0 ** -24 * size + 2.0 ** -8 * 1.01 * want.abs() + 1e-6)
        exact = want + bias.double()
        assert torch.all((biased.double() - exact).abs() <= (k + 2) * 2.0 ** -24 * (size + bias.double().abs()) + 2.0 ** -8 * 1.01 * exact.abs() + 1e-6)
        assert torch.all((parts.double().sum(0) - want).abs() <= k * 2.0 ** -24 * size + 1e-6)
        first = first or (plain, biased, parts)
        assert all(torch.equal(x, y) for x, y in zip(first, (plain, biased, parts)))
        held = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device="cuda")
        assert ops._core.velox_tiles_bf16(a.data_ptr(), w.data_ptr(), None, held.data_ptr(), m, n, k, 1, 1, tile, ops._stream()) == 0
        assert torch.equal(held[:m], plain) and torch.all(held[m] == 7.0)


@pytest.mark.parametrize("activation", ["silu", "relu"])
@pytest.mark.parametrize("m, n, k", [(65, 8, 64), (129, 132, 256), (193, 136, 128), (257, 264, 192), (1030, 776, 448), (2100, 3080, 320)])
def test_gated_products_in_every_tile(ops, m, n, k, activation):
    """The product's own bits, then the activation in float32 and one rounding: the bits of the kernel behind a product; rows with
    infinities and NaN too."""
    a, w = rand((m, k), torch.bfloat16, m), rand((2 * n, k), torch.bfloat16, n, 3 * k ** -0.5)
    a[m // 2, 3] = float("inf")
    a[m - 1, 5] = float("nan")
    product = ops.gemm_tiles(a, w)
    g, u = product[:, :n].double(), product[:, n:].double()
    want = (g * torch.sigmoid(g) if activation == "silu" else g.clamp(min=0)) * u
    behind = ops.silu_mul(product) if activation == "silu" else ops.gated_act_mul(product, activation)
    for tile in TILES:
        got = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device="cuda")
        assert ops._core.velox_tiles_glu_bf16(a.data_ptr(), w.data_ptr(), got.data_ptr(), m, n, k, 0 if activation == "silu" else 2, tile, ops._stream()) == 0
        finite = torch.isfinite(want)
        assert torch.all(got[m] == 7.0) and torch.equal(torch.isnan(got[:m]), torch.isnan(behind)) and torch.equal(torch.isinf(got[:m]), torch.isinf(behind))
        error = (got[:m].double() - want).abs() - 2.0 ** -8 * 1.01 * want.abs() - 1e-30
        assert torch.all(error[finite] <= 0) and torch.equal(got[:m][finite], behind[finite])


@pytest.mark.parametrize("m, n, k, own", [(64, 4096, 2048, False), (65, 4096, 2048, True), (300, 4608, 3584, False), (836, 37888, 3584, True), (836, 4608, 3584, True), (1036, 64, 2048, False),
                                          (768, 64, 2048, True), (769, 64, 2048, False), (2421, 128, 2048, False), (1408, 1536, 1024, False), (1409, 1536, 1024, True), (1536, 2048, 8192, False), (1793, 2048, 8192, True), (1536, 2048, 8128, True), (1036, 56, 2048, False), (1036, 4100, 2048, False), (1036, 4096, 2056, False), (1036, 4096, 192, False)])
def test_which_products_run_in_the_own_tiles(ops, monkeypatch, m, n, k, own):
    calls = []
    monkeypatch.setattr(ops, "gemm_tiles", lambda *a, **more: calls.append(a) or type(ops).gemm_tiles(ops, *a, **more))
    x, w, bias = rand((m, k), torch.bfloat16, 1), rand((n, k), torch.bfloat16, 2, k ** -0.5), rand((n,), torch.float32, 3)
    got = ops.linear(x, w, bias, torch.bfloat16)
    assert ops.tiles_serve(m, n, k) == own and len(calls) == int(own) and type(ops).library_serves(ops, m, n, k) == (m > 64 and not own)
    want = x.double() @ w.double().T + bias.double()
    assert torch.all((got.double() - want).abs() <= 2.0 ** -7 * (want.abs() + bias.double().abs()) + k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T))


@pytest.mark.parametrize("m, n, k, own", [(128, 64, 2048, False), (100, 2048, 2048, False), (200, 1536, 1024, False), (256, 768, 256, False), (128, 18432, 256, True)])
def test_products_of_recorded_steps(ops, monkeypatch, m, n, k, own):
    """What is recorded takes the library where tiles are few, and another thread's products do not.  Replays on other rows, with eager work between
    them, against float64 within a rounding of the result and the additions' own."""
    calls = []
    monkeypatch.setattr(ops, "gemm_tiles", lambda *a, **more: calls.append(a) or type(ops).gemm_tiles(ops, *a, **more))
    x, w = rand((m, k), torch.bfloat16, 1), rand((n, k), torch.bfloat16, 2, k ** -0.5)
    elsewhere = []
    with ops.recording():
        thread = threading.Thread(target=lambda: elsewhere.append(ops.tiles_serve(m, n, k)))
        thread.start()
        thread.join()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            ops.linear(x, w, None, torch.bfloat16)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with collection_held(), torch.cuda.graph(graph):
            out = ops.linear(x, w, None, torch.bfloat16)
    assert elsewhere == [True] and len(calls) == 2 * int(own)
    for seed in range(4):
        x.copy_(rand((m, k), torch.bfloat16, 10 + seed))
        graph.replay()
        torch.cuda.synchronize()
        want = x.double() @ w.double().T
        assert torch.all((out.double() - want).abs() <= 2.0 ** -8 * 1.01 * want.abs() + k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T))
        ops.linear(x, w, None, torch.bfloat16)
    assert len(calls) == 4 + 2 * int(own)


@pytest.mark.parametrize("m, n, k, in_parts", [(128, 10240, 8192, 6), (128, 7168, 5120, 8), (700, 7168, 5120, 1), (300, 4608, 3584, 0), (836, 4608, 3584, 1), (70, 2048, 2048, 1)])
def test_the_library_is_said_to_serve_what_linear_hands_to_it(ops, monkeypatch, m, n, k, in_parts):
    """With a bias, whole and in parts: a long sum over few tiles runs in the own tiles where its parts are wanted and in the library where not."""
    calls = []
    monkeypatch.setattr(ops, "gemm_tiles", lambda *a, **more: calls.append(a) or type(ops).gemm_tiles(ops, *a, **more))
    x, w, bias = rand((m, k), torch.bfloat16, 1), rand((n, k), torch.bfloat16, 2, k ** -0.5), rand((n,), torch.float32, 3)
    for given in (bias, None):
        calls.clear()
        assert ops.linear(x, w, given, torch.bfloat16).shape == (m, n)
        assert type(ops).library_serves(ops, m, n, k) == (not calls) == (in_parts != 1)
    calls.clear()
    got = ops.linear(x, w, None, torch.bfloat16, partials_ok=True)
    assert ops.own_tile_parts(m, n, k, True) == in_parts and len(calls) == (in_parts > 0) and (got.shape == (in_parts, m, n) if in_parts > 1 else got.shape == (m, n))


@pytest.mark.parametrize("m, n, k, parts", [(65, 2560, 8192, 8), (300, 2048, 8448, 8), (700, 2048, 5632, 5), (700, 1024, 28672, 8), (300, 4096, 16512, 5), (129, 8192, 16384, 4), (700, 8192, 29568, 2), (400, 12288, 29568, 2), (1280, 6144, 24576, 2)])
def test_linear_with_parts_of_a_long_sum_into_every_consumer(ops, ref, m, n, k, parts):
    """More than 64 rows of a long product come back as partial sums.  Each kernel that takes them gives what it gives for their float32
    sum (a handful of float32 additions in another order), which is the product within its own float32 sums' rounding."""
    assert ops.tile_splits(m, n, k) == parts
    parts_into_every_consumer(ops, m, n, k, parts, torch.bfloat16)


@pytest.mark.parametrize("m, n, k", [(17, 256, 512), (64, 1536, 1536), (65, 1536, 8960), (300, 2048, 1536), (616, 1536, 8960), (2400, 1024, 2048)])
def test_float32_linear_with_parts_into_every_consumer(ops, m, n, k):
    """The same in float32, where sums of 512 terms and more are cut."""
    parts = ops.split_f32_parts(m, n, k, True)
    assert parts > 1
    parts_into_every_consumer(ops, m, n, k, parts, torch.float32)


@pytest.mark.parametrize("m, n, k, whole, most", [(16, 2048, 2048, 0, 0), (17, 2048, 480, 0, 0), (17, 2048, 528, 0, 0), (17, 2046, 2048, 0, 0), (64, 17920, 1536, 0, 8), (100, 11264, 2048, 1, 8), (256, 2048, 1536, 0, 8),
                                                  (330, 2048, 1536, 1, 8), (4000, 11264, 2048, 1, 8), (33, 512, 512, 0, 8), (5000, 4096, 512, 1, 8)])
def test_float32_products_in_parts_and_whole(ops, m, n, k, whole, most):
    """Which products are worked as products of bfloat16 parts, and that no part of a sum is empty: each has whole inner sums of 128 terms but the last."""
    assert ops.split_f32_parts(m, n, k, False) == whole
    parts = ops.split_f32_parts(m, n, k, True)
    assert whole <= parts <= max(whole, most)
    if parts > 1:
        each = -(-(-(-k // 128)) // parts) * 128
        assert (parts - 1) * each < k
    x, w = rand((m, k), torch.float32, 1), rand((n, k), torch.float32, 2, k ** -0.5)
    assert ops.linear(x, w, None, torch.float32, partials_ok=True).shape == ((parts, m, n) if parts > 1 else (m, n))
    assert ops.linear(x, w, rand((n,), torch.float32, 3), torch.float32, partials_ok=True).shape == (m, n)  # (a bias belongs to a whole sum)


def parts_into_every_consumer(ops, m, n, k, parts, dtype):
    from velox_amd.parts.base import NormedSum, SumOf
    from velox_amd.parts.norms import StreamNorm

    generator = torch.Generator(device="cuda").manual_seed(m)
    x, w = torch.randn(m, k, generator=generator, device="cuda").to(dtype), (k ** -0.5 * torch.randn(n, k, generator=generator, device="cuda")).to(dtype)
    got = ops.linear(x, w, None, dtype, partials_ok=True)
    assert got.shape == (parts, m, n) and got.dtype == torch.float32
    assert ops.linear(x, w, None, dtype).shape == (m, n)  # (who cannot take parts gets none)
    whole = got.double().sum(0).float()
    for rows in (slice(0, 17), slice(m - 17, m)):
        want = x[rows].double() @ w.double().T
        assert float((whole[rows].double() - want).abs().max()) <= k * 2.0 ** -24 * float((x[rows].double().abs() @ w.double().abs().T).max())
    residual, weight = rand((m, n), torch.float32, 5), 1 + rand((n,), torch.float32, 6, 0.02)
    rows = torch.tensor([m - 1, 0, m // 2], dtype=torch.int32).cuda()
    close = dict(rtol=2e-5, atol=2e-5)
    calls = [lambda r, delta: ops.add_rmsnorm(r, delta, weight, 1e-5, torch.float32), lambda r, delta: ops.add_rmsnorm_rows(r, delta, rows, weight, 1e-5, torch.float32),
             lambda r, delta: ops.norm_add(r, delta, weight, 1e-5, 0.7, torch.float32), lambda r, delta: ops.norm_add_norm(r, delta, weight, 1e-5, weight, 1e-6, torch.float32),
             lambda r, delta: ops.add_dynamic_tanh(r, delta, weight, weight, weight[:1], torch.float32), lambda r, delta: ops.join_rows(r, delta, residual, torch.float32),
             lambda r, delta: ops.normed_sum_norm(r, NormedSum((delta, delta), (weight, weight), (0.5, 2.0), 1e-5), weight, 1e-5, torch.float32),
             lambda r, delta: ops.normed_sum_norm(r, NormedSum((delta,), (weight,), (0.5,), 1e-5, delta), weight, 1e-5, torch.float32),
             lambda r, delta: ops.add_rmsnorm(r, SumOf(delta, residual), weight, 1e-5, torch.float32)]
    for call in calls:
        a, b = residual.clone(), residual.clone()
        torch.testing.assert_close(call(a, got).float(), call(b, whole).float(), **close)
        torch.testing.assert_close(a, b, **close)

    class Context:
        dtype = torch.float32

    Context.ops = ops
    norm = StreamNorm("", n, 1e-5, streams=2, center=False)
    norm.weight = weight
    wide = torch.cat([residual, -residual], 1)
    a, b = wide.clone(), wide.clone()
    torch.testing.assert_close(norm.forward(a, got, Context), norm.forward(b, whole, Context), **close)
    torch.testing.assert_close(a, b, **close)


# (what is cut into no parts; which of these the library gets and which the own tiles take whole is tiles_serve's to say)
@pytest.mark.parametrize("m, n, k", [(128, 2048, 8448), (128, 2048, 5632), (512, 1024, 5632), (128, 1536, 8960), (128, 1024, 8192), (300, 2048, 5112), (256, 512, 16384), (400, 256, 12288), (1024, 8192, 16320), (1025, 8192, 29568),
                                     (513, 16384, 16384), (1536, 5120, 13824), (64, 3584, 18944), (4096, 3584, 18944)])
def test_products_whose_sum_is_not_cut(ops, m, n, k):
    assert ops.tile_splits(m, n, k) == 0
    assert type(ops).library_serves(ops, m, n, k) == (m > 64 and not ops.tiles_serve(m, n, k)) and ops.tiles_serve(m, n, k) == (-(-m // 128) * -(-n // 128) >= (224 if k >= 8192 else 192) and k % 64 == 0)


def test_products_whose_library_kernel_was_timed_elsewhere_stay_with_it(ops, tmp_path, monkeypatch):
    """Timings that come from a file, and products that TunableOp is about to time, are respected like those of this object; without them
    the same product takes the own tiles."""
    m, n, k = 300, 2560, 8192
    x, w = rand((m, k), torch.bfloat16, 1), rand((n, k), torch.bfloat16, 2, k ** -0.5)
    own = []
    monkeypatch.setattr(ops, "gemm_tiles", lambda *a, **more: own.append(a) or type(ops).gemm_tiles(ops, *a, **more))
    tunable = torch.cuda.tunable
    held = tunable.get_filename(), tunable.get_max_tuning_duration(), tunable.get_max_tuning_iterations()

    def calls_own():
        own.clear()
        ops.linear(x, w, None, torch.bfloat16, partials_ok=True)
        return len(own) == 1

    assert calls_own()
    try:
        tunable.set_filename(str(tmp_path / "timed.csv"))
        tunable.set_max_tuning_duration(1)
        tunable.set_max_tuning_iterations(1)
        tunable.enable(True)
        tunable.tuning_enable(False)
        assert calls_own()  # (switched on, but nothing known about this product)
        tunable.tuning_enable(True)
        assert not calls_own()  # (timed now, by the library's call)
        tunable.tuning_enable(False)
        assert not calls_own()
        assert ops.linear(x, w, None, torch.bfloat16, partials_ok=True).shape == (m, n)
    finally:
        tunable.tuning_enable(False)
        tunable.enable(False)
        tunable.set_max_tuning_duration(held[1])
        tunable.set_max_tuning_iterations(held[2])
        tunable.set_filename(held[0])
    assert calls_own()


@pytest.mark.parametrize("top_p, top_k", [(1.0, 0), (0.9, 0), (1e-6, 0), (1.0, 1), (1.0, 50), (0.5, 20)])
@pytest.mark.parametrize("temperature", [0.7, 1e-30, float("inf")])
def test_rows_with_numbers_that_are_not_finite_get_a_token_of_the_row(ops, top_p, top_k, temperature):
    """Whatever a row holds, the token lies in the vocabulary and does not depend on how the row is cut; a NaN is never drawn and, behind
    top-p, does not change the draw (its probability counts as none)."""
    vocab, inf, nan = 32773, float("inf"), float("nan")
    logits = rand((9, vocab), torch.float32, 3, 3.0)
    logits[0, 777] = inf
    logits[1, [5, 9000]] = inf
    logits[2, [333, 20000]] = nan
    logits[3] = -inf
    logits[4, 40:] = -inf
    logits[5] = torch.finfo(torch.float32).min
    logits[6] *= 1e37
    logits[7] = nan
    logits[8] = logits[2].nan_to_num(nan=-inf)
    options = np.zeros((9, 6), dtype=np.int32)
    options.view(np.float32)[:, 0], options.view(np.float32)[:, 1] = temperature, top_p
    options[:, 2], options[:, 3] = top_k, 11
    options = torch.from_numpy(options).cuda()
    whole = ops.sample(logits, options, chunks=1)
    for chunks in (2, 3, 8):
        assert torch.equal(ops.sample(logits, options, chunks=chunks), whole)
    assert torch.all((whole >= 0) & (whole < vocab))
    if top_k == 0:
        assert whole[2] == whole[8]


def test_experts_whose_weights_lie_off_16_byte_boundaries(ops):
    """More than 64 pairs then take the multiply-add tiles: the same products in another order of float32 sums, the units' middles and the
    result rounded to bfloat16 on both paths (2^-8 each, of terms that add up to a few times the result)."""
    tokens, top, experts, hidden, inter = 60, 2, 4, 72, 40
    x, weight = rand((tokens, hidden), torch.bfloat16, 1), rand((tokens, top), torch.float32, 2).abs()
    choice = torch.randint(0, experts, (tokens, top), generator=torch.Generator().manual_seed(3)).to(torch.int32).cuda()
    first, down = rand((experts * 2 * inter, hidden), torch.bfloat16, 4, hidden ** -0.5), rand((experts * hidden, inter), torch.bfloat16, 5, inter ** -0.5)

    def moved(w):
        flat = torch.empty(w.numel() + 2, dtype=w.dtype, device=w.device)
        flat[2:] = w.reshape(-1)
        return flat[2:].view(w.shape)

    want = ops.routed_experts(x, choice, weight, first, down, experts, False, None, torch.bfloat16)
    for a, b in ((moved(first), down), (first, moved(down))):
        assert (a.data_ptr() | b.data_ptr()) % 16 == 4
        torch.testing.assert_close(ops.routed_experts(x, choice, weight, a, b, experts, False, None, torch.bfloat16).float(), want.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("tile", [128256, 128192, 96192, 64256, 64128, 64064, 32128, 0])
@pytest.mark.parametrize("m, n, k, splits", [(17, 64, 32, 1), (129, 260, 160, 1), (97, 388, 672, 3), (300, 132, 4096, 8), (65, 4100, 128, 1), (33, 132, 2080, 1), (70, 64, 6176, 1)])
def test_float32_products_of_split_operands(ops, tile, m, n, k, splits):
    """Every tile, remainders of rows and columns, last sums of fewer than 128 terms, sums of more than one level.  A term's left-out products are below 2^-24 of it;
    an instruction is off by at most 2^-22 of the sizes it adds (24 of them in a sum of 128 terms, on average over half of these); each sum of
    128 terms, of 2,048, part and bias is added with a rounding: (24 + min(k / 128, 16) + k / 2048 + splits + 3) 2^-23 of the sum of the terms' sizes."""
    generator = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w, bias = (torch.randn(*shape, generator=generator, device="cuda") for shape in ((m, k), (n, k), (n,)))
    a *= 10.0 ** torch.randint(-6, 7, (m, 1), generator=generator, device="cuda")
    got = ops.split_f32(a, w, None if splits > 1 else bias, splits, tile)
    want, sizes = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    if splits > 1:
        got = got.sum(0)
    else:
        want, sizes = want + bias.double(), sizes + bias.double().abs()
    assert torch.all((got.double() - want).abs() <= (24 + min(k / 128, 16) + k / 2048 + splits + 3) * 2.0 ** -23 * sizes)
    # errors of random signs: 1.6e-7 to 1.9e-7 of a row's norm; without one of the three smallest products of parts it is 1.7e-6 at least, worked in
    # float64
    if splits > 1 or k >= 512:
        assert torch.all((got.double() - want).norm(dim=1) <= 4e-7 * want.norm(dim=1))


@pytest.mark.parametrize("tile", [128256, 128192, 96192, 64256, 64128, 64064, 32128])
@pytest.mark.parametrize("k", [128, 480])
def test_every_product_of_parts_is_there(ops, tile, k):
    """Sums in which all products of parts but one cancel exactly.  1 + 2^-9 + 2^-20 has the parts 1, 2^-9 and 2^-20; the results are exact: the rest of
    a sum is zeros."""
    from velox_amd.kernels.hip_ops import KernelError

    m, n, u, v, low = 130, 260, 2.0 ** -9, 2.0 ** -10, 2.0 ** -20
    at = 4 * torch.randint(0, k // 4, (m,), generator=torch.Generator().manual_seed(k)).cuda()
    rows = torch.arange(m, device="cuda")

    def a_of(*values):
        a = torch.zeros(m, k, device="cuda")
        for i, value in enumerate(values):
            a[rows, at + i] = value
        return a

    def w_of(*values):
        return torch.tensor(values, dtype=torch.float32, device="cuda").repeat(n, k // 4)

    with pytest.raises(KernelError):
        ops.split_f32(a_of(1, 0, 0, 0), w_of(1, 0, 0, 0).double(), tile=tile)
    cases = [(a_of(1, 0, 0, 0), w_of(1, 0, 0, 0), 1.0),  # hi hi
             (a_of(1 + u, -1, 0, 0), w_of(1, 1, 0, 0), u),  # mid hi
             (a_of(1, -1, 0, 0), w_of(1 + u, 1, 0, 0), u),  # hi mid
             (a_of(1 + u + low, -(1 + u), 0, 0), w_of(1, 1, 0, 0), low),  # lo hi
             (a_of(1, -1, 0, 0), w_of(1 + u + low, 1 + u, 0, 0), low),  # hi lo
             (a_of(1 + u, -(1 + u), -1, 1), w_of(1 + v, 1, 1 + v, 1), u * v)]  # mid mid
    for which, (a, w, want) in enumerate(cases):
        got = ops.split_f32(a, w, tile=tile)
        assert torch.all(got == want), (which, float(got.min()), float(got.max()), want)


@pytest.mark.parametrize("tile", [128256, 128192, 64064])
def test_float32_products_of_numbers_that_do_not_split(ops, tile):
    """Infinities, NaN, numbers that round to an infinity and numbers without lower parts: as the float32 instructions have them.  Those add
    in another order, so finite outcomes differ by their two roundings."""
    m, n, k = 150, 324, 288
    generator = torch.Generator(device="cuda").manual_seed(5)
    a, w = (torch.randn(*shape, generator=generator, device="cuda") for shape in ((m, k), (n, k)))
    a[3, 7], a[40, 100], a[77, 30], a[78, 31] = float("inf"), float("-inf"), float("nan"), 3.4e38
    w[100, 5], w[200, 287] = float("inf"), 0.0
    w[:, 31] *= 0.01
    a[120:130] *= 1e-36
    a[131] = 0.0
    got, want = ops.split_f32(a, w, tile=tile), ops.gemm_fma(a, w, None, torch.float32)
    assert torch.equal(got.isnan(), want.isnan())
    whole = want.isfinite()
    assert torch.equal(got[~whole & ~want.isnan()], want[~whole & ~want.isnan()])
    sizes = torch.where(a.isfinite(), a, 0).double().abs() @ torch.where(w.isfinite(), w, 0).double().abs().T
    assert torch.all(((got.double() - want.double()).abs() <= 160 * 2.0 ** -23 * sizes)[whole])
    assert torch.all(got[131][want[131].isfinite()] == 0)


@pytest.mark.parametrize("tile", [128256, 96192, 64064])
@pytest.mark.parametrize("exponent", [-44, -40, -38, -36, -34, -30])
def test_float32_products_of_tiny_and_huge_numbers(ops, tile, exponent):
    """Operands whose lower parts are far below bfloat16's smallest numbers, times large ones: as exact as any.  The sums of 512 terms of random signs
    show 1.6e-7 of their norm."""
    generator = torch.Generator(device="cuda").manual_seed(-exponent)
    tiny, huge = (torch.randn(132, 512, generator=generator, device="cuda").double() * s for s in (10.0 ** exponent, 1e20))
    tiny, huge = tiny.float(), huge.float()
    for a, w in ((tiny, huge), (huge, tiny)):
        want = a.double() @ w.double().T
        assert float((ops.split_f32(a, w, tile=tile).double() - want).norm() / want.norm()) <= 3e-7


@pytest.mark.parametrize("m, n, k, splits, tile", [(150, 324, 288, 1, 128256), (150, 324, 288, 1, 96192), (97, 132, 4192, 1, 64064), (97, 132, 2080, 3, 0)])
def test_rows_beside_numbers_that_do_not_split_keep_their_bits(ops, m, n, k, splits, tile):
    """A row with an infinity, NaN, a number near float32's end or tiny ones changes no other row."""
    a, w = rand((m, k), torch.float32, m), rand((n, k), torch.float32, n)
    strange = a.clone()
    strange[3, 7], strange[20, k - 1], strange[37, 30], strange[m - 1] = float("inf"), float("nan"), 3e38, a[m - 1] * 1e-37
    plain, got = ops.split_f32(a, w, None, splits, tile), ops.split_f32(strange, w, None, splits, tile)
    same = [r for r in range(m) if r not in (3, 20, 37, m - 1)]
    assert torch.equal(got[..., same, :], plain[..., same, :])
    last = a[m - 1:].double() * 1e-37 @ w.double().T
    whole = got.double().sum(0) if splits > 1 else got.double()
    assert float((whole[m - 1] - last[0]).norm() / last.norm()) <= 1e-6  # (the row itself, its numbers rounded once more)
    assert whole[3].isinf().any() and whole[20].isnan().all() and not whole[37].isnan().any()


@pytest.mark.parametrize("m, n, k, splits, tile", [(616, 2048, 1536, 1, 128256), (616, 1536, 8960, 1, 96192), (616, 1536, 8960, 4, 64128), (616, 2048, 1536, 1, 64064)])
def test_float32_products_of_split_operands_are_off_to_either_side(ops, m, n, k, splits, tile):
    """The instructions round down, 3e-8 of the result's norm on average at 1,536 terms and 8e-8 at 8,960 if every sum is added: inner sums of alternating
    signs leave nothing of it but the chance of 1e6 outputs (2e-10) and a last sum without a partner (one of 12 here at most)."""
    a, w = rand((m, k), torch.float32, m), rand((n, k), torch.float32, n)
    got, want = ops.split_f32(a, w, None, splits, tile), a.double() @ w.double().T
    error = (got.double().sum(0) if splits > 1 else got.double()) - want
    assert abs(float(error.mean())) * error.numel() ** 0.5 <= 5e-9 * float(want.norm())
    assert float(error.norm()) <= 2.1e-7 * float(want.norm())


@pytest.mark.parametrize("up", [1.0, -3.0, 1e30])
def test_gated_products_of_every_gate_have_the_bits_of_the_kernel_behind_a_product(ops, up):
    """All finite bfloat16 gates, down to those whose result only a large factor shows: the activation where the sums end, and the kernel with the
    library's exponential and division."""
    bits = torch.arange(65536, dtype=torch.int32, device="cuda")
    gates = torch.where(bits >= 32768, bits - 65536, bits).to(torch.int16).view(torch.bfloat16)
    gates = gates[gates.isfinite()]
    a, w = torch.zeros((gates.numel(), 64), dtype=torch.bfloat16, device="cuda"), torch.zeros((16, 64), dtype=torch.bfloat16, device="cuda")
    a[:, 0], a[:, 1], w[:8, 0], w[8:, 1] = gates, up, 1.0, 1.0
    product = ops.gemm_tiles(a, w)
    assert torch.equal(product[:, :8], gates[:, None].expand(-1, 8))
    want = ops.silu_mul(product)
    for tile in (128128, 256256):
        got = torch.empty_like(want)
        assert ops._core.velox_tiles_glu_bf16(a.data_ptr(), w.data_ptr(), got.data_ptr(), gates.numel(), 8, 64, 0, tile, ops._stream()) == 0
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("up", [1.0, -3.0, 1e30])
def test_gated_gelu_does_not_depend_on_the_number_of_rows(ops, up):
    """Sums of one term for all finite bfloat16 gates: steps of 16 rows, of 48, of 700 and of 65,280 give a row the same bits, those of the
    activation's kernel behind a product."""
    bits = torch.arange(65536, dtype=torch.int32, device="cuda")
    gates = torch.where(bits >= 32768, bits - 65536, bits).to(torch.int16).view(torch.bfloat16)
    gates = gates[gates.isfinite()]
    a, w = torch.zeros((gates.numel(), 256), dtype=torch.bfloat16, device="cuda"), torch.zeros((128, 256), dtype=torch.bfloat16, device="cuda")
    a[:, 0], a[:, 1], w[:64, 0], w[64:, 1] = gates, up, 1.0, 1.0
    want = ops.gated_act_mul(ops.gemm_tiles(a, w), "gelu_tanh")
    for rows in (16, 48, 700, gates.numel()):
        for first in sorted({0, 16100, 16500, 49000, gates.numel() - rows}):  # (from 16,100 and 49,000 on: gates of 0.4 to 12 and -1.8 to -82)
            part = slice(first, first + rows)
            if part.stop <= gates.numel():
                got = ops.linear_gated_act(a[part].contiguous(), w, torch.bfloat16, "gelu_tanh")
                assert torch.equal(got.view(torch.int16), want[part].view(torch.int16)), (rows, first)


def test_an_experts_silu_does_not_depend_on_the_number_of_pairs(ops):
    """Sums of one term, so that the kernels for few pairs and for many differ in nothing but the unit's middle: the same bits, for gates
    down to the last one with a result."""
    gates = torch.cat([torch.linspace(-89, -86, 60), torch.linspace(-30, 30, 200)]).cuda()
    x = torch.zeros((gates.numel(), 64), dtype=torch.bfloat16, device="cuda")
    x[:, 0], x[:, 1] = gates.bfloat16(), 1e30
    first, down = torch.zeros((2, 128, 64), dtype=torch.bfloat16, device="cuda"), torch.eye(64, dtype=torch.bfloat16, device="cuda").repeat(2, 1)
    first[:, :64, 0], first[:, 64:, 1] = 1.0, 1.0
    choice, weight = (torch.arange(gates.numel(), device="cuda") % 2).int()[:, None], torch.ones((gates.numel(), 1), device="cuda")

    def run(lo, hi):
        return ops.routed_experts(x[lo:hi], choice[lo:hi].contiguous(), weight[lo:hi], first.view(256, 64), down, 2, False, None, torch.bfloat16)

    whole = run(0, gates.numel())
    assert torch.equal(whole, torch.cat([run(at, min(at + 40, gates.numel())) for at in range(0, gates.numel(), 40)]))
    assert int((whole[:60] != 0).all(1).sum()) >= 50  # (all but those below -88.72)


@pytest.mark.parametrize("scale_input", [False, True])
def test_experts_of_rows_further_apart_than_the_tiles_loads_reach(ops, monkeypatch, scale_input):
    """131,080 rows of 8,192 channels, more than 2 GiB: on the matrix cores, with the bits that the same rows have in a small step (each output is one
    chain of sums whatever else is in its tile)."""
    monkeypatch.setattr(ops._core, "velox_grouped_glu", None)  # (the multiply-adds)
    tokens, hidden, inter, experts = 131080, 8192, 64, 2
    x = torch.empty((tokens, hidden), dtype=torch.bfloat16, device="cuda").normal_(generator=torch.Generator(device="cuda").manual_seed(1))
    first, down = rand((experts * 2 * inter, hidden), torch.bfloat16, 2, hidden ** -0.5), rand((experts * hidden, inter), torch.bfloat16, 3, inter ** -0.5)
    choice, weight = (torch.arange(tokens, device="cuda") // 3 % experts).int()[:, None].contiguous(), torch.rand((tokens, 1), device="cuda")

    def run(rows):
        return ops.routed_experts(x[rows], choice[rows], weight[rows], first, down, experts, scale_input, None, torch.bfloat16)

    whole = run(slice(0, tokens))
    for rows in (slice(0, 150), slice(65500, 65640), slice(tokens - 300, tokens)):
        assert torch.equal(whole[rows], run(rows))


def test_experts_whose_gate_and_up_rows_are_further_apart_than_the_tiles_loads_reach(ops, monkeypatch):
    """One expert of 65,536 x 16,384, 2 GiB a branch: on the matrix cores, in tiles of 64 rows and so with the bits of steps of at most 64 pairs."""
    monkeypatch.setattr(ops._core, "velox_grouped_glu", None)
    tokens, hidden, inter = 150, 16384, 65536
    generator = torch.Generator(device="cuda").manual_seed(1)
    first, down = (torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(std=0.01, generator=generator) for shape in ((2 * inter, hidden), (hidden, inter)))
    x, choice, weight = rand((tokens, hidden), torch.bfloat16, 4), torch.zeros((tokens, 1), dtype=torch.int32, device="cuda"), torch.rand((tokens, 1), device="cuda")
    for scale_input in (False, True):
        whole = ops.routed_experts(x, choice, weight, first, down, 1, scale_input, None, torch.bfloat16)
        for at in (0, 64, 86):
            rows = slice(at, at + 64)
            assert torch.equal(whole[rows], ops.routed_experts(x[rows], choice[rows], weight[rows], first, down, 1, scale_input, None, torch.bfloat16))
