"""GPU INT8 attention on the reference kernel's scheme (128-key blocks): the
preparation bit for bit against the oracle's restatement (kitchen_prepare),
the attention within 1e-5 of kitchen_attention (the same u8 codes; the GPU
uses the hardware exp2 and its own FP32 summation order, measured below 1e-6
at 130 to 53504 keys) and close to exact softmax attention."""
import numpy as np
import pytest
import torch

from oracle import int8_attention as oa
from helpers import np_of
from w8a8 import int8_attention, kernels

pytestmark = pytest.mark.gpu

SHAPES = [
    # b, h, nq, nk, dtype
    (1, 1, 1, 1, torch.float16),
    (1, 2, 70, 130, torch.float16),
    (2, 3, 200, 64, torch.float32),
    (1, 1, 128, 300, torch.float16),
    (1, 2, 257, 1000, torch.float16),
    # 13, 14 and 15 key blocks, key counts that are and are not multiples of
    # 128, and long sequences (queries are independent, so a short query set
    # exercises the whole key loop). One or two heads of few queries take the
    # kernel that splits the keys over a workgroup's waves, from two blocks on.
    (1, 1, 64, 1600, torch.float16),
    (1, 1, 33, 1664, torch.float16),
    (1, 1, 40, 1792, torch.float16),
    (1, 1, 40, 1920, torch.float16),
    (1, 2, 40, 4000, torch.float16),
    (1, 2, 48, 16384, torch.float16),
]


def _qkv(g, b, h, nq, nk, dtype, kshift=0.5, qmul=1.0):
    q = torch.randn((b, h, nq, 128), generator=g) * qmul
    k = torch.randn((b, h, nk, 128), generator=g) + kshift
    v = torch.randn((b, h, nk, 128), generator=g)
    return q.to(dtype), k.to(dtype), v.to(dtype)


def _np(t):
    return np_of(t).astype(np.float32) if t.dtype == torch.float16 else np_of(t)


@pytest.mark.parametrize('b,h,nq,nk,dtype', SHAPES)
def test_prepare_matches_oracle(gpu, b, h, nq, nk, dtype):
    g = torch.Generator().manual_seed(nq * 7 + nk)
    q, k, v = _qkv(g, b, h, nq, nk, dtype)
    prep = kernels.attention_prepare(q.to(gpu), k.to(gpu), v.to(gpu))
    want = oa.gpu_operands(oa.kitchen_prepare(_np(q), _np(k), _np(v), cta_k=oa.GPU_CTA_K))
    for name in oa.GPU_OPERANDS:
        got = np_of(prep[name])
        assert got.shape == want[name].shape, name
        if got.dtype == np.float32:
            assert np.array_equal(got.view(np.uint32), want[name].view(np.uint32)), name
        else:
            assert np.array_equal(got, want[name]), name


def _check(out, want, exact, tol, min_cos=0.999):
    out = np_of(out).astype(np.float64)
    err = np.abs(out - want).max()
    scale = np.abs(want).max()
    assert err <= tol * scale, (err, scale)
    cos = (out * exact).sum() / np.sqrt((out * out).sum() * (exact * exact).sum())
    assert cos > min_cos, cos
    return err / scale


@pytest.mark.parametrize('b,h,nq,nk,dtype', SHAPES)
def test_attention_matches_oracle(gpu, b, h, nq, nk, dtype):
    g = torch.Generator().manual_seed(nq * 13 + nk)
    q, k, v = _qkv(g, b, h, nq, nk, dtype)
    prep = kernels.attention_prepare(q.to(gpu), k.to(gpu), v.to(gpu))
    out = kernels.attention(prep, out_dtype=torch.float32)
    oprep = oa.kitchen_prepare(_np(q), _np(k), _np(v), cta_k=oa.GPU_CTA_K)
    want = oa.kitchen_attention(oprep).astype(np.float64)
    exact = oa.reference_attention(_np(q), _np(k), _np(v))
    # Tile-relative u8 probabilities keep their accuracy on long rows; the
    # GPU-vs-oracle bound (hardware exp2, FP32 order) is the same at every
    # length.
    rel = _check(out, want, exact, 1e-5, min_cos=0.9995)
    print(f'b={b} h={h} nq={nq} nk={nk}: max |gpu - oracle| / max |oracle| = {rel:.2e}')
    out16 = kernels.attention(prep, out_dtype=torch.float16)
    assert torch.equal(out16, out.half())


@pytest.mark.parametrize('nk', [1024, 4096, 16384, 53504])
def test_error_vs_exact_no_worse_than_restatement(gpu, nk):
    # Long rows up to the DiT sequence (53504 keys), a short query set: the
    # kernel's error against exact float64 attention stays within 2% of the
    # restatement's (whose exp2 is exact), at every length.
    g = torch.Generator().manual_seed(nk)
    q, k, v = _qkv(g, 1, 1, 32, nk, torch.float16)
    prep = kernels.attention_prepare(q.to(gpu), k.to(gpu), v.to(gpu))
    out = np_of(kernels.attention(prep, out_dtype=torch.float32)).astype(np.float64)
    want = oa.kitchen_attention(oa.kitchen_prepare(_np(q), _np(k), _np(v), cta_k=oa.GPU_CTA_K)).astype(np.float64)
    exact = oa.reference_attention(_np(q), _np(k), _np(v))
    scale = np.abs(exact).max()
    err_gpu = np.abs(out - exact).max() / scale
    err_oracle = np.abs(want - exact).max() / scale
    print(f'nk={nk}: max error / max |exact|: kernel {err_gpu:.4e}, restatement {err_oracle:.4e}')
    assert err_gpu <= 1.02 * err_oracle + 1e-5, (err_gpu, err_oracle)
    assert np.abs(out - want).max() <= 1e-5 * np.abs(want).max()


def test_large_logits_and_uniform_keys(gpu):
    g = torch.Generator().manual_seed(5)
    q, k, v = _qkv(g, 1, 1, 96, 200, torch.float32, qmul=40.0)     # sharp softmax, large running maxima
    k[:, :, 100:] = k[:, :, :100]
    prep = kernels.attention_prepare(q.to(gpu), k.to(gpu), v.to(gpu))
    out = kernels.attention(prep, out_dtype=torch.float32)
    want = oa.kitchen_attention(oa.kitchen_prepare(_np(q), _np(k), _np(v), cta_k=oa.GPU_CTA_K)).astype(np.float64)
    exact = oa.reference_attention(_np(q), _np(k), _np(v))
    # A near one-hot softmax magnifies the Q/K quantization error: the scheme
    # itself is looser here, the kernel still follows the oracle closely.
    print(f'sharp softmax: max |gpu - oracle| / max |oracle| = {_check(out, want, exact, 1e-5, min_cos=0.95):.2e}')
    # identical keys (a partial last block: the floor scale keeps its padded
    # keys masked): every query averages the quantized values
    ku = torch.ones((1, 1, 250, 128)) * torch.randn((1, 1, 1, 128), generator=g)
    vu = torch.randn((1, 1, 250, 128), generator=g)
    prep = kernels.attention_prepare(q[:, :, :64].to(gpu), ku.to(gpu), vu.to(gpu))
    out = np_of(kernels.attention(prep, out_dtype=torch.float32))
    op = oa.kitchen_prepare(_np(q[:, :, :64]), _np(ku), _np(vu), cta_k=oa.GPU_CTA_K)
    mean_v = (op['v8'][:, :, :250].astype(np.float64) * op['vs'][:, :, None, :]).mean(2)
    assert np.abs(out - mean_v[:, :, None, :]).max() <= 1e-5 * np.abs(mean_v).max()


def test_reference_api(gpu):
    g = torch.Generator().manual_seed(9)
    q, k, v = _qkv(g, 1, 2, 100, 150, torch.float16)
    q, k, v = q.to(gpu), k.to(gpu), v.to(gpu)
    out = int8_attention.int8_attention(q, k, v)
    assert out.dtype == torch.float16 and out.shape == q.shape
    prepared = int8_attention.prequantize_int8_attention(q, k, v)
    assert torch.equal(int8_attention.int8_attention_from_prequantized(prepared), out)
    prepared.release()
    with pytest.raises(ValueError):
        int8_attention.int8_attention_from_prequantized(prepared)
    with pytest.raises(ValueError):
        int8_attention.int8_attention(q, k, v, attn_mask=torch.ones((100, 150), device=gpu))
    with pytest.raises(ValueError):
        int8_attention.int8_attention(q[..., :64], k[..., :64], v[..., :64])
    scaled = int8_attention.int8_attention(q, k, v, scale=0.05)
    want = oa.kitchen_attention(oa.kitchen_prepare(_np(q.cpu()), _np(k.cpu()), _np(v.cpu()), cta_k=oa.GPU_CTA_K,
                                                   sm_scale=0.05))
    # fp16 output: within one fp16 rounding of the restatement
    assert np.abs(np_of(scaled).astype(np.float64) - want).max() <= 2 ** -10 * np.abs(want).max()


@pytest.mark.parametrize('b,h,n,dtype', [(1, 3, 150, torch.float16), (2, 2, 70, torch.float32)])
def test_strided_operands_and_output(gpu, b, h, n, dtype):
    """q, k, v read in place from a packed [b, n, 3 h 128] projection and the
    output written as [b, n, h, 128] rows give the bits of the contiguous
    route."""
    g = torch.Generator().manual_seed(31 + n)
    packed = torch.randn((b, n, 3 * h * 128), generator=g).to(dtype).to(gpu)
    q, k, v = (packed[..., i * h * 128:(i + 1) * h * 128].view(b, n, h, 128).transpose(1, 2) for i in range(3))
    assert kernels._row_strides(q) is not None and not q.is_contiguous()
    prep = kernels.attention_prepare(q, k, v)
    flat = kernels.attention_prepare(q.contiguous(), k.contiguous(), v.contiguous())
    for name in ('q8', 'qs', 'k8', 'ks', 'vt8', 'vs', 'vsum'):
        assert torch.equal(prep[name], flat[name]), name
    for out_dtype in (torch.float16, torch.float32):
        want = kernels.attention(flat, out_dtype=out_dtype)
        rows = torch.full((b, n, h, 128), float('nan'), dtype=out_dtype, device=gpu)
        got = kernels.attention(prep, out_dtype=out_dtype, out=rows.transpose(1, 2))
        assert got.data_ptr() == rows.data_ptr()
        assert torch.equal(rows, want.transpose(1, 2).contiguous())
    # misaligned rows fall back to a copy on input and are refused as output
    odd = torch.randn((1, 1, 40, 129), generator=g).to(dtype).to(gpu)[..., 1:]
    assert kernels._row_strides(odd) is None
    kernels.attention_prepare(odd, odd, odd)
    with pytest.raises(ValueError):
        kernels.attention(flat, out_dtype=torch.float32, out=torch.empty((b, h, n, 130), device=gpu)[..., :128])


# The preparation's own edges: chunks of 256 keys and their batches of 32
# (remainders), fp32's two phases to a chunk, 32 chunks (the last count the
# quantizer reduces itself) and 33 (the finishing kernel).
@pytest.mark.parametrize('nq,nk,dtype', [(5, 31, torch.float32), (130, 33, torch.float16), (1, 255, torch.float32),
                                         (128, 256, torch.float16), (129, 257, torch.float32), (3, 385, torch.float32),
                                         (2, 8192, torch.float16), (2, 8193, torch.float32)])
def test_prepare_chunk_edges(gpu, nq, nk, dtype):
    g = torch.Generator().manual_seed(nq + 31 * nk)
    q, k, v = _qkv(g, 1, 2, nq, nk, dtype)
    prep = kernels.attention_prepare(q.to(gpu), k.to(gpu), v.to(gpu))
    want = oa.gpu_operands(oa.kitchen_prepare(_np(q), _np(k), _np(v), cta_k=oa.GPU_CTA_K))
    for name in oa.GPU_OPERANDS:
        assert np_of(prep[name]).tobytes() == np.ascontiguousarray(want[name]).tobytes(), name


def test_prepare_ties_and_wide_scales(gpu):
    """Codes where x / s lies on or next to a tie (the reciprocal product does
    not decide), and scales whose reciprocal is not a normal number."""
    g = torch.Generator().manual_seed(77)
    half = torch.randint(-254, 255, (1, 3, 140, 128), generator=g).float() * 0.5
    half[..., 0] = 127.0
    q, k, v = half.clone(), half - half.mean(2, keepdim=True), half.clone()
    q[:, 1] *= 3e38 / 127.0
    v[:, 1] *= 3e38 / 127.0
    q[:, 2] *= 1e-38
    v[:, 2] *= 1e-38
    prep = kernels.attention_prepare(q.to(gpu), k.to(gpu), v.to(gpu))
    want = oa.gpu_operands(oa.kitchen_prepare(_np(q), _np(k), _np(v), cta_k=oa.GPU_CTA_K))
    for name in oa.GPU_OPERANDS:
        assert np_of(prep[name]).tobytes() == np.ascontiguousarray(want[name]).tobytes(), name


# (queries, heads, keys) and whether the call splits the keys over a
# workgroup's waves, on 256 CUs (test_plans.py asks the library). 260 heads of
# 100 or more queries fill the GPU with 128-query workgroups: the step loop's
# two-step unroll and every tail (13, 14 and 15 blocks: after the loop one or no
# further step, then the step whose next block is the last, alternating tiles),
# two, three and one block, whole and ragged query tiles and last blocks.
BOTH_KERNELS = [(128, 260, 1600, False), (100, 260, 1664, False), (129, 260, 1792, False), (128, 260, 1920, False),
                (100, 260, 130, False), (129, 260, 384, False), (200, 260, 64, False),
                (33, 260, 1600, True), (64, 260, 1664, True), (40, 260, 1792, True), (33, 260, 1920, True),
                (32, 260, 130, True)]
# A few heads of enough queries for five rounds of split workgroups, many keys.
LONG_PLAIN = (9000, 4, 16384, False)


@pytest.mark.parametrize('nq,heads,nk,split', BOTH_KERNELS)
def test_both_kernels_match_oracle(gpu, nq, heads, nk, split):
    """The kernel that the whole call takes, and one head alone (always split
    here, but for a single block), against the oracle."""
    g = torch.Generator().manual_seed(nq + nk)
    q, k, v = _qkv(g, 1, heads, nq, nk, torch.float16)
    many = np_of(kernels.attention(kernels.attention_prepare(q.to(gpu), k.to(gpu), v.to(gpu)), out_dtype=torch.float32))
    for h in (0, heads - 1):
        qh, kh, vh = (t[:, h:h + 1].contiguous() for t in (q, k, v))
        one = np_of(kernels.attention(kernels.attention_prepare(qh.to(gpu), kh.to(gpu), vh.to(gpu)),
                                      out_dtype=torch.float32))
        want = oa.kitchen_attention(oa.kitchen_prepare(_np(qh), _np(kh), _np(vh), cta_k=oa.GPU_CTA_K))
        # 1e-5: the bound of test_attention_matches_oracle (hardware exp2, FP32 order)
        for out in (many[:, h:h + 1], one):
            assert np.abs(out - want).max() <= 1e-5 * np.abs(want).max()


def test_long_rows_without_the_split(gpu):
    """Many keys on the kernel of 128-query workgroups: the first 32 queries
    and the ragged last ones of two heads (queries are independent, and a
    32-row group shares its scales)."""
    nq, heads, nk, _ = LONG_PLAIN
    g = torch.Generator().manual_seed(nk)
    q, k, v = _qkv(g, 1, heads, nq, nk, torch.float16)
    out = np_of(kernels.attention(kernels.attention_prepare(q.to(gpu), k.to(gpu), v.to(gpu)), out_dtype=torch.float32))
    for h in (0, heads - 1):
        for a, b in ((0, 32), (nq // 32 * 32, nq)):
            qh, kh, vh = q[:, h:h + 1, a:b].contiguous(), k[:, h:h + 1].contiguous(), v[:, h:h + 1].contiguous()
            want = oa.kitchen_attention(oa.kitchen_prepare(_np(qh), _np(kh), _np(vh), cta_k=oa.GPU_CTA_K))
            assert np.abs(out[:, h:h + 1, a:b] - want).max() <= 1e-5 * np.abs(want).max()
