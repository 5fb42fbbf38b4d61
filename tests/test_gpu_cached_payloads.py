"""Cached weight copies whose payload is not what the operator's config says: the codes' own format decides, and a copy
in host memory is refused."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(gpu, n=160, k=96):
    g = torch.Generator().manual_seed(2)
    x = torch.randn(71, k, generator=g).bfloat16().to(gpu)
    return x, (torch.randn(n, k, generator=g) * 0.05).bfloat16().to(gpu)


def _configs():
    from primus_amd.pytorch.core import Float4QuantConfig, Float8QuantConfig, Format, ScaleDtype, ScalingGranularity

    return (Float8QuantConfig(granularity=ScalingGranularity.MX_BLOCKWISE, scale_dtype=ScaleDtype.E8M0, block_size=32),
            Float4QuantConfig(activation_format=Format.E4M3))


def test_the_codes_format_decides(gpu):
    from primus_amd.pytorch import kernels as K
    from primus_amd.pytorch import ops
    from primus_amd.pytorch.core import QuantizedTensorPair, create_quantized_weight, float4_e2m1fn_x2, float8_e4m3

    x, w = _operands(gpu)
    fp8, fp4w = _configs()
    c8, c4 = create_quantized_weight(w, float8_e4m3, fp8)[0], create_quantized_weight(w, float4_e2m1fn_x2, fp4w)[0]
    assert c8.kchunk == c4.kchunk == K.LAYOUT_KSTEP
    want8, want4 = ops.gemm_fp8(x, QuantizedTensorPair(c8), config=fp8), ops.gemm_fp4(x, QuantizedTensorPair(c4), config=fp4w)
    assert not torch.equal(want8, want4)
    assert torch.equal(ops.gemm_fp8(x, c4, config=fp8), want4)
    assert torch.equal(ops.gemm_fp4(x, c8, config=fp4w), want8)


def test_a_copy_in_host_memory_is_refused(gpu):
    from primus_amd.pytorch import ops
    from primus_amd.pytorch.core import QuantizedTensor, create_quantized_weight, float8_e4m3

    x, w = _operands(gpu)
    fp8, _ = _configs()
    q = create_quantized_weight(w, float8_e4m3, fp8)[0]
    host = QuantizedTensor(q.codes.cpu(), q.scales.cpu(), logical_shape=q.shape, axis=-1, use_2d_block=True, kchunk=q.kchunk)
    with pytest.raises(ValueError, match="CPU tensor"):
        ops.gemm_fp8(x, host, config=fp8)
