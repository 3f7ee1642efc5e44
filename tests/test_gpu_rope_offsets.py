"""The fused q/k RoPE kernel with the packed sequences' offsets in place of
per-token positions: the same bits as with positions_from_cu_seqlens (the
rotation itself is the same code), at the edges of what it takes: one sequence,
64 of them (the most its table holds), 65 (the layer falls back to positions),
empty sequences at the start, between and at the end, and offsets that it does
not take as they are (int64, a strided view)."""

import pytest
import torch

from flashprefill_amd.attention_layer import (PrefillAttention, fused_rope_qk,
                                              positions_from_cu_seqlens)

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

LENS = {"one": [777], "single_token": [1], "two": [300, 212],
        "empty": [0, 5, 0, 0, 130, 0], "most": [(7 * i) % 23 for i in range(64)],
        "beyond": [(5 * i) % 17 + 1 for i in range(65)]}


def _cu(lens):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return torch.tensor(cu, dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 128), (torch.float16, 64),
                                     (torch.bfloat16, 256)])
@pytest.mark.parametrize("name", list(LENS))
def test_offsets_give_the_bits_of_positions(name, dtype, d):
    cu = _cu(LENS[name])
    T = int(cu[-1].item())
    g = torch.Generator(device=DEV).manual_seed(5)
    qkv = torch.randn(T, 6, d, generator=g, device=DEV).to(dtype)
    ref = qkv.clone()
    fused_rope_qk(ref[:, :4], ref[:, 4:5], positions_from_cu_seqlens(cu, T), 1e6, max_position=T)
    if len(LENS[name]) > 64:
        with pytest.raises(ValueError):  # the kernel's table holds 64
            fused_rope_qk(qkv[:, :4], qkv[:, 4:5], None, 1e6, max_position=T, cu_seqlens=cu)
    else:
        fused_rope_qk(qkv[:, :4], qkv[:, 4:5], None, 1e6, max_position=T, cu_seqlens=cu)
        assert torch.equal(qkv, ref)

    layer = PrefillAttention(64, 4, 1, d, rope_theta=1e6, dtype=dtype, device=DEV, seed=7)
    x = torch.randn(T, 64, generator=g, device=DEV).to(dtype)
    want = (x @ layer.w_qkv.t()).view(T, 6, d)
    fused_rope_qk(want[:, :4], want[:, 4:5], positions_from_cu_seqlens(cu, T), 1e6,
                  max_position=T)
    strided = torch.stack([cu, cu], dim=1)[:, 0]
    for form in (cu, cu.long(), strided):
        q, k, v = layer.project_qkv(x, form)
        assert torch.equal(torch.cat([q, k, v], dim=1), want)
