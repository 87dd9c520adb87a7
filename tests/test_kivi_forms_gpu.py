"""The KIVI kernels at the edges of their forms: group scales on both sides of
the range whose codes need no division (a block with one outside divides
throughout), fp16 ranges that round to a zero scale, block counts off the
dequantiser's blocks per workgroup, and buffers without 16-byte alignment.
Blocks and values are the oracle's bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import kivi as K
from oracle.inputs import round_to

pytestmark = pytest.mark.gpu
TDT = {"bfloat16": torch.bfloat16, "float16": torch.float16}


def _inputs(dtype, D, n):
    rng = np.random.default_rng(D + n)
    x = rng.standard_normal((2, 1, 1, 32 * n, D)).astype(np.float32)
    if dtype == "bfloat16":  # per-token magnitudes: V groups far apart, K groups of the widest
        x[:, :, :, 32:64] *= np.exp2(rng.integers(-100, -50, (32, 1))).astype(np.float32)
        x[:, :, :, 64:96] *= np.exp2(rng.integers(45, 70, (32, 1))).astype(np.float32)
    else:  # ranges of a few subnormal steps: the scale of range 1/qmax rounds to 0
        x[:, :, :, 32:64] = rng.integers(-1, 2, (2, 1, 1, 32, D)) * 2.0 ** -24
        x[:, :, :, 64:96, ::2] = 0.0
    x[:, :, :, 96:128, :32] = np.where(rng.random((2, 1, 1, 32, 32)) < 0.5, 0.0, -0.0)
    k, v = round_to(x[0], dtype), round_to(x[1], dtype)
    return k, v


def _zeros_positive(blocks, D, bits):
    """Blocks (..., bytes) with -0 as +0 in the zeros of K and V (2D bytes each
    behind the side's codes and scales)."""
    out = blocks.copy()
    codes = 32 * D * bits // 8
    for end in (codes + 4 * D, 2 * codes + 8 * D):
        z = np.ascontiguousarray(out[..., end - 2 * D:end]).view(np.uint16)
        z[z == 0x8000] = 0
        out[..., end - 2 * D:end] = z.view(np.uint8)
    return out


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("D,n", [(64, 5), (128, 5), (256, 4)])
@pytest.mark.parametrize("bits", [2, 4, 8])
def test_quantise_and_dequantise_forms(dev, dtype, D, n, bits):
    from halo_amd import kivi
    k, v = _inputs(dtype, D, n)
    kt, vt = (torch.from_numpy(a).to(dev).to(TDT[dtype]) for a in (k, v))
    blocks = kivi.quantize(kt, vt, bits=bits)
    want = K.pack_blocks(k, v, bits=bits, dtype=dtype)
    got = blocks.cpu().numpy()
    # the sign of a zero minimum is not pinned: block 3 holds the signed zeros
    assert np.array_equal(np.delete(got, 3, axis=2), np.delete(want, 3, axis=2))
    assert np.array_equal(_zeros_positive(got[:, :, 3], D, bits), _zeros_positive(want[:, :, 3], D, bits))
    rk, rv = K.unpack_blocks(got, D=D, bits=bits, dtype=dtype)
    wk, wv = K.unpack_blocks(want, D=D, bits=bits, dtype=dtype)
    assert np.array_equal(rk, wk) and np.array_equal(rv, wv)  # 0 == -0
    kd, vd = kivi.dequantize(blocks, D=D, dtype=TDT[dtype], bits=bits)
    assert np.array_equal(kd.float().cpu().numpy(), rk)
    assert np.array_equal(vd.float().cpu().numpy(), rv)
    # one byte row off 16: the element form
    off = torch.empty(blocks.numel() + 8, device=dev, dtype=torch.uint8)[8:].view(blocks.shape)
    off.copy_(blocks)
    ku, vu = kivi.dequantize(off, D=D, dtype=TDT[dtype], bits=bits)
    assert torch.equal(ku.view(torch.int16), kd.view(torch.int16))
    assert torch.equal(vu.view(torch.int16), vd.view(torch.int16))
    # rows off 16 bytes: the tiles are loaded by element
    ke = torch.empty(kt.numel() + 1, device=dev, dtype=kt.dtype)[1:].view(kt.shape)
    ke.copy_(kt)
    assert torch.equal(kivi.quantize(ke, vt, bits=bits), blocks)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("bits", [2, 4, 8])
def test_signalling_nan(dev, D, bits):
    """bf16 NaN elements get code 0 and leave the range of their group to the
    others, quiet or signalling alike."""
    from halo_amd import kivi
    rng = np.random.default_rng(bits)
    x = torch.from_numpy(rng.standard_normal((1, 2, 96, D), dtype=np.float32)).to(dev).to(torch.bfloat16)
    blocks = []
    for nan in (0x7FC1, 0x7F81, 0xFF82 - 0x10000):
        y = x.clone()
        y.view(torch.int16)[:, :, 5::7, 3::5] = nan
        y.view(torch.int16)[:, 1, 32:64:2, 9] = nan
        blocks.append(kivi.quantize(y, y.flip(2).contiguous(), bits=bits))
    assert torch.equal(blocks[0], blocks[1]) and torch.equal(blocks[0], blocks[2])
    kd, vd = kivi.dequantize(blocks[0], D=D, dtype=torch.bfloat16, bits=bits)
    assert not kd.isnan().any() and not vd.isnan().any()
    keep = ~y.isnan()  # the codes of the numbers: within half a step of their group's range, which is below 10
    assert (kd - y).abs()[keep].max().item() <= 10 / (2 ** bits - 1) / 2 + 0.05
