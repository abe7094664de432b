"""The kernels that bring a weight into the kernels' operand format (onebit_format.hip), byte for byte: the prepared
operand against its definition in onebit_device.h, worked out with numpy from the oracle's metadata offsets."""
import numpy as np
import pytest
import torch

import oracle
import onebitsparsemul_amd as ob
from onebitsparsemul_amd import _native


def prepared_by_definition(a, e, m, k, layout):
    """a: (m k / 16,) uint8, e: (m k / 16,) int16 as stored -> the prepared bytes, K padded to whole chunks with +1 on
    positions 0 and 1 of every group."""
    chunks = (k + 255) // 256
    bits = np.unpackbits(a, bitorder="little").reshape(k // 2, m).T      # (row, compressed column), 1 = +1
    values = np.ones((m, chunks * 128), dtype=np.uint32)
    values[:, :k // 2] = bits
    r, c = np.meshgrid(np.arange(m), np.arange(k // 16), indexing="ij")
    offsets = np.array([oracle.meta_offset(int(i), int(j), m, layout) for i, j in zip(r.ravel(), c.ravel())]) \
        if layout != _native.META_LOGICAL else r.ravel() * (k // 16) + c.ravel()
    words = np.full((m, chunks * 16), 0x4444, dtype=np.uint32)
    words[:, :k // 16] = e.view(np.uint16)[offsets].reshape(m, k // 16)
    out = np.zeros((m // 32, chunks, 1536), dtype=np.uint8)
    for rb in range(m // 32):
        for kc in range(chunks):
            meta = np.zeros((64, 4), dtype=np.uint32)
            sign = np.zeros((64, 2), dtype=np.uint32)
            for lane in range(64):
                row, ga = 32 * rb + lane % 32, lane // 32
                for s in range(8):
                    meta[lane, s // 2] |= words[row, 16 * kc + 2 * s + ga] << (16 * (s % 2))
                    for t in range(8):
                        j = 4 * (s % 4) + t // 2
                        minus = 1 - values[row, 128 * kc + 8 * (2 * s + ga) + t]
                        sign[lane, s // 4] |= np.uint32(minus) << np.uint32((31 if t % 2 else 15) - j)
            out[rb, kc] = np.concatenate([meta.view(np.uint8).ravel(), sign.view(np.uint8).ravel()])
    return out.ravel()


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [_native.META_REFERENCE, _native.META_CUTLASS, _native.META_LOGICAL])
@pytest.mark.parametrize("m,k,a_shift,e_shift", [
    (64, 32, 0, 0),      # one row pair, a K tail of one step
    (320, 288, 0, 0),    # more row pairs than a workgroup holds; a second chunk of one step
    (1088, 544, 0, 0),   # more than one strip of sixteen row pairs, the last one mostly empty
    (128, 256, 4, 0),    # `a` off its 8-byte boundary
    (192, 96, 1, 1),     # `a` off every boundary, metadata off its dword boundary
])
def test_prepared_operand_bytes(m, k, a_shift, e_shift, layout):
    rng = np.random.default_rng(m + k + layout)
    count = m * k // 16
    a = rng.integers(0, 256, count, dtype=np.uint8)
    e = rng.integers(-32768, 32768, count, dtype=np.int64).astype(np.int16)
    a_gpu = torch.zeros(count + 16, dtype=torch.uint8, device="cuda")
    e_gpu = torch.zeros(count + 8, dtype=torch.int16, device="cuda")
    a_gpu[a_shift:a_shift + count] = torch.from_numpy(a).cuda()
    e_gpu[e_shift:e_shift + count] = torch.from_numpy(e).cuda()
    got = _native.prepare(a_gpu[a_shift:a_shift + count], e_gpu[e_shift:e_shift + count], m, k, layout)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), prepared_by_definition(a, e, m, k, layout))


def stored_by_oracle(w, prune, layout):
    """mask -> compress -> quantise -> pack of the dense weight w (float32 values), as the oracle does it."""
    if prune:
        w = np.where(oracle.mask_creator(w) != 0, w, 0).astype(np.float32)
    sparse, meta = oracle.sparse_from_dense(w, layout)
    return oracle.pack_binary(np.ascontiguousarray(oracle.binary_quant(sparse).T)), meta


@pytest.mark.gpu
@pytest.mark.parametrize("prune", [True, False])
@pytest.mark.parametrize("m,k,layout", [
    (64, 32, _native.META_REFERENCE),     # one row tile, half a K tile
    (320, 96, _native.META_REFERENCE),    # more row tiles than a workgroup holds, a K tail of half a tile
    (1088, 192, _native.META_REFERENCE),  # more than one strip of sixteen row tiles
    (128, 160, _native.META_CUTLASS),
])
def test_packed_weight_bytes(m, k, layout, prune):
    rng = np.random.default_rng(m + k)
    # few distinct magnitudes (ties), zeros of both signs, the smallest half-precision number, infinities
    values = np.array([0.0, -0.0, 1.0, -1.0, 0.5, -0.5, 2.0**-24, -2.0**-24, np.inf, -np.inf], dtype=np.float32)
    w = rng.normal(0, 0.02, (m, k)).astype(np.float16).astype(np.float32)
    picked = rng.random((m, k)) < 0.6
    w[picked] = rng.choice(values, picked.sum())
    a, meta = _native.pack_weight(torch.from_numpy(w).cuda().half(), prune=prune, layout=layout)
    torch.cuda.synchronize()
    want_a, want_meta = stored_by_oracle(w, prune, layout)
    assert np.array_equal(a.cpu().numpy().ravel(), want_a.ravel())
    assert np.array_equal(meta.cpu().numpy().ravel(), want_meta.ravel())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,k", [(64, 32), (320, 96), (1088, 192)])
def test_pack_of_bf16_and_fp32_weights(m, k, dtype):
    """The fused kernel against the layer's tensor route on the CPU, with ties, zeros, the values around the smallest
    half-precision number, infinities and NaN (w * mask makes a NaN of an infinity that the mask removes)."""
    rng = np.random.default_rng(m + k)
    values = np.array([0.0, -0.0, 1.0, -1.0, 0.5, -0.5, 2.0**-24, -2.0**-24, 2.0**-25, -2.0**-25, 2.0**-25 * 1.01, 2.0**-130,
                       7e4, np.inf, -np.inf, np.nan], dtype=np.float32)
    w = rng.normal(0, 0.02, (m, k)).astype(np.float32)
    picked = rng.random((m, k)) < 0.6
    w[picked] = rng.choice(values, picked.sum())
    w = torch.from_numpy(w).to(dtype)
    on_cpu, on_gpu = ob.BinaryLinear_2_4(k, m), ob.BinaryLinear_2_4(k, m)
    on_cpu.pack(w)
    on_gpu.pack(w.cuda())
    torch.cuda.synchronize()
    assert torch.equal(on_gpu.packed_binary_sparse.cpu(), on_cpu.packed_binary_sparse)
    assert torch.equal(on_gpu.meta.cpu(), on_cpu.meta)
