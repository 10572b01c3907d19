"""The GEMMs of the 32-value formats, TQ2_0, Q4_K and expanded Q6_K at the edges of their tiles, against the oracle bit for bit.

A workgroup computes 128 rows in four groups of 32 and 8, 16 or 32 tokens, over chunks of 256 values: rows,
tokens and values that fall short of each, the token tile of every width, and scales that are not finite
(the products then are not single fused operations).  Launches of at most 256 groups of 32 rows x 8 tokens share
a row's chunks between eight waves, which add in turn: fewer chunks than waves, as many, and a remainder; so partial
chunks and scales that are not finite come at that kernel and at each tile of the other.  Sums are in block order
(src/quant.cpp:445-482, :500-521, :549-563, :580-596), so the results equal the oracle's matvec of each token.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from brisk_hip import lib as L  # noqa: E402
import pyoracle  # noqa: E402
from test_gpu_kernels import BLOCK, Q4_0, Q4_1, Q4_K, Q5_0, Q6_K, Q8_0, Q8K, TQ2_0, activations, dev, host, p, packed, quant_ref, weights  # noqa: E402

TYPES = (Q4_0, Q4_1, Q5_0, Q8_0, TQ2_0, Q4_K, Q6_K)
# rows, values, tokens: short of a row group, of a workgroup, of a chunk; then enough workgroups for the wider token tiles
SHAPES = [(1, 256, 2), (31, 512, 8), (33, 1024, 9), (129, 768, 31), (300, 256, 33), (1153, 512, 250), (2100, 512, 513),
          (70, 2048, 8), (33, 2304, 9), (65, 4352, 7), (8161, 256, 3), (8193, 256, 3), (3001, 512, 190)]
PARTIAL = [(40, 32, 3), (130, 288, 17), (65, 1120, 40), (1153, 288, 80), (1153, 1120, 250), (2100, 288, 513)]
NOT_FINITE = [(70, 512, 20), (70, 512, 700), (1153, 512, 250), (2100, 512, 513)]  # shared chunks, then 8, 16 and 32 tokens


def run(type_, rows, cols, n, w):
    lib, orc = L.load(), pyoracle.oracle_lib()
    q8k = type_ in Q8K
    bits = orc.or_activation_bits(type_, rows)
    xq = np.concatenate([quant_ref(orc, activations(cols, 300 + t), q8k, bits) for t in range(n)])
    rb = cols // BLOCK[type_][0] * (292 if q8k else 34)
    want = np.zeros((n, rows), np.float32)
    for t in range(n):
        orc.or_matvec(type_, pyoracle.ptr(w), rows, cols, pyoracle.ptr(xq[t * rb:(t + 1) * rb]), pyoracle.ptr(want[t]))
    flags = 1 if (type_ == TQ2_0 and rows % 16 == 0) else 0
    wd, xd = packed(lib, type_, w, rows, cols), dev(xq)
    out = torch.full((n, rows + 5), 7.0, dtype=torch.float32, device="cuda")
    L.check(lib.brisk_hip_matmul(type_, flags, p(wd), rows, cols, p(xd), n, p(out), rows + 5, None))
    got = host(out, np.float32).reshape(n, rows + 5)
    assert (got[:, rows:] == 7.0).all()  # nothing past the rows
    return got[:, :rows], want


@pytest.mark.parametrize("type_", TYPES)
def test_tile_edges(type_):
    assert torch.cuda.is_available()
    for rows, cols, n in SHAPES + ([] if type_ in Q8K else PARTIAL):
        print(f"[block gemm] type {type_} {rows} x {cols}, {n} tokens", flush=True)
        got, want = run(type_, rows, cols, n, weights(type_, rows, cols, rows * 31 + cols + n))
        np.testing.assert_array_equal(got, want, err_msg=f"{rows} x {cols}, {n} tokens")


@pytest.mark.parametrize("type_", TYPES)
def test_scales_that_are_not_finite(type_):
    be, bb = BLOCK[type_]
    at = bb - 2 if type_ in (TQ2_0, Q6_K) else 0  # the block's fp16 scale
    for rows, cols, n in NOT_FINITE:
        print(f"[block gemm] type {type_} {rows} x {cols}, {n} tokens, scales not finite", flush=True)
        w = weights(type_, rows, cols, 5).view(np.uint8).reshape(rows, cols // be, bb).copy()
        for row, blk, bits in ((3, 1, 0x7C00), (34, 0, 0xFC00), (69, cols // be - 1, 0x7E00), (40, 0, 0x7BFF), (41, 1, 0x0001)):
            w[row, blk, at:at + 2] = np.frombuffer(np.uint16(bits).tobytes(), np.uint8)
        got, want = run(type_, rows, cols, n, w.reshape(-1))
        assert not np.isfinite(want[:, (3, 34, 69)]).any() and np.isfinite(np.delete(want, (3, 34, 69), axis=1)).all()
        np.testing.assert_array_equal(got, want, err_msg=f"{rows} x {cols}, {n} tokens")
