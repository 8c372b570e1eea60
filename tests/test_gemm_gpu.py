"""GPU parity of the prefill Q4_0 GEMM (kdq_quantize_q8, kdq_gemm_q4_0, and
kdq_gemm_q4_0_packed over the tile-packed layout of kdq_gguf_pack).

The activation codes and scales must be bit-exact to the oracle's restatement of
ggml's x86 quantize_row_q8_0 (which tests/test_oracle.py pins to the compiled
reference).  The fp16 output must be within rel-L2 <= 1e-3 and max-abs <= 2e-2 of the
output RMS of the oracle's Q4_0 x Q8 product over the same codes (double accumulation).
"""
import numpy as np
import pytest

from kadan_amd import synth
from tests.util import assert_close

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    return torch


@pytest.mark.parametrize("m,k", [(1, 32), (3, 256), (64, 4096), (512, 4096), (7, 14336)])
def test_quantize_bit_exact(device, oracle, m, k):
    torch = _torch()
    x = synth.normal(0xC3 + m, 1, m * k).reshape(m, k).astype(np.float16)
    # exact half-way cases: values that land on .5 after scaling by 127/amax
    x[0, 0] = np.float16(127.0)
    if k >= 32:
        x[0, 1] = np.float16(0.5)   # 0.5 * 127/127 = 0.5 -> 0 (even)
        x[0, 2] = np.float16(1.5)   # -> 2
        x[0, 3] = np.float16(-2.5)  # -> -2
    if m > 1:
        x[1, :32] = 0  # all-zero block: d = 0, codes 0
    qs, d = oracle.quantize_q8_f16(x.view(np.uint16))
    from kadan_amd import ops
    gq, gd = ops.quantize_q8(torch.from_numpy(x).to(device))
    assert np.array_equal(gq.cpu().numpy(), qs)
    assert np.array_equal(gd.cpu().numpy().view(np.uint32), d.view(np.uint32))


SHAPES = [(1, 256, 1), (5, 256, 130), (128, 512, 128), (130, 1024, 300), (33, 4096, 256),
          (256, 4096, 1024), (512, 4096, 640)]
# token tiles of 32, 64 and 128 at their edges, K slices (odd m * n, partial weight tiles)
SHAPES += [(2, 2560, 770), (31, 1280, 33), (32, 2304, 512), (63, 1536, 257), (65, 5632, 131),
           (129, 2048, 1001)]


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_gemm_q4_0_parity(device, oracle, m, k, n):
    torch = _torch()
    seed = (m * 131 + k * 7 + n) & 0xFFFF
    w = synth.q4_0_weights(seed, n, k)
    x = synth.normal(seed, 9, m * k).reshape(m, k).astype(np.float16)
    xq, xd = oracle.quantize_q8_f16(x.view(np.uint16))
    expected = oracle.gemm_q4_0_q8(w, n, k, xq, xd)
    from kadan_amd import ops
    y = ops.gemm_q4_0(torch.from_numpy(w).to(device), torch.from_numpy(x).to(device), n)
    got = y.float().cpu().numpy()
    assert_close(got, expected, what=f"gemm m={m} k={k} n={n}")


def test_gemm_q4_0_baseline_shape_property(device, oracle):
    """C3 at full size (M=512, K=4096, N=14336): a column sample against the oracle, and
    linearity in the activations through the exact-code path (scaling x by 2 scales the
    codes' scale exactly, so the output doubles up to fp16 rounding)."""
    torch = _torch()
    m, k, n = 512, 4096, 14336
    w = synth.q4_0_weights(0xC3, n, k)
    x = synth.normal(0xC3, 9, m * k).reshape(m, k).astype(np.float16)
    from kadan_amd import ops
    wd = torch.from_numpy(w).to(device)
    xd_ = torch.from_numpy(x).to(device)
    y = ops.gemm_q4_0(wd, xd_, n).float().cpu().numpy()
    cols = np.arange(0, n, 97)
    xq, xs = oracle.quantize_q8_f16(x.view(np.uint16))
    expected = oracle.gemm_q4_0_q8(np.ascontiguousarray(w[cols]), cols.size, k, xq, xs)
    assert_close(y[:, cols], expected, what="C3 column sample")
    y2 = ops.gemm_q4_0(wd, xd_ * 2, n).float().cpu().numpy()
    assert_close(y2, 2 * y, rel=1e-6, mabs=1e-5, what="doubling")


# odd group counts (k / 256), ragged n (not a multiple of 16, 8 or 4), m below, at and
# above the 128-token tile
PACKED_SHAPES = SHAPES + [(1, 768, 16), (129, 1280, 250), (200, 768, 301), (64, 512, 514)]


def _packed(torch, device, w, k):
    from kadan_amd import ops
    return ops.gguf_pack(2, torch.from_numpy(w).to(device), k)


@pytest.mark.parametrize("m,k,n", PACKED_SHAPES)
def test_gemm_q4_0_packed_parity(device, oracle, m, k, n):
    torch = _torch()
    seed = (m * 131 + k * 7 + n) & 0xFFFF
    w = synth.q4_0_weights(seed, n, k)
    x = synth.normal(seed, 9, m * k).reshape(m, k).astype(np.float16)
    xq, xd = oracle.quantize_q8_f16(x.view(np.uint16))
    expected = oracle.gemm_q4_0_q8(w, n, k, xq, xd)
    from kadan_amd import ops
    packed = _packed(torch, device, w, k)
    y = torch.full((m, n), float("nan"), dtype=torch.float16, device=device)
    ops.gemm_q4_0_packed(packed, torch.from_numpy(x).to(device), n, out=y)
    got = y.float().cpu().numpy()
    assert np.isfinite(got).all(), "an output element was not written"
    assert_close(got, expected, what=f"packed gemm m={m} k={k} n={n}")
    # same fp16 operands as the row-major kernel: only the fp32 summation order differs
    y_row = ops.gemm_q4_0(torch.from_numpy(w).to(device), torch.from_numpy(x).to(device), n)
    assert_close(got, y_row.float().cpu().numpy(), rel=1e-4, mabs=1e-2,
                 what=f"packed vs row-major m={m} k={k} n={n}")


def test_gemm_q4_0_packed_baseline_shape_property(device, oracle):
    """C3 at full size through the packed layout: a column sample against the oracle, the
    doubling property, and a second call with fewer tokens into the same output (rows
    past the new m stay untouched)."""
    torch = _torch()
    m, k, n = 512, 4096, 14336
    w = synth.q4_0_weights(0xC3, n, k)
    x = synth.normal(0xC3, 9, m * k).reshape(m, k).astype(np.float16)
    from kadan_amd import ops
    packed = _packed(torch, device, w, k)
    xd_ = torch.from_numpy(x).to(device)
    y = ops.gemm_q4_0_packed(packed, xd_, n).float().cpu().numpy()
    cols = np.arange(0, n, 97)
    xq, xs = oracle.quantize_q8_f16(x.view(np.uint16))
    expected = oracle.gemm_q4_0_q8(np.ascontiguousarray(w[cols]), cols.size, k, xq, xs)
    assert_close(y[:, cols], expected, what="C3 packed column sample")
    y2 = ops.gemm_q4_0_packed(packed, xd_ * 2, n).float().cpu().numpy()
    assert_close(y2, 2 * y, rel=1e-6, mabs=1e-5, what="doubling")
    out = torch.full((m, n), 7.0, dtype=torch.float16, device=device)
    ops.gemm_q4_0_packed(packed, xd_[:100].contiguous(), n, out=out[:100])
    got = out.float().cpu().numpy()
    assert_close(got[:100], y[:100], rel=1e-6, mabs=1e-5, what="first 100 tokens")
    assert (got[100:] == 7.0).all()


def _rows_case(device, m, k, n):
    torch = _torch()
    w = synth.q4_0_weights(m + k + n, n, k)
    x = synth.normal(m + k + n, 9, m * k).reshape(m, k).astype(np.float16)
    return w, x, torch.from_numpy(w).to(device), torch.from_numpy(x).to(device)


@pytest.mark.parametrize("m,k,n,packs", [
    (1, 512, 300, False), (64, 512, 12288, False), (513, 256, 640, False),   # short rows
    (1, 768, 12161, False), (64, 1024, 16384, False), (300, 768, 9217, False),  # wide outputs
    (200, 2048, 24449, False), (5, 2304, 32641, False),
    (9, 768, 1000, True), (64, 768, 12160, True), (300, 768, 9088, True),    # packed first,
    (200, 2048, 24448, True), (70, 2304, 300, True)])                        # K whole or sliced
def test_gemm_q4_0_rows_packed_first_or_not(device, oracle, m, k, n, packs):
    """Both ways that row-major weights take, at the edges of the rule between them: against
    the oracle on a sample of columns, and, packed first, the bits of kdq_gemm_q4_0_packed."""
    torch = _torch()
    from kadan_amd import ops
    w, x, wd, xd = _rows_case(device, m, k, n)
    y = torch.full((m, n), float("nan"), dtype=torch.float16, device=device)
    ops.gemm_q4_0(wd, xd, n, out=y)
    assert torch.isfinite(y).all(), "an output element was not written"
    cols = np.unique(np.concatenate([np.arange(0, n, max(1, n // 150)), [n - 1]]))
    xq, xs = oracle.quantize_q8_f16(x.view(np.uint16))
    want = oracle.gemm_q4_0_q8(np.ascontiguousarray(w[cols]), cols.size, k, xq, xs)
    assert_close(y.float().cpu().numpy()[:, cols], want, what=f"rows gemm m={m} k={k} n={n}")
    if packs:
        packed = ops.gemm_q4_0_packed(ops.gguf_pack(2, wd, k), xd, n)
        assert torch.equal(y.view(torch.int16), packed.view(torch.int16))


@pytest.mark.parametrize("m,k,n", [(4, 4096, 131072), (300, 8192, 65536)])
def test_gemm_q4_0_rows_holds_no_copy_of_large_weights(device, m, k, n):
    """302 MB of row-major weights: the workspace holds the activations, no second copy."""
    torch = _torch()
    import kadan_amd
    from kadan_amd import ops
    w = torch.zeros(n, k // 32 * 18, dtype=torch.uint8, device=device)
    x = torch.ones(m, k, dtype=torch.float16, device=device)
    y = torch.full((m, n), 1.0, dtype=torch.float16, device=device)
    ops.gemm_q4_0(w[:16], x[:1].contiguous(), 16)  # the kernels are loaded
    kadan_amd.call("kdq_release_scratch")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    ops.gemm_q4_0(w, x, n, out=y)
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] < 64 << 20
    assert not y.any()  # d = 0


def test_gemm_q4_0_rows_captured_in_a_small_workspace(device):
    """A shape that packs first, captured while the workspace holds its activations but not the
    weights' copy (which a capture cannot allocate): taken from the rows.  Each replay is
    within this file's tolerance of the eager result (the same fp16 weights and activations,
    summed in another order)."""
    torch = _torch()
    import kadan_amd
    from kadan_amd import ops
    m, k, n = 70, 2304, 2000
    _, _, wd, xd = _rows_case(device, m, k, n)
    xs = [xd, (xd * 0.5).contiguous(), xd.flip(0).contiguous()]
    eager = [ops.gemm_q4_0(wd, x, n).clone() for x in xs]
    torch.cuda.synchronize()
    kadan_amd.call("kdq_release_scratch")
    _, _, ws, xsmall = _rows_case(device, m, 512, 300)
    ops.gemm_q4_0(ws, xsmall, 300)  # the least workspace, 1 MiB: not the 2.6 MB copy
    static = xs[0].clone()
    out = torch.zeros(m, n, dtype=torch.float16, device=device)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.gemm_q4_0(wd, static, n, out=out)
    for i in (1, 0, 2, 2, 1):
        static.copy_(xs[i])
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert_close(out.float().cpu().numpy(), eager[i].float().cpu().numpy(), rel=1e-3,
                     mabs=2e-2, what=f"replay of input {i}")
        ops.gemm_q4_0(ws, xsmall, 300)  # eager work between replays, in the same workspace
