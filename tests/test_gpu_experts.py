"""GPU parity for the expert GEMMs (A5, A5', A6, A9) and the fused MoE block
(A11): bit-exact against the oracle's restatement of the limb arithmetic,
within tolerance against the reference W8A32 / FP32 numerics."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import hm_oracle as O
from conftest import assert_bitexact, assert_compare, normwise, oracle_by_token_chunks
from hmoe import capi, synth
from hmoe.block import DeviceExpertLayer, MoEBlock

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,inner,cols,limbs,zp", [
    (1, 2048, 768, 2, 0), (5, 2048, 64, 3, 0), (16, 768, 2048, 2, -3), (3, 129, 7, 1, 5),
    (2, 4097, 67, 3, -128)])
def test_limb_partials_exact(dev, rows, inner, cols, limbs, zp):
    """INT8 int32 partials: device digits and partials equal the oracle's
    brute-force int64 dot products bit for bit."""
    rng = np.random.default_rng(inner + cols)
    x = (rng.standard_normal((rows, inner)) * 2).astype(np.float32)
    q = rng.integers(-128, 128, (inner, cols)).astype(np.int8)
    digits, scales = O.limb_quantize(x, limbs)
    ddig = dev.empty((limbs, rows, inner), np.int8)
    dsc = dev.empty(rows, np.float32)
    dev.call("hm_limb_quantize_rows", dev.to(x).data_ptr(), rows, inner, limbs, ddig.data_ptr(),
             dsc.data_ptr(), dev.stream)
    assert_bitexact(dev.host(ddig), digits, "digits")
    assert_bitexact(dev.host(dsc), scales, "row scales")
    part = dev.empty((limbs, rows, cols), np.int32)
    qt = np.ascontiguousarray(q.T)  # packed [cols x inner]
    dev.call("hm_limb_partials", ddig.data_ptr(), rows, inner, limbs, dev.to(qt).data_ptr(), zp,
             cols, part.data_ptr(), dev.stream)
    expected = O.limb_partials(digits, q, zp)
    brute = np.einsum("lrk,kc->lrc", digits.astype(np.int64), q.astype(np.int64) - zp)
    assert_bitexact(expected, brute.astype(np.int32), "oracle partials vs brute force")
    assert_bitexact(dev.host(part), expected, "device partials")


PHASE23_SHAPES = [(1, 8, 8), (1, 257, 65), (2, 513, 33), (1, 1031, 31), (1, 2048, 768),
                  (1, 768, 2048), (3, 129, 7), (1, 4097, 67)]


@pytest.mark.parametrize("rows,inner,cols", PHASE23_SHAPES)
def test_w8a32_reference_inputs(dev, rows, inner, cols):
    """tests/phase23_tests.cpp:189-240: x=((i%29)-14)/29, q=((i*13)%255)-127,
    {0.003, -3}.  Reference mode is bit-exact with the CPU path; cooperative
    (split-K) within 1e-5 + 1e-5|ref| and of an independent double oracle."""
    i = np.arange(rows * inner)
    x = (((i % 29) - 14).astype(np.float32) / np.float32(29.0)).reshape(rows, inner)
    j = np.arange(inner * cols)
    q = (((j * 13) % 255) - 127).astype(np.int8).reshape(inner, cols)
    cpu = O.matmul_w8a32(x, q, 0.003, -3)
    for mode in (1, 2, 0):
        plan = capi.HmInt8GemmPlan()
        capi.call("hm_plan_int8_gemm", rows, inner, cols, mode, C.byref(plan))
        scratch = dev.empty(max(1, plan.scratch_elements), np.float32)
        y = dev.empty((rows, cols), np.float32)
        dev.call("hm_matmul_w8a32", dev.to(x).data_ptr(), dev.to(q).data_ptr(), 0.003, -3,
                 y.data_ptr(), rows, inner, cols, mode, scratch.data_ptr(),
                 scratch.numel() * 4, dev.stream)
        got = dev.host(y)
        if plan.implementation == 1:
            assert_bitexact(got, cpu, f"reference mode {rows}x{inner}x{cols}")
        assert_compare(got, cpu, 1e-5, 1e-5, f"mode {mode} vs CPU")
        w = (q.astype(np.float32) - np.float32(-3)) * np.float32(0.003)
        dbl = x.astype(np.float64) @ w.astype(np.float64)
        assert np.all(np.abs(got - dbl) <= 1e-5 + 1e-5 * np.abs(cpu))


# edges of the op-level kernels: 16-row and 32/64-column tiles, 16- and
# 32-wide K steps, fewer K steps than waves, row counts that pick each tile
OP_SHAPES = [(1, 1, 1), (1, 256, 64), (16, 31, 33), (17, 33, 31), (33, 257, 66), (65, 1000, 130),
             (150, 768, 2048), (300, 2048, 768), (333, 519, 1027), (1200, 64, 2050)]


def _op_call(dev, x, w, y, scale=None, zp=0):
    rows, inner, cols = x.shape[0], x.shape[1], w.shape[1]
    if scale is None:
        dev.call("hm_matmul_f32", x.data_ptr(), w.data_ptr(), y.data_ptr(), rows, inner, cols, dev.stream)
        return
    plan = capi.HmInt8GemmPlan()
    capi.call("hm_plan_int8_gemm", rows, inner, cols, 2, C.byref(plan))
    scratch = dev.empty(max(1, plan.scratch_elements), np.float32)
    dev.call("hm_matmul_w8a32", x.data_ptr(), w.data_ptr(), scale, zp, y.data_ptr(), rows, inner, cols, 2,
             scratch.data_ptr(), scratch.numel() * 4, dev.stream)


def _event_ms(call, n=5):
    import torch
    call()
    best = float("inf")
    for _ in range(n):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        call()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


@pytest.mark.parametrize("int8", [True, False])
@pytest.mark.parametrize("rows,inner,cols", OP_SHAPES)
def test_op_gemm_edges(dev, rows, inner, cols, int8):
    """The op-level products against 64-bit sums at the edges of their tiles and
    K steps, from operands off their vector alignment: each output within
    (K + 32) u sum |x w|, u = 2^-24 (K additions, at most 16 waves' sums and
    the scale, each rounding once)."""
    rng = np.random.default_rng(rows + inner + cols)
    x = (rng.standard_normal((rows, inner)) * np.exp2(rng.integers(-12, 12, (rows, inner)))).astype(np.float32)
    dx = dev.to(np.concatenate([np.zeros(1, np.float32), x.reshape(-1)]))[1:].view(rows, inner)
    y = dev.empty((rows, cols), np.float32)
    if int8:
        zp, scale = (-128, 127, 0)[(rows + cols) % 3], float(np.float32(0.0031))
        q = rng.integers(-128, 128, (inner, cols)).astype(np.int8)
        dw = dev.to(np.concatenate([np.zeros(1, np.int8), q.reshape(-1)]))[1:].view(inner, cols)
        _op_call(dev, dx, dw, y, scale, zp)
        w = (q.astype(np.float64) - zp) * scale
    else:
        wf = rng.standard_normal((inner, cols)).astype(np.float32)
        dw = dev.to(np.concatenate([np.zeros(1, np.float32), wf.reshape(-1)]))[1:].view(inner, cols)
        _op_call(dev, dx, dw, y)
        w = wf.astype(np.float64)
    got = dev.host(y)
    x64 = x.astype(np.float64)
    assert np.all(np.abs(got - x64 @ w) <= (inner + 32) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w)))


@pytest.mark.parametrize("int8", [True, False])
def test_op_gemm_special_values(dev, int8):
    """Non-finite operands reach exactly the outputs that the reference's loop
    gives them (also in the last K step, past which the operands are zero), and
    rows near the ends of the float range keep their 24 bits."""
    M, K, N = 35, 301, 70
    rng = np.random.default_rng(77)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[3, 5], x[4, 300], x[5, 7], x[33, 299] = np.inf, -np.inf, np.nan, np.inf
    x[6], x[7] = x[6] * np.float32(2.0 ** -100), x[7] * np.float32(2.0 ** 100)
    q = rng.integers(-127, 128, (K, N)).astype(np.int8)
    q[5, 9] = q[300, 11] = 0
    wf = (q.astype(np.float32) * np.float32(0.01)).astype(np.float32)
    if not int8:
        wf[300, 13], wf[2, 14] = np.inf, np.nan
    y = dev.empty((M, N), np.float32)
    _op_call(dev, dev.to(x), dev.to(q if int8 else wf), y, 0.01 if int8 else None)
    got = dev.host(y)
    with np.errstate(all="ignore"):
        ref = O.matmul_w8a32(x, q, 0.01, 0) if int8 else O.matmul_f32(x, wf)
    fine = np.isfinite(ref)
    assert_bitexact(np.isnan(got), np.isnan(ref), "NaN outputs")
    inf = ~fine & ~np.isnan(ref)
    assert_bitexact(got[inf], ref[inf], "infinite outputs")
    x64, w64 = np.where(np.isfinite(x), x, 0).astype(np.float64), np.where(np.isfinite(wf), wf, 0).astype(np.float64)
    bound = (K + 32) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64))
    if int8:
        w64 = q.astype(np.float64) * float(np.float32(0.01))
    assert np.all(np.abs(got - x64 @ w64)[fine] <= bound[fine])


def test_op_gemm_tiny_activations(dev):
    """Activations down to the smallest subnormal keep all their bits (times a
    scale that brings the results back to the middle of the range): within
    (K + 32) u sum |x w| of 64-bit sums, as any other row."""
    M, K, N = 40, 301, 70
    rng = np.random.default_rng(5)
    x = (rng.standard_normal((M, K)) * np.exp2(-109.0 - np.arange(M)[:, None])).astype(np.float32)
    q = rng.integers(-127, 128, (K, N)).astype(np.int8)
    scale = float(np.float32(0.011) * np.float32(2.0 ** 70))
    y = dev.empty((M, N), np.float32)
    _op_call(dev, dev.to(x), dev.to(q), y, scale, 3)
    x64, w64 = x.astype(np.float64), (q.astype(np.float64) - 3) * scale
    assert np.all(np.abs(dev.host(y) - x64 @ w64) <= (K + 32) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64)))


def test_op_gemm_scale_past_the_range(dev):
    """Weights (q - zp) * scale beyond the float range are infinite, as in the
    reference's loop, however small the activations."""
    M, K, N, zp = 20, 96, 40, -28
    rng = np.random.default_rng(6)
    x = (rng.standard_normal((M, K)) * 2.0 ** -60).astype(np.float32)
    x[2, 5] = 0.0
    q = rng.integers(-60, 60, (K, N)).astype(np.int8)
    q[5, 3], q[7, 9], q[5, 11], q[6, 11] = 100, 127, 110, 120
    scale = float(np.float32(2.0 ** 121))
    y = dev.empty((M, N), np.float32)
    _op_call(dev, dev.to(x), dev.to(q), y, scale, zp)
    got = dev.host(y)
    with np.errstate(all="ignore"):
        ref = O.matmul_w8a32(x, q, scale, zp)
    fine = np.isfinite(ref)
    assert not fine[:, [3, 9, 11]].any() and fine[:, 20].all()
    assert_bitexact(np.isnan(got), np.isnan(ref), "NaN outputs")
    assert_bitexact(got[np.isinf(ref)], ref[np.isinf(ref)], "infinite outputs")
    x64, w64 = x.astype(np.float64), (q.astype(np.float64) - zp) * scale
    assert np.all((np.abs(got - x64 @ w64) <= (K + 32) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64)))[fine])


def test_op_gemm_nonfinite_rows_keep_the_speed(dev):
    """Outputs that are not finite come from the matrix cores too: a call whose
    every output is infinite takes no more than ten times the finite one's time
    (one lane summing over K in turn took hundreds of times)."""
    M, K, N = 300, 2048, 768
    rng = np.random.default_rng(8)
    x = rng.standard_normal((M, K)).astype(np.float32)
    q, y = dev.to(rng.integers(1, 128, (K, N)).astype(np.int8)), dev.empty((M, N), np.float32)
    dx = dev.to(x)
    x[:, 17] = np.inf
    dinf = dev.to(x)
    fine = _event_ms(lambda: _op_call(dev, dx, q, y, 0.01))
    inf = _event_ms(lambda: _op_call(dev, dinf, q, y, 0.01))
    print(f"[gpu] finite {fine:.3f} ms, infinite {inf:.3f} ms", flush=True)
    assert np.isposinf(dev.host(y)).all()
    assert inf < 10 * fine


def test_matmul_f32_closed_form(dev):
    """tests/phase5_tests.cpp:147-160: [[1,2,3],[4,5,6]] x [[7,8],[9,10],[11,12]]."""
    a = np.array([[1, 2, 3], [4, 5, 6]], np.float32)
    b = np.array([[7, 8], [9, 10], [11, 12]], np.float32)
    y = dev.empty((2, 2), np.float32)
    dev.call("hm_matmul_f32", dev.to(a).data_ptr(), dev.to(b).data_ptr(), y.data_ptr(), 2, 3, 2,
             dev.stream)
    assert dev.host(y).tolist() == [[58, 64], [139, 154]]


def test_elementwise(dev):
    """SiLU bit-exact with Activation.cpp:44 (glibc expf); mul/add exact."""
    rng = np.random.default_rng(3)
    x = (rng.standard_normal(100003) * 8).astype(np.float32)
    b = rng.standard_normal(100003).astype(np.float32)
    y = dev.empty(x.shape, np.float32)
    dev.call("hm_silu", dev.to(x).data_ptr(), y.data_ptr(), x.size, dev.stream)
    assert_bitexact(dev.host(y), O.silu(x), "silu")
    dev.call("hm_mul", dev.to(x).data_ptr(), dev.to(b).data_ptr(), y.data_ptr(), x.size, dev.stream)
    assert_bitexact(dev.host(y), x * b, "mul")
    dev.call("hm_add", dev.to(x).data_ptr(), dev.to(b).data_ptr(), y.data_ptr(), x.size, dev.stream)
    assert_bitexact(dev.host(y), x + b, "add")


def _tiles(w_kn: np.ndarray) -> np.ndarray:
    """The kernels' INT8 tile layout of one projection W [K x N] (K inner):
    zero-padded to multiples of 32, tile (n // 32, k // 32) at
    ((n // 32) * K32/32 + k // 32) KB, inside it lane n % 32 + 32 ((k // 16) % 2)
    holding the 16 bytes k % 16 = 0..15."""
    K, N = w_kn.shape
    K32, N32 = -(-K // 32) * 32, -(-N // 32) * 32
    p = np.zeros((K32, N32), np.int8)
    p[:K, :N] = w_kn
    t = p.reshape(K32 // 32, 2, 16, N32 // 32, 32)     # kb, half, j, cb, col
    return np.ascontiguousarray(t.transpose(3, 0, 1, 4, 2)).reshape(-1)  # cb, kb, half, col, j


@pytest.mark.parametrize("E,H,I", [(3, 40, 70), (2, 2048, 768)])
def test_pack_layer_tile_layout(dev, E, H, I):
    """hm_pack_layer writes every INT8 projection as 32 x 32 tiles in the MFMA
    B-operand order (one wave-wide 16-byte load = one contiguous kilobyte),
    projections gate | up | down of each expert back to back, padding zero."""
    rng = np.random.default_rng(E * H)
    payload = rng.integers(-128, 128, (E, 3, H * I)).astype(np.int8)
    nbytes = capi.load().hm_packed_layer_bytes(E, H, I, capi.HM_DTYPE_INT8)
    packed = dev.empty(nbytes, np.uint8)
    dev.call("hm_pack_layer", dev.to(payload).data_ptr(), E, H, I, capi.HM_DTYPE_INT8,
             packed.data_ptr(), dev.stream)
    got = dev.host(packed).view(np.int8)
    expected = np.concatenate([
        _tiles(payload[e, p].reshape(H, I) if p < 2 else payload[e, p].reshape(I, H))
        for e in range(E) for p in range(3)])
    assert_bitexact(got, expected, "tile layout")


def _layer_inputs(seed, T, H, E, I, int8, skew=False):
    payload, scale, zp = synth.expert_layer(seed, 0, E, H, I, int8)
    h = O.rmsnorm(synth.raw_hidden(seed, T, H), np.ones(H, np.float32))
    w = synth.router_weights(seed, 0, H, E)
    if skew:
        synth.apply_skew(h, w, synth.zipf_bias(seed, E))
    return payload, scale, zp, h, w


BLOCK_CASES = [  # (T, H, E, I, k, X digits, Z digits) -- MFMA shapes and generic shapes
    (1, 2048, 128, 768, 8, 2, 3), (4, 2048, 128, 768, 8, 3, 3), (16, 2048, 128, 768, 8, 2, 2),
    (70, 512, 16, 256, 4, 2, 3), (5, 64, 8, 32, 2, 2, 2), (6, 96, 5, 40, 3, 3, 3), (3, 2, 3, 2, 2, 2, 3),
    # several row tiles per expert (ragged last tile) through the MFMA kernels
    (300, 2048, 4, 768, 2, 2, 3), (300, 2048, 4, 768, 2, 3, 2), (203, 1024, 3, 384, 2, 3, 3),
    (90, 1024, 6, 512, 3, 2, 3), (150, 512, 2, 128, 1, 1, 1), (300, 512, 4, 256, 2, 2, 3),
    # more than 1024 pairs with E % 64 == 0: the prefill router's select
    # kernel counts the permutation's chunk histograms (the count pass is
    # skipped)
    (160, 2048, 64, 768, 8, 2, 3), (160, 512, 64, 256, 8, 2, 2)]


# shapes off the ring kernel's tile grid: K with one or two 32-wide tiles in
# its last 64-byte stage, exactly four stages, fewer columns than a tile,
# ragged last column blocks, widths off 4 (the scalar SwiGLU) and past 2048
RAGGED_CASES = [
    (70, 1024, 60, 704, 4, 2, 3), (45, 320, 5, 272, 2, 3, 2), (150, 448, 9, 336, 3, 2, 3),
    (40, 225, 4, 1000, 2, 1, 3), (33, 608, 6, 450, 3, 2, 1), (130, 256, 3, 2052, 2, 2, 3),
    (90, 200, 4, 198, 2, 2, 2)]


@pytest.mark.parametrize("T,H,E,I,k,LX,LZ", RAGGED_CASES)
def test_block_int8_ragged_tiles(dev, T, H, E, I, k, LX, LZ):
    """Shapes off the tile grid run the ring kernels too: the same bits as the
    limb oracle, as the generic kernels (what they ran before), and with the
    split-K kernel taking the small groups; zero points other than zero, and a
    workspace full of other values (pad digits must come from the quantisers)."""
    print(f"[gpu] ragged int8 T={T} H={H} E={E} I={I} k={k} limbs=({LX}, {LZ})", flush=True)
    payload, scale, zp, h, w = _layer_inputs(61 + T, T, H, E, I, True)
    zp = np.random.default_rng(T).integers(-20, 21, zp.shape).astype(np.int32)
    block = MoEBlock(DeviceExpertLayer(payload, scale, zp, H, I), k, limbs_x=LX, limbs_z=LZ)
    block.execute_batch(dev.to(h), dev.to(w), exec_flags=capi.HM_EXEC_LIMBS)
    block._ws.fill_(0x55)
    res = block.execute_batch(dev.to(h), dev.to(w), exec_flags=capi.HM_EXEC_LIMBS)
    out = dev.host(res.output)
    lout, lids, _ = O.moe_block_limbs(payload, scale, zp, h, w, k, I, LX, LZ)
    assert_bitexact(res.ids, lids, "ids")
    assert_bitexact(out, lout, "block output vs limb oracle")
    for flags in (capi.HM_EXEC_GENERIC, capi.HM_EXEC_LIMBS | capi.HM_EXEC_SPLIT_K):
        other = block.execute_batch(dev.to(h), dev.to(w), exec_flags=flags)
        assert_bitexact(dev.host(other.output), out, f"exec flags {flags:#x}")
        assert_bitexact(dev.host(other.expert_out), dev.host(res.expert_out), f"expert rows, flags {flags:#x}")


@pytest.mark.parametrize("T,H,E,I,k,LX,LZ", BLOCK_CASES)
def test_block_int8_bitexact_vs_limb_oracle(dev, T, H, E, I, k, LX, LZ):
    print(f"[gpu] block int8 T={T} H={H} E={E} I={I} k={k} limbs=({LX}, {LZ})", flush=True)
    payload, scale, zp, h, w = _layer_inputs(11 + T, T, H, E, I, True)
    layer = DeviceExpertLayer(payload, scale, zp, H, I)
    block = MoEBlock(layer, k, limbs_x=LX, limbs_z=LZ)
    # the limb arithmetic at every batch size (decode sizes default to the GEMV)
    res = block.execute_batch(dev.to(h), dev.to(w), exec_flags=capi.HM_EXEC_LIMBS)
    out = dev.host(res.output)
    lout, lids, lsc = O.moe_block_limbs(payload, scale, zp, h, w, k, I, LX, LZ)
    assert_bitexact(res.ids, lids, "ids")
    assert_bitexact(res.scores, lsc, "scores")
    assert_bitexact(out, lout, "block output vs limb oracle")
    # generic (scalar) kernels give the same bits
    res2 = block.execute_batch(dev.to(h), dev.to(w), exec_flags=capi.HM_EXEC_GENERIC)
    assert_bitexact(dev.host(res2.output), out, "MFMA vs generic kernels")
    if T <= capi.HM_GEMV_MAX_TOKENS:
        # the default decode path: the W8A32 GEMV in FP32 up to
        # HM_GEMV_MAX_PAIRS pairs (against the reference), the limb GEMMs
        # beyond (the same bits as above)
        rout_, _, _ = O.moe_block(payload, scale, zp, h, w, k, I)
        gres = block.execute_batch(dev.to(h), dev.to(w))
        assert_bitexact(gres.ids, res.ids, "default decode path routing")
        if T * k <= capi.HM_GEMV_MAX_PAIRS:
            assert_compare(dev.host(gres.output), rout_, 1e-4, 1e-4,
                           "GEMV block vs reference (1e-4)")
        else:
            assert_bitexact(dev.host(gres.output), out, "default decode path vs limb GEMMs")
    # reference W8A32 numerics
    rout, rids, rsc = O.moe_block(payload, scale, zp, h, w, k, I)
    assert_bitexact(res.ids, rids, "ids vs reference path")
    counts, offsets, ptok, pw, _ = O.group(rids, rsc, E)
    assert_bitexact(res.perm_tokens, ptok, "permutation vs reference path")
    nw = normwise(out, rout)
    if min(LX, LZ) == 1:  # one digit = plain int8 activations: W8A8 accuracy
        assert nw < 5e-2
    elif LX >= 2 and LZ >= 3:
        # the block's default digit counts
        assert_compare(out, rout, 1e-4, 1e-4, "block vs reference W8A32 (1e-4)")
        assert nw < 1e-4
        if LX == 3:
            assert_compare(out, rout, 1e-5, 1e-5, "three-digit block vs reference W8A32 (1e-5)")
    else:  # two Z digits with one scale per row: about 16-bit Z
        assert nw < 3e-4


@pytest.mark.parametrize("T,H,E,I,k,LX,LZ,skew", [
    (400, 1024, 16, 512, 4, 2, 3, True), (256, 2048, 128, 768, 8, 3, 3, False),
    (256, 512, 32, 256, 8, 1, 2, True)])
def test_block_skinny_split_k(dev, T, H, E, I, k, LX, LZ, skew):
    """With HM_EXEC_SPLIT_K, experts of at most 32 grouped rows run the
    bounded split-K kernel (K split over the workgroup's waves, int32 limb
    partials summed exactly), the others the tile kernels, in one block: a
    skewed batch with both kinds, a mid-size batch where most experts are
    skinny, one to three digit planes.  Bit-exact against the limb oracle,
    against the generic kernels and against the tile kernels alone."""
    print(f"[gpu] skinny split-K T={T} H={H} E={E} I={I} k={k} limbs=({LX}, {LZ})", flush=True)
    payload, scale, zp, h, w = _layer_inputs(41 + T, T, H, E, I, True, skew=skew)
    block = MoEBlock(DeviceExpertLayer(payload, scale, zp, H, I), k, limbs_x=LX, limbs_z=LZ)
    res = block.execute_batch(dev.to(h), dev.to(w),
                              exec_flags=capi.HM_EXEC_LIMBS | capi.HM_EXEC_SPLIT_K)
    counts = np.asarray(res.counts)
    assert ((counts > 0) & (counts <= 32)).any(), "no skinny group in this batch"
    if skew:
        assert (counts > 32).any(), "no tiled group in this batch"
    out = dev.host(res.output)
    lout, lids, _ = O.moe_block_limbs(payload, scale, zp, h, w, k, I, LX, LZ)
    assert_bitexact(res.ids, lids, "ids")
    assert_bitexact(out, lout, "split-K block vs limb oracle")
    gen = block.execute_batch(dev.to(h), dev.to(w), exec_flags=capi.HM_EXEC_GENERIC)
    assert_bitexact(dev.host(gen.output), out, "split-K kernels vs generic kernels")
    tiles = block.execute_batch(dev.to(h), dev.to(w), exec_flags=capi.HM_EXEC_LIMBS)
    assert_bitexact(dev.host(tiles.output), out, "split-K kernels vs tile kernels")


def test_block_int8_nonzero_zero_points(dev):
    """Zero points other than 0 (validateParameters allows [-128, 127])."""
    T, H, E, I, k = 24, 2048, 8, 768, 2
    payload, scale, zp, h, w = _layer_inputs(5, T, H, E, I, True)
    zp = np.random.default_rng(1).integers(-5, 6, zp.shape).astype(np.int32)
    layer = DeviceExpertLayer(payload, scale, zp, H, I)
    block = MoEBlock(layer, k, limbs_x=2, limbs_z=3)
    out = dev.host(block.execute_batch(dev.to(h), dev.to(w)).output)
    lout, _, _ = O.moe_block_limbs(payload, scale, zp, h, w, k, I, 2, 3)
    assert_bitexact(out, lout, "block with zero points vs limb oracle")
    # decode-size batch with zero points through the GEMV
    hs = np.ascontiguousarray(h[:5])
    gout = dev.host(block.execute_batch(dev.to(hs), dev.to(w)).output)
    rout, _, _ = O.moe_block(payload, scale, zp, hs, w, k, I)
    assert_compare(gout, rout, 1e-4, 1e-4, "GEMV with zero points vs reference (1e-4)")
    gen = block.execute_batch(dev.to(h), dev.to(w), exec_flags=capi.HM_EXEC_GENERIC)
    assert_bitexact(dev.host(gen.output), out, "MFMA vs generic with zero points")


@pytest.mark.parametrize("T,H,E,I,k,skew", [
    (1, 2048, 128, 768, 8, False), (4, 2048, 128, 768, 8, False), (8, 2048, 128, 768, 8, True),
    (16, 512, 4, 256, 2, False), (13, 1024, 3, 512, 3, False), (9, 256, 2, 1024, 1, False),
    (16, 256, 64, 1024, 4, False), (5, 528, 6, 400, 2, False), (2, 2048, 128, 768, 8, False),
    (3, 256, 8, 96, 5, False), (1, 1024, 16, 512, 1, False), (1, 128, 4, 32, 1, False),
    (3, 1024, 16, 512, 8, False)])
def test_block_gemv_decode(dev, T, H, E, I, k, skew):
    """Decode-size blocks of at most HM_GEMV_MAX_PAIRS pairs take the W8A32
    GEMV (FP32): ids bit-exact, output
    within 1e-4 of the reference; several rows per expert (the register
    row blocks), skewed groups, every supported K length, the four-column-
    tile down workgroups (32 or more active experts) at their largest K, and
    H, I off the 32-column tile grid (zero-padded K tiles, a partial last
    column tile).  With T*k <= 16 the down projection and the combine run as
    one kernel: one active expert (sixteen waves on its K range; with I=32
    fifteen of them have no K tile), eight, and sixteen (one wave per
    expert, K in two register chunks).  Three tokens at top-8 over sixteen
    experts (24 pairs) take the separate down GEMV and combine with twelve
    to sixteen active experts."""
    print(f"[gpu] gemv T={T} H={H} E={E} I={I} k={k} skew={skew}", flush=True)
    payload, scale, zp, h, w = _layer_inputs(7 + T, T, H, E, I, True, skew=skew)
    block = MoEBlock(DeviceExpertLayer(payload, scale, zp, H, I), k)
    res = block.execute_batch(dev.to(h), dev.to(w))
    rout, rids, rsc = O.moe_block(payload, scale, zp, h, w, k, I)
    assert_bitexact(res.ids, rids, "ids")
    assert_bitexact(res.scores, rsc, "scores")
    out = dev.host(res.output)
    assert_compare(out, rout, 1e-4, 1e-4, "GEMV block vs reference W8A32 (1e-4)")
    assert normwise(out, rout) < 1e-5
    # per-expert outputs: the grouped rows equal the reference expert MLP
    y = dev.host(res.expert_out)
    for b in res.batches[:4]:
        lo = int(res.offsets[b.expert_id])
        xe = np.ascontiguousarray(h[b.token_indices])
        ref = O.expert_mlp(payload, scale, zp, b.expert_id, xe, I)
        assert_compare(y[lo:lo + len(b.token_indices)], ref, 1e-4, 1e-4, "expert rows")


@pytest.mark.parametrize("T,skew", [(16, True), (9, False)])
def test_block_limb_decode(dev, T, skew):
    """Decode-size blocks of more than HM_GEMV_MAX_PAIRS pairs (C3-16: 128
    pairs over about 80 experts) take the limb GEMMs, their activation digits
    cut by the fused decode router's select kernel: output bit-exact against
    the limb oracle and within 1e-4 of the reference, routing and grouping
    bit-exact."""
    H, E, I, k = 2048, 128, 768, 8
    assert T * k > capi.HM_GEMV_MAX_PAIRS
    print(f"[gpu] limb decode T={T} skew={skew}", flush=True)
    payload, scale, zp, h, w = _layer_inputs(29 + T, T, H, E, I, True, skew=skew)
    block = MoEBlock(DeviceExpertLayer(payload, scale, zp, H, I), k)
    res = block.execute_batch(dev.to(h), dev.to(w))
    lout, lids, lsc = O.moe_block_limbs(payload, scale, zp, h, w, k, I, block.limbs_x,
                                        block.limbs_z)
    assert_bitexact(res.ids, lids, "ids")
    assert_bitexact(res.scores, lsc, "scores")
    out = dev.host(res.output)
    assert_bitexact(out, lout, "block output vs limb oracle")
    _, _, ptok, _, _ = O.group(lids, lsc, E)
    assert_bitexact(res.perm_tokens, ptok, "grouping")
    rout, _, _ = O.moe_block(payload, scale, zp, h, w, k, I)
    assert_compare(out, rout, 1e-4, 1e-4, "limb decode block vs reference W8A32 (1e-4)")


@pytest.mark.parametrize("T,E", [(16, 64), (1, 64), (5, 8), (40, 8), (300, 4)])
def test_block_fp32_vs_reference(dev, T, E):
    """FP32 experts (C1 shape): within 1e-3 of the reference (north star).
    T <= 16 takes the FP32 GEMV (T = 5, E = 8: five rows on most experts,
    two LDS passes); T=300 with E=4, k=2 puts about 150 rows on each
    expert: several 64-row matrix-core tiles per expert with a ragged last
    tile."""
    H, I, k = 2048, 768, 8 if E >= 8 else 2
    print(f"[gpu] fp32 block T={T} E={E} k={k}", flush=True)
    payload, scale, zp, h, w = _layer_inputs(3, T, H, E, I, False)
    layer = DeviceExpertLayer(payload, None, None, H, I)
    block = MoEBlock(layer, k)
    res = block.execute_batch(dev.to(h), dev.to(w))
    rout, rids, rsc = oracle_by_token_chunks(O.moe_block, h, payload, scale, zp, w, k, I)
    assert_bitexact(res.ids, rids, "ids")
    assert_bitexact(res.scores, rsc, "scores")
    if T > 64:
        assert int(np.bincount(rids.ravel(), minlength=E).max()) > 64
    assert_compare(dev.host(res.output), rout, 1e-3, 1e-3, "fp32 block (1e-3)")
    assert normwise(dev.host(res.output), rout) < 1e-5


def test_block_c4_prefill_properties(dev):
    """C4 at full size (T=4096, skewed): routing bit-exact against the
    oracle, MFMA == generic on a token subset is covered above; here:
    determinism across runs, finite output, and exact linearity of the
    combine over a duplicated batch."""
    cfg = synth.CONFIGS["C4"]
    T, H, E, I, k = cfg.tokens, cfg.hidden, cfg.experts, cfg.inter, cfg.top_k
    payload, scale, zp, h, w = _layer_inputs(cfg.seed, T, H, E, I, True, skew=True)
    layer = DeviceExpertLayer(payload, scale, zp, H, I)
    block = MoEBlock(layer, k, limbs_x=2, limbs_z=3)
    r1 = block.execute_batch(dev.to(h), dev.to(w))
    o1 = dev.host(r1.output).copy()
    r2 = block.execute_batch(dev.to(h), dev.to(w))
    assert_bitexact(dev.host(r2.output), o1, "run-to-run determinism")
    assert np.isfinite(o1).all()
    rc, ids, scores = O.route(h, w, k, 1, 1)
    assert_bitexact(r1.ids, ids, "C4 ids")
    assert_bitexact(r1.scores, scores, "C4 scores")
    # the permutation (its chunk histograms counted by the prefill select
    # kernel at this size) against the oracle's grouping, bit for bit
    counts, offsets, ptok, pw, _ = O.group(ids, scores, E)
    assert_bitexact(r1.offsets, offsets, "C4 offsets")
    assert_bitexact(r1.perm_tokens, ptok, "C4 permutation")
    assert_bitexact(r1.perm_weights, pw, "C4 permuted weights")
    # a token's output depends only on its own row: a 64-token slice run alone
    # gives the same bits (routing, permutation and tiling are per token/row)
    sub = slice(1000, 1064)
    r3 = block.execute_batch(dev.to(np.ascontiguousarray(h[sub])), dev.to(w))
    assert_bitexact(dev.host(r3.output), o1[sub], "token-slice invariance")
    lout, _, _ = O.moe_block_limbs(payload, scale, zp, np.ascontiguousarray(h[sub]), w, k, I, 2, 3)
    assert_bitexact(o1[sub], lout, "C4 slice vs limb oracle")
    # every token against the reference W8A32 block
    rout, _, _ = oracle_by_token_chunks(O.moe_block, h, payload, scale, zp, w, k, I)
    assert_compare(o1, rout, 1e-4, 1e-4, "C4 full batch vs reference W8A32 (1e-4)")
    nw = normwise(o1, rout)
    print(f"[gpu] C4 full batch normwise error {nw:.3e}", flush=True)
    assert nw < 1e-4


@pytest.mark.parametrize("T,E,k", [(2, 64, 32), (13, 70, 5), (3, 22, 22), (16, 128, 8), (16, 200, 13), (16, 64, 64)])
@pytest.mark.parametrize("int8", [False, True])
def test_block_decode_groups(dev, T, E, k, int8):
    """The decode step's grouping by the workgroup that arrives last: 64 pairs,
    65 and 66, whole and ragged runs of 64, and the most there are (1024), over
    one to four rows of experts, with the pairs of the popular experts spread
    over all the runs; bit-exact against the oracle's grouping."""
    print(f"[gpu] decode groups T={T} E={E} k={k} int8={int8}", flush=True)
    H, I = 64, 32
    payload, scale, zp, h, w = _layer_inputs(5 + E, T, H, E, I, int8, skew=True)
    layer = DeviceExpertLayer(payload, scale if int8 else None, zp if int8 else None, H, I)
    res = MoEBlock(layer, k).execute_batch(dev.to(h), dev.to(w))
    rc, ids, scores = O.route(h, w, k, 1, 1)
    assert rc == 0
    counts, offsets, ptok, pw, _ = O.group(ids, scores, E)
    assert_bitexact(res.ids, ids, "ids")
    assert_bitexact(res.scores, scores, "scores")
    assert_bitexact(res.counts, counts, "counts")
    assert_bitexact(res.offsets, offsets, "offsets")
    assert_bitexact(res.perm_tokens, ptok, "permutation")
    assert_bitexact(res.perm_weights, pw, "permuted weights")


def test_block_one_token_select_at_rounding_boundaries(dev):
    """One token on the GEMV path: every workgroup of the gate/up launch
    redoes the select (select_gateup_kernel).  Logits the bound cannot
    settle (experts 0-3: 1 + 2^-24, an exact tie that rounds to 1.0) take
    the reference's chain inside that kernel; ids and scores bit-exact
    against the reference, the output within 1e-4, and the sequential-chain
    flag gives the same bits."""
    from hmoe import capi
    H, E, I, k = 256, 64, 64, 2
    rng = np.random.default_rng(5)
    payload, scale, zp = synth.expert_layer(21, 0, E, H, I, True)
    h = np.zeros((1, H), np.float32)
    w = np.zeros((H, E), np.float32)
    h[0, 0], h[0, 1] = 1.0, 2.0 ** -24
    h[0, 2:] = rng.standard_normal(H - 2).astype(np.float32)
    w[0, :], w[1, :] = 1.0, 1.0
    w[2:, 4:] = (0.02 * rng.standard_normal((H - 2, E - 4))).astype(np.float32)
    block = MoEBlock(DeviceExpertLayer(payload, scale, zp, H, I), k)
    res = block.execute_batch(dev.to(h), dev.to(w))
    rout, rids, rsc = O.moe_block(payload, scale, zp, h, w, k, I)
    assert_bitexact(res.ids, rids, "ids")
    assert_bitexact(res.scores, rsc, "scores")
    out = dev.host(res.output)
    assert_compare(out, rout, 1e-4, 1e-4, "one-token block vs reference (1e-4)")
    seq = block.execute_batch(dev.to(h), dev.to(w), exec_flags=capi.HM_EXEC_ROUTE_SEQUENTIAL)
    assert_bitexact(seq.ids, res.ids, "ids, sequential chains")
    assert_bitexact(dev.host(seq.output), out, "output, sequential chains")


def test_block_one_token_nonfinite_score(dev):
    """A non-finite router score at one token (the select inside the gate/up
    launch) sets HM_STATUS_NONFINITE_SCORE, as CpuRouterBackend.cpp:47
    throws; the block raises, and the next call on clean weights is right."""
    H, E, I, k = 256, 64, 64, 2
    payload, scale, zp, h, w = _layer_inputs(23, 1, H, E, I, True)
    block = MoEBlock(DeviceExpertLayer(payload, scale, zp, H, I), k)
    bad = w.copy()
    bad[3, 5] = np.inf
    from hmoe import capi
    with pytest.raises(RuntimeError, match="status bits") as err:
        block.execute_batch(dev.to(h), dev.to(bad))
    bits = int(str(err.value).split("status bits ")[1].rstrip(")"), 16)
    assert bits & capi.HM_STATUS_NONFINITE_SCORE
    res = block.execute_batch(dev.to(h), dev.to(w))
    rout, rids, _ = O.moe_block(payload, scale, zp, h, w, k, I)
    assert_bitexact(res.ids, rids, "ids after the failed call")
    assert_compare(dev.host(res.output), rout, 1e-4, 1e-4, "output after the failed call")


@pytest.mark.parametrize("T,H,E,I,k,skew", [
    (17, 128, 3, 64, 2, False), (64, 256, 1, 128, 1, False), (65, 128, 1, 64, 1, False),
    (130, 1024, 4, 192, 1, True), (250, 2048, 16, 768, 4, True)])
def test_block_fp32_split_tiles(dev, T, H, E, I, k, skew):
    """FP32 experts on the split bf16 tiles: fragment and tile edges (16, 64, 65
    rows of an expert, one K stage of slack, fewer tiles than XCDs).  An expert
    output is two chained sums: within (H + I + 64) 2^-22 of the absolute sums
    (a product's left-out parts are below 2^-32, each FP32 addition 2^-24)."""
    print(f"[gpu] fp32 split T={T} H={H} E={E} I={I}", flush=True)
    payload, scale, zp, h, w = _layer_inputs(5 + T, T, H, E, I, False, skew=skew)
    block = MoEBlock(DeviceExpertLayer(payload, scale, zp, H, I), k)
    res = block.execute_batch(dev.to(h), dev.to(w))
    got = dev.host(res.expert_out).astype(np.float64)
    P = payload.astype(np.float64)
    for b in res.batches:
        x = h[b.token_indices].astype(np.float64)
        g, u, d = (P[b.expert_id, j].reshape(s) for j, s in enumerate([(H, I), (H, I), (I, H)]))
        gg, uu = x @ g, x @ u
        z = gg / (1 + np.exp(-gg)) * uu
        zabs = (np.abs(x) @ np.abs(g)) * (np.abs(x) @ np.abs(u)) + np.abs(z)
        lo = res.offsets[b.expert_id]
        rows = got[lo:lo + len(x)]
        assert np.all(np.abs(rows - z @ d) <= (H + I + 64) * 2.0 ** -22 * (zabs @ np.abs(d)))
        err = np.linalg.norm(rows - z @ d) / np.linalg.norm(z @ d)
        assert err < 1e-6, err


def test_block_fp32_nonfinite_values(dev):
    """Non-finite activations and weights reach exactly the expert outputs that
    the reference's sums give them (their bf16 parts are no numbers: those sums
    are redone)."""
    T, H, E, I, k = 40, 128, 2, 64, 2
    payload, scale, zp, h, w = _layer_inputs(9, T, H, E, I, False)
    h = h.copy()
    w = w.copy()
    w[3:6] = 0                               # the router does not read the features below
    h[:, 3:6] = 0.5
    payload = payload.copy()
    payload[1, 0].reshape(H, I)[4, 7] = np.inf
    payload[0, 2].reshape(I, H)[9, 11] = np.nan
    layer = DeviceExpertLayer(payload, scale, zp, H, I)
    res = MoEBlock(layer, k).execute_batch(dev.to(h), dev.to(w))
    got = dev.host(res.expert_out)
    with np.errstate(all="ignore"):
        for b in res.batches:
            x = h[b.token_indices]
            e = b.expert_id
            g, u = O.matmul_f32(x, payload[e, 0].reshape(H, I)), O.matmul_f32(x, payload[e, 1].reshape(H, I))
            ref = O.matmul_f32(O.silu(g) * u, payload[e, 2].reshape(I, H))
            rows = got[res.offsets[e]:res.offsets[e] + len(x)]
            assert_bitexact(np.isnan(rows), np.isnan(ref), "NaN outputs")
            inf = np.isinf(ref)
            assert_bitexact(rows[inf], ref[inf], "infinite outputs")
            fine = np.isfinite(ref)
            assert np.allclose(rows[fine], ref[fine], rtol=1e-4, atol=1e-5)


def _one_term_layer(t, d):
    """One FP32 expert of H = len(d), I = 64 for one-hot rows: feature r gives
    the intermediate value t[r] in column 0 (silu(32) = 32 times t[r] / 32) and 0
    in the others, and the output is the single product t[r] * d[n]."""
    H, I = len(d), 64
    payload = np.zeros((1, 3, H * I), np.float32)
    payload[0, 0].reshape(H, I)[:, 0] = 32.0
    payload[0, 1].reshape(H, I)[:, 0] = t / np.float32(32.0)
    payload[0, 2].reshape(I, H)[0] = d
    return DeviceExpertLayer(payload, None, None, H, I)


def test_block_fp32_one_term_sums(dev):
    """An expert sum of a single product is that product, rounded once: a
    product's parts left out and the small parts' own roundings are below 2^-6
    of a rounding.  Values with all 24 bits, among them those whose low parts
    are largest."""
    T = H = 128
    rng = np.random.default_rng(12)
    t = (1 + rng.random(H)).astype(np.float32)
    d = (1 + rng.random(H)).astype(np.float32) * rng.choice([-1, 1], H).astype(np.float32)
    t[:2], d[:2] = np.float32(1 + 2.0 ** -7 - 2.0 ** -23), np.float32(1 + 2.0 ** -7 - 2.0 ** -23)
    t[2:4], d[2:4] = np.float32(1 + 2.0 ** -8 - 2.0 ** -16), np.float32(-1 - 2.0 ** -8 + 2.0 ** -23)
    w = rng.standard_normal((H, 1)).astype(np.float32)
    res = MoEBlock(_one_term_layer(t, d), 1).execute_batch(dev.to(np.eye(T, H, dtype=np.float32)), dev.to(w))
    exact = t.astype(np.float64)[:, None] * d.astype(np.float64)
    assert np.all(np.abs(dev.host(res.expert_out) - exact) <= 2.0 ** -24 * (1 + 2.0 ** -6) * np.abs(exact))


def test_block_fp32_tiny_values(dev):
    """Operands down to the smallest subnormal keep all their bits in a product
    of normal size, and operands up to the largest float theirs."""
    T = H = 128
    rng = np.random.default_rng(13)
    t = np.ldexp((1 + rng.random(H)).astype(np.float32), np.arange(H) * 2 - 144)   # 2^-144 .. 2^110
    t = np.float32(32) * (t / np.float32(32))
    d = np.ldexp((1 + rng.random(H)).astype(np.float32), 126 - np.arange(H) * 2)   # 2^126 .. 2^-128
    w = rng.standard_normal((H, 1)).astype(np.float32)
    res = MoEBlock(_one_term_layer(t, d), 1).execute_batch(dev.to(np.eye(T, H, dtype=np.float32)), dev.to(w))
    got = dev.host(res.expert_out).astype(np.float64)
    exact = t.astype(np.float64)[:, None] * d.astype(np.float64)
    normal = (np.abs(exact) < 2.0 ** 127) & (np.abs(exact) > 2.0 ** -100)
    assert normal.sum() > H * H // 2
    assert np.all((np.abs(got - exact) <= 2.0 ** -24 * (1 + 2.0 ** -6) * np.abs(exact))[normal])


def test_block_fp32_nonfinite_values_keep_the_speed(dev):
    """Experts whose every sum is NaN take no more than ten times the time of
    finite ones (one lane summing over K in turn took hundreds of times)."""
    T, H, E, I, k = 512, 1024, 8, 512, 2
    payload, scale, zp, h, w = _layer_inputs(3, T, H, E, I, False)
    dh, dw = dev.to(h), dev.to(w)
    bad = payload.copy()
    bad[:, 0].reshape(E, H, I)[:, 5] = np.nan
    blocks = [MoEBlock(DeviceExpertLayer(p, scale, zp, H, I), k) for p in (payload, bad)]
    ms = [_event_ms(lambda: b.launch(dh, dw)) for b in blocks]
    print(f"[gpu] finite {ms[0]:.3f} ms, NaN {ms[1]:.3f} ms", flush=True)
    assert np.isnan(dev.host(blocks[1].launch(dh, dw)["expert_out"])).all()
    assert ms[1] < 10 * ms[0]


@pytest.mark.parametrize("T", [1, 16, 300])
def test_block_graph_replay(dev, T):
    """The block's launch sequence captured as one HIP graph (kernels only:
    no memset or copy nodes) replays to the eager result every time, with
    eager work and synchronisations between the replays."""
    import torch
    print(f"[gpu] graph replay T={T}", flush=True)
    H, E, I, k = 2048, 128, 768, 8
    payload, scale, zp, h, w = _layer_inputs(31 + T, T, H, E, I, True)
    block = MoEBlock(DeviceExpertLayer(payload, scale, zp, H, I), k)
    dh, dw = dev.to(h), dev.to(w)
    eager = block.launch(dh, dw)["out"].clone()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        block.launch(dh, dw)
    for i in range(3):
        block._io_bufs["out"].fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(block._io_bufs["out"], eager), f"replay {i} differs"
        # eager work between replays
        again = block.launch(dh, dw)["out"]
        torch.cuda.synchronize()
        assert torch.equal(again, eager)
