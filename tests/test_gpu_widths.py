"""GPU parity of the kernels that take any width or format, at the sizes where
they can go wrong: edges of tiles, remainders, the smallest and largest of
their ranges. Bars as in test_gpu_parity (assert_close)."""
import numpy as np
import pytest

from test_gpu_parity import assert_close, ctx, f32_bits, mx4  # noqa: F401  (ctx, mx4: fixtures)
from test_launch_rules import GEMM_SHAPES, SKINNY_SHAPES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 32), (5, 96), (3, 32 * 16), (41, 32 * 50), (700, 32 * 33), (4100, 32 * 40)])
@pytest.mark.parametrize("shift", [0, 1, 13])
def test_wrapped_scale_range(mx4, ctx, rows, cols, shift):
    """mx4_weight_wrap scans the scales for NaN bytes and for bytes that the
    folding paths refuse; a planted byte is found at the first, the last and
    the piece-boundary positions, at any alignment of the scales."""
    count = rows * cols // 32
    packed = ctx.buffer(rows * cols // 2)
    buf = ctx.buffer(count + shift + 16)
    # K % 128 == 0 lets the GEMM path accept the weight, so that its refusal names the byte
    foldable_path = cols % 128 == 0
    x, y = ctx.buffer(64 * cols * 4), ctx.buffer(64 * rows * 4)
    head = (16 - shift) % 16
    spots = {0, count - 1, min(head, count - 1), max(min(head, count) - 1, 0), count // 2,
             head + (count - head) // 16 * 16 if head < count - 1 else 0}
    for at in sorted(p for p in spots if 0 <= p < count):
        for byte in (255, 1, 253, None):
            s = np.full(count + shift + 16, 255, np.uint8)  # what lies around the scales is not read
            s[shift:shift + count] = 120
            if byte is not None:
                s[shift + at] = byte
            buf.upload(s)
            if byte == 255:
                with pytest.raises(mx4.Mx4Error, match="NaN scale"):
                    ctx.wrap_weight(packed, buf, rows, cols, 0, shift)
                continue
            w = ctx.wrap_weight(packed, buf, rows, cols, 0, shift)
            if foldable_path and byte is not None:
                with pytest.raises(mx4.Mx4Error, match="2..252"):
                    ctx.matmul(x, mx4.F32, 64, w, y, mx4.PATH_GEMM)
            w.release()


def planted(rng, n, k):
    """Random codes and scales of an n x k weight (scale bytes 118..129)."""
    packed = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
    scales = rng.integers(118, 130, (n, k // 32), dtype=np.uint8)
    return packed, scales


def wrapped(ctx, packed, scales, shift):
    """The weight in device memory, its scales `shift` bytes off a word and NaN
    scale bytes and full codes all around both arrays."""
    n, k = packed.shape[0], 2 * packed.shape[1]
    pb = np.full(packed.size + 64, 0xff, np.uint8)
    pb[:packed.size] = packed.reshape(-1)
    sb = np.full(scales.size + shift + 64, 0xff, np.uint8)
    sb[shift:shift + scales.size] = scales.reshape(-1)
    return ctx.wrap_weight(ctx.to_device(pb), ctx.to_device(sb), n, k, 0, shift)


def activations(mx4, ctx, rng, m, k, xt):
    """(device buffer, f32 values): m rows with NaN rows behind them."""
    x = rng.standard_normal((m, k)).astype(np.float32)
    if xt == mx4.BF16:
        bits = (x.view(np.uint32) >> 16).astype(np.uint16)
        x = (bits.astype(np.uint32) << 16).view(np.float32)
        return ctx.to_device(np.concatenate([bits.reshape(-1), np.full(2 * k, 0x7fc0, np.uint16)])), x
    return ctx.to_device(np.concatenate([x.reshape(-1), np.full(2 * k, np.nan, np.float32)])), x


def check_any_width(mx4, ctx, oracle, seed, m, ns, k, shift):
    """One weight (ns[0]) and the group of all of ns through the default path,
    bf16 and f32 activations, against the oracle. Scaled: the planted scale
    bytes make outputs of any size."""
    rng = np.random.default_rng(seed)
    stored = [planted(rng, n, k) for n in ns]
    ws = [wrapped(ctx, p, s, shift) for p, s in stored]
    for xt in (mx4.BF16, mx4.F32):
        xb, x = activations(mx4, ctx, rng, m, k, xt)
        refs = [oracle.matmul(x, p.reshape(-1), s.reshape(-1)) for p, s in stored]
        what = f"m={m} ns={ns} k={k} shift={shift} xt={xt}"
        y = ctx.to_device(np.full(m * ns[0] + 64, 7.0, np.float32))
        ctx.matmul(xb, xt, m, ws[0], y)
        out = y.download(np.float32)
        assert np.all(out[m * ns[0]:] == 7.0), f"{what}: written past the output"
        assert_close(out[:m * ns[0]].reshape(m, ns[0]), refs[0], what, scaled=True)
        ys = [ctx.to_device(np.full(m * n + 64, 7.0, np.float32)) for n in ns]
        ctx.matmul_group(xb.ptr, xt, m, ws, [b.ptr for b in ys])
        for n, b, ref in zip(ns, ys, refs):
            out = b.download(np.float32)
            assert np.all(out[m * n:] == 7.0), f"{what}: written past a group's output"
            assert_close(out[:m * n].reshape(m, n), ref, f"{what} group", scaled=True)
    for w in ws:
        w.release()


# more than 32 token rows: K below, at and past a 128-element stage and with 1
# to 3 blocks left in the last one; rows and columns around 64; enough stages that
# the K split's last slice is short. (All but a few on 64 x 64 tiles; the other
# instances: test_any_width_gemm_instances)
@pytest.mark.parametrize("m,ns,k,shift", [
    (33, (1, 65, 31), 32, 0), (64, (64, 192), 96, 1), (65, (129, 3), 160, 2), (77, (320, 64, 64), 416, 3),
    (129, (50, 257), 352, 0), (40, (193, 33, 7, 64), 1600, 1), (200, (640, 96), 544, 2), (260, (2100,), 288, 3),
    (50, (256, 64, 33), 512, 0)])  # (a group of whole stages: f32 split, bf16 not)
def test_prompt_any_width(mx4, ctx, oracle, m, ns, k, shift):
    check_any_width(mx4, ctx, oracle, m + k, m, ns, k, shift)


# one token row: every number of rows side by side (up to 16, 32, more blocks),
# blocks a lane, waves a team and rows a team, each with its lanes full, one
# short and one over, K past the shared copy of x, and row counts that leave
# row-sets ragged
@pytest.mark.parametrize("ns,k,shift", [
    ((1, 2, 5), 32, 0), ((70, 33), 512, 1), ((67, 4), 544, 2), ((1030, 6), 1024, 3), ((515, 1), 1056, 0),
    ((9000, 130), 1600, 1), ((18000, 7), 480, 2), ((70000,), 992, 0), ((40001,), 288, 1), ((300, 20, 20), 2080, 3),
    ((8200, 9), 3264, 0), ((33, 5), 4064, 0), ((300, 31), 5184, 1), ((65, 3), 6176, 2), ((513, 2), 8960, 0),
    ((40, 41), 11008, 3), ((21, 8), 13824, 0), ((5, 9), 24576, 1), ((3, 2), 24608, 0)])
def test_decode_any_width(mx4, ctx, oracle, ns, k, shift):
    check_any_width(mx4, ctx, oracle, ns[0] + k, 1, ns, k, shift)


@pytest.mark.parametrize("n,k", [(20001, 480), (20001, 992), (40003, 1024), (40003, 1600), (20002, 3264), (5000, 5184),
                                 (100, 96)])
def test_argmax_any_width(mx4, ctx, oracle, n, k):
    """The fused lm_head: the logits are the projection's bit for bit, the
    index the first maximum of them (a tie planted across the vocabulary)."""
    rng = np.random.default_rng(n + k)
    packed, scales = planted(rng, n, k)
    packed[n - 1], scales[n - 1] = packed[7], scales[7]
    w = wrapped(ctx, packed, scales, 1)
    for xt in (mx4.BF16, mx4.F32):
        xb, x = activations(mx4, ctx, rng, 1, k, xt)
        y, z, idx = ctx.buffer(n * 4), ctx.buffer(n * 4), ctx.buffer(4)
        ctx.matmul(xb, xt, 1, w, y)
        ctx.matmul_argmax(xb, xt, w, z, idx)
        logits = z.download(np.float32)
        assert np.array_equal(y.download(np.uint32), logits.view(np.uint32)), (n, k, xt)
        assert idx.download(np.uint32)[0] == int(np.argmax(logits)), (n, k, xt)
        ctx.matmul_argmax(xb, xt, w, None, idx)
        assert idx.download(np.uint32)[0] == int(np.argmax(logits)), (n, k, xt)
    w.release()


# one-row projections, whose fused form takes another launch shape
@pytest.mark.parametrize("n,k", [(5000, 2048), (20002, 2048), (9001, 4096), (16383, 4096), (33000, 4096), (5001, 8192)])
def test_argmax_tuned_widths(mx4, ctx, oracle, n, k):
    if k == 8192:  # (two waves a team there, one here: another order of the same sums)
        rng = np.random.default_rng(n)
        packed, scales = planted(rng, n, k)
        w = wrapped(ctx, packed, scales, 0)
        xb, x = activations(mx4, ctx, rng, 1, k, mx4.BF16)
        z, idx = ctx.buffer(n * 4), ctx.buffer(4)
        ctx.matmul_argmax(xb, mx4.BF16, w, z, idx)
        logits = z.download(np.float32)
        assert_close(logits.reshape(1, n), oracle.matmul(x, packed.reshape(-1), scales.reshape(-1)), (n, k), scaled=True)
        assert idx.download(np.uint32)[0] == int(np.argmax(logits))
        w.release()
    else:
        test_argmax_any_width(mx4, ctx, oracle, n, k)


# 2 to 32 token rows: one and two token tiles, chunks of 128 that leave 1 to 3
# blocks, fewer chunks than waves, one to four chunks a wave, several slices of
# K, and one, two and four row tiles a workgroup with several sets of them
@pytest.mark.parametrize("m,ns,k,shift", [
    (2, (1, 17, 33), 32, 0), (7, (100, 16), 96, 1), (16, (50, 7, 65, 16), 416, 2), (17, (130, 31), 1024, 3),
    (3, (320, 64), 1600, 0), (32, (65, 40), 1632, 1), (9, (200, 3), 3264, 2), (29, (48, 70), 3104, 3),
    (5, (33, 50), 4160, 0), (31, (90, 20), 4288, 1), (12, (35, 64), 9216 + 32, 2), (2, (8300, 9), 160, 0),
    (16, (16500, 40), 224, 1), (20, (33000, 5), 96, 0), (4, (17000,), 1312, 3), (32, (9000, 700), 2304, 2)])
def test_verify_any_width(mx4, ctx, oracle, m, ns, k, shift):
    check_any_width(mx4, ctx, oracle, m + ns[0] + k, m, ns, k, shift)


# the instances that turn the weights through the wave's LDS stage with several
# tiles and slices in a row: four chunks a wave (two tiles; more than 256 row
# tiles of K > 2048), two (one and two tiles; two and four with two token tiles)
@pytest.mark.parametrize("m,ns,k,shift", [
    (7, (4200, 16), 3264, 0), (16, (9000, 40), 2592, 1), (9, (5000,), 8224, 2), (5, (600, 50), 2080, 3),
    (12, (4500,), 1056, 1), (29, (4300, 17), 1600, 0), (20, (9000,), 3104, 3)])
def test_verify_staged_weights(mx4, ctx, oracle, m, ns, k, shift):
    check_any_width(mx4, ctx, oracle, m + ns[0] + k, m, ns, k, shift)


@pytest.mark.parametrize("m,k", [(1, 416), (5, 416), (13, 1600), (29, 544), (40, 352)])
def test_nonfinite_activations_any_width(mx4, ctx, oracle, m, k):
    """An inf, a NaN or the largest finite value in one token row shows in that
    row as the reference's loop has it, and nowhere else; f32 and bf16."""
    rng = np.random.default_rng(m * k)
    n = 70
    packed, scales = planted(rng, n, k)
    scales[:] = np.minimum(scales, 123)  # the largest product stays below 2^128
    w = wrapped(ctx, packed, scales, 1)
    for xt in (mx4.BF16, mx4.F32):
        for value in (np.inf, -np.inf, np.nan, np.float32(3.0e38)):
            for at in (0, 33, k - 1):
                x = rng.standard_normal((m, k)).astype(np.float32)
                x[m // 2, at] = value
                if xt == mx4.BF16:
                    bits = (x.view(np.uint32) >> 16).astype(np.uint16)
                    x = (bits.astype(np.uint32) << 16).view(np.float32)
                xb = ctx.to_device(bits if xt == mx4.BF16 else x)
                y = ctx.buffer(m * n * 4)
                ctx.matmul(xb, xt, m, w, y)
                out = y.download(np.float32).reshape(m, n)
                with np.errstate(all="ignore"):
                    ref = oracle.matmul(x, packed.reshape(-1), scales.reshape(-1))
                what = f"m={m} k={k} xt={xt} value={value} at={at}"
                assert np.array_equal(np.isnan(out), np.isnan(ref)), what
                assert np.array_equal(np.isinf(out), np.isinf(ref)), what
                ok = np.isfinite(ref)
                assert np.array_equal(np.sign(out[np.isinf(ref)]), np.sign(ref[np.isinf(ref)])), what
                for row in range(m):
                    if ok[row].all():
                        assert_close(out[row:row + 1], ref[row:row + 1], what, scaled=True)
    w.release()


def check_bf16_weights(mx4, ctx, oracle, seed, m, ns, k):
    """bf16 weights (one, and the group of all of ns) through the default path
    against the oracle, bf16 and f32 activations."""
    rng = np.random.default_rng(seed)
    ws, vals = [], []
    for n in ns:
        bits = (rng.standard_normal((n, k)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
        vals.append(bits)
        ws.append(ctx.upload_weight_bf16(bits, n, k))
    for xt in (mx4.BF16, mx4.F32):
        xb, x = activations(mx4, ctx, rng, m, k, xt)
        refs = [oracle.matmul_bf16(x, b) for b in vals]
        what = f"bf16 weights m={m} ns={ns} k={k} xt={xt}"
        y = ctx.to_device(np.full(m * ns[0] + 64, 7.0, np.float32))
        ctx.matmul(xb, xt, m, ws[0], y)
        out = y.download(np.float32)
        assert np.all(out[m * ns[0]:] == 7.0), f"{what}: written past the output"
        assert_close(out[:m * ns[0]].reshape(m, ns[0]), refs[0], what, scaled=True)
        ys = [ctx.to_device(np.full(m * n + 64, 7.0, np.float32)) for n in ns]
        ctx.matmul_group(xb.ptr, xt, m, ws, [b.ptr for b in ys])
        for n, b, ref in zip(ns, ys, refs):
            out = b.download(np.float32)
            assert np.all(out[m * n:] == 7.0), f"{what}: written past a group's output"
            assert_close(out[:m * n].reshape(m, n), ref, f"{what} group", scaled=True)
    for w in ws:
        w.release()


# K of whole 16-byte pieces and not (9, 1604: the element-wise kernel)
@pytest.mark.parametrize("m,ns,k", [
    (2, (1, 17), 8), (5, (33, 16), 9), (7, (100, 3), 120), (16, (50, 64, 7), 136), (17, (70, 40), 1024),
    (32, (65, 2), 1608), (3, (40, 20), 1604), (12, (8200, 5), 264), (29, (17000,), 136), (9, (70, 300), 4104)])
def test_bf16_verify(mx4, ctx, oracle, m, ns, k):
    check_bf16_weights(mx4, ctx, oracle, m + k, m, ns, k)


@pytest.mark.parametrize("m,k", [(1, 264), (5, 264), (29, 136), (40, 264), (70, 72)])
def test_bf16_nonfinite(mx4, ctx, oracle, m, k):
    """inf and NaN weights, and inf, NaN and 3e38 activations, give what the
    reference's loop gives, f32 and bf16 activations."""
    rng = np.random.default_rng(m * k)
    n = 40
    for value in (np.inf, np.nan, np.float32(3.0e38)):
        for where in ("weight", "x"):
            wf = rng.standard_normal((n, k)).astype(np.float32) * 0.1
            x = rng.standard_normal((m, k)).astype(np.float32)
            x[:, 8] = 1.0  # a value whose lower bf16 terms are zero
            if where == "weight":
                wf[3, 8] = wf[20, k - 1] = value
            else:
                x[m // 2, 8] = value
            wbits = (f32_bits(wf) >> 16).astype(np.uint16) | (np.isnan(wf) * 0x40).astype(np.uint16)
            xbits = (f32_bits(x) >> 16).astype(np.uint16) | (np.isnan(x) * 0x40).astype(np.uint16)
            w = ctx.upload_weight_bf16(wbits, n, k)
            for xt, host, dev in ((mx4.F32, x, ctx.to_device(x)),
                                  (mx4.BF16, (xbits.astype(np.uint32) << 16).view(np.float32), ctx.to_device(xbits))):
                y = ctx.buffer(m * n * 4)
                ctx.matmul(dev, xt, m, w, y)
                out = y.download(np.float32).reshape(m, n)
                with np.errstate(all="ignore"):
                    ref = oracle.matmul_bf16(host, wbits)
                what = f"m={m} k={k} xt={xt} {where}={value}"
                assert np.array_equal(np.isnan(out), np.isnan(ref)), what
                assert np.array_equal(np.isinf(out), np.isinf(ref)), what
                inf = np.isinf(ref)
                assert np.array_equal(np.sign(out[inf]), np.sign(ref[inf])), what
                ok = np.isfinite(ref)
                assert np.all(np.abs(out[ok].astype(np.float64) - ref[ok]) <= 1e-3 + 1e-5 * np.abs(ref[ok].astype(np.float64))), what
            w.release()


# K of one turn and several with lanes past its end, K past the LDS copy of x
# (24576 f32: the row-per-wave kernel) and K of no whole pieces
@pytest.mark.parametrize("ns,k", [
    ((1, 3), 8), ((33, 5), 520), ((50, 64, 7), 1024), ((130, 2), 1608), ((70, 9), 2056), ((5000, 1), 264),
    ((9000, 4000, 3), 136), ((40, 41), 12296), ((20, 3), 20480), ((17, 5), 24576), ((40, 20), 1604)])
def test_bf16_decode(mx4, ctx, oracle, ns, k):
    check_bf16_weights(mx4, ctx, oracle, ns[0] + k, 1, ns, k)


# rows and columns around 64 and 128; K below, at and past a 64-element stage, odd
# and even stage counts, K splits with a short last slice, and K of no whole pieces
# (small weights run the row-per-wave kernel, the others the smallest tiles; every
# tile: test_bf16_gemm_instances)
@pytest.mark.parametrize("m,ns,k", [
    (33, (1, 65), 8), (64, (64, 128, 2), 64), (65, (127, 33), 72), (129, (130, 5), 200), (40, (300, 7, 64, 1), 1032),
    (200, (257, 64), 2056), (500, (1100, 40), 328), (70, (60, 9), 4100), (1000, (520,), 136)])
def test_bf16_prompt(mx4, ctx, oracle, m, ns, k):
    check_bf16_weights(mx4, ctx, oracle, m + k, m, ns, k)


@pytest.mark.parametrize("team", [1, 2, 4])
def test_explicit_team_keeps_a_default_that_fits(mx4, ctx, oracle, team):
    """An explicit team size with the default number of teams a workgroup, at
    the width whose default is several two-wave teams (K = 8192)."""
    rng = np.random.default_rng(team)
    n, k = 70, 8192
    packed, scales = planted(rng, n, k)
    w = wrapped(ctx, packed, scales, 0)
    for xt in (mx4.BF16, mx4.F32):
        xb, x = activations(mx4, ctx, rng, 1, k, xt)
        ref = oracle.matmul(x, packed.reshape(-1), scales.reshape(-1))
        for teams in (0, 7):
            y = ctx.to_device(np.full(n, np.nan, np.float32))
            ctx.gemv_config(xb.ptr, xt, w, y.ptr, team, 1, teams, 0)
            assert_close(y.download(np.float32).reshape(1, n), ref, f"team={team} xt={xt} teams={teams}", scaled=True)
    w.release()


# Distance from the sum in 64 bits, relative to its length: of all outputs and of
# one token row's. Products are exact, and a chain of 32-bit additions is at most
# 24 long (three terms of eight MFMAs) before it continues in 64 bits: 24 roundings
# of at most 2^-24 of a partial sum walk to about 24^0.5 2^-24 / 3^0.5 = 1.7e-7 of
# its size (measured 0.5 to 1.3e-7), a single row of few large outputs to three
# times that. One chain over all of K or a lost third term shows as 4e-7 and more
# over all outputs.
ALL_TOL, ROW_TOL = 2.5e-7, 6e-7


def check_rows(out, x, w, what, alike=True):
    """Every token row of out, and all of them (if they are of one size), against
    x . w^T in 64 bits."""
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    diff, size = np.linalg.norm(out.astype(np.float64) - ref, axis=1), np.linalg.norm(ref, axis=1)
    err = diff / size
    assert np.all(err <= ROW_TOL), f"{what}: row {int(np.argmax(err))} of {len(err)}: {np.max(err):.2e}"
    whole = np.linalg.norm(diff) / np.linalg.norm(size) if alike else np.sqrt(np.mean(err * err))
    assert whole <= ALL_TOL, f"{what}: {whole:.2e} over all outputs"


def tiny_rows(rng, m, k, exponent):
    """f32 activations of size 2^-20 but for a few token rows: the first and the
    last all of size 2^exponent, the second that in every other run of 64."""
    x = np.ldexp(rng.standard_normal((m, k)), -20)
    small = np.ldexp(rng.standard_normal((m, k)), exponent)
    x[0], x[-1] = small[0], small[-1]
    x[1, np.arange(k) // 64 % 2 == 0] = small[1, np.arange(k) // 64 % 2 == 0]
    return x.astype(np.float32)


@pytest.mark.parametrize("exponent", [-100, -112, -118, -126, -140])
@pytest.mark.parametrize("m,n,k", [(2, 50, 416), (9, 4200, 992), (16, 8300, 160), (29, 70, 1600), (23, 600, 2048),
                                   (40, 130, 352), (77, 70, 1632), (200, 320, 1600)])
def test_tiny_f32_activations(mx4, ctx, oracle, m, n, k, exponent):
    """Activations down to subnormal ones keep all their bits on the kernels for
    any width (and f32 verify steps of the tuned ones) and for bf16 weights."""
    rng = np.random.default_rng(m + n - exponent)
    up = min(120 - exponent, 245)
    packed = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
    scales = rng.integers(up - 3, up + 1, (n, k // 32)).astype(np.uint8)
    bits = (f32_bits(np.ldexp(rng.standard_normal((n, k)), up - 127).astype(np.float32)) >> 16).astype(np.uint16)
    x = tiny_rows(rng, m, k, exponent)
    xb, y = ctx.to_device(x), ctx.buffer(m * n * 4)
    for what, w, values in (("mxfp4", wrapped(ctx, packed, scales, 1), oracle.dequantize(packed, scales)),
                            ("bf16", ctx.upload_weight_bf16(bits, n, k), oracle.bf16_to_f32(bits))):
        ctx.matmul(xb, mx4.F32, m, w, y)
        check_rows(y.download(np.float32).reshape(m, n), x, values, f"{what} m={m} n={n} k={k} 2^{exponent}", alike=False)
        w.release()


@pytest.mark.parametrize("m,n,k", [(5, 100, 264), (29, 5000, 1032), (40, 70, 264), (150, 200, 1608)])
def test_bf16_inf_weight_rows(mx4, ctx, oracle, m, n, k):
    """Weight rows with infs beside token rows with a NaN, an inf or both signs
    of inf: every output is what the reference's loop gives."""
    rng = np.random.default_rng(m + n)
    w = (rng.standard_normal((n, k)) * 0.1).astype(np.float32)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[:, 8] = 1.0  # a value whose lower bf16 terms are zero
    w[3, 8], w[n - 1, [8, 9]], w[20, k - 1] = np.inf, [-np.inf, np.inf], np.nan
    x[1, 17], x[m - 1, k - 2] = np.nan, np.inf
    x[2, [30, 31]] = [np.inf, -np.inf]
    bits = (f32_bits(w) >> 16).astype(np.uint16) | (np.isnan(w) * 0x40).astype(np.uint16)
    weight = ctx.upload_weight_bf16(bits, n, k)
    y = ctx.buffer(m * n * 4)
    ctx.matmul(ctx.to_device(x), mx4.F32, m, weight, y)
    out = y.download(np.float32).reshape(m, n)
    with np.errstate(all="ignore"):
        ref = oracle.matmul_bf16(x, bits)
    assert np.array_equal(np.isnan(out), np.isnan(ref))
    assert np.array_equal(np.isposinf(out), np.isposinf(ref)) and np.array_equal(np.isneginf(out), np.isneginf(ref))
    ok = np.isfinite(ref)
    assert np.all(np.abs(out[ok].astype(np.float64) - ref[ok]) <= 1e-3 + 1e-5 * np.abs(ref[ok].astype(np.float64)))
    weight.release()


def call_us(ctx, call):
    """Microseconds of a call, from recorded passes of sixteen."""
    step = ctx.record(lambda: [call() for _ in range(16)])
    runs = []
    for _ in range(7):
        ctx.timer_begin()
        step.launch()
        runs.append(ctx.timer_end())
    step.release()
    return sorted(runs)[3] / 16 * 1e3


@pytest.mark.parametrize("kind", ["nan", "infs", "nan weights", "tiny"])
@pytest.mark.parametrize("m", [16, 64])
def test_odd_values_cost_no_more_than_a_few_calls(mx4, ctx, m, kind):
    """Activations or bf16 weights full of NaNs, infs or subnormals take a small
    multiple of the usual call (at most two passes over everything, the weights
    read up to three times over; once every NaN was summed again by itself, a
    hundred times the usual)."""
    rng = np.random.default_rng(m)
    n, k = 2048, 4096
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    x = rng.standard_normal((m, k)).astype(np.float32)
    odd_w, odd_x = w, x
    if kind == "nan":
        odd_x = np.full_like(x, np.nan)
    elif kind == "infs":
        odd_x = x.copy()
        odd_x[:, 100:110] = np.inf
    elif kind == "nan weights":
        odd_w = np.full_like(w, np.nan)
    else:
        odd_x = np.ldexp(x, -130).astype(np.float32)
    times = []
    for ww, xx in ((w, x), (odd_w, odd_x)):
        bits = (f32_bits(ww) >> 16).astype(np.uint16)
        weight = ctx.upload_weight_bf16(bits, n, k)
        xb, y = ctx.to_device(xx), ctx.buffer(m * n * 4)
        times.append(call_us(ctx, lambda: ctx.matmul(xb, mx4.F32, m, weight, y)))
        weight.release()
    print(f"m={m} {kind}: {times[0]:.1f} -> {times[1]:.1f} us", flush=True)
    assert times[1] <= 25 * times[0], (m, kind, times)


def check_not_slower(mx4, ctx, w, m, k, n, what):
    """The default path's time within a third of the general kernel's."""
    y = ctx.buffer(m * n * 4)
    for xt in (mx4.BF16, mx4.F32):
        x = ctx.to_device(np.ones(m * k * (1 if xt == mx4.F32 else 2), np.float32 if xt == mx4.F32 else np.uint16))
        auto, general = (call_us(ctx, lambda: ctx.matmul(x, xt, m, w, y, path)) for path in (mx4.PATH_AUTO, mx4.PATH_GENERIC))
        print(f"{what} m={m} n={n} k={k} xt={xt}: {auto:.1f} us, general {general:.1f}", flush=True)
        assert auto <= 1.33 * general + 0.5, (what, m, n, k, xt, auto, general)


@pytest.mark.parametrize("n,k", [(16, 1024), (64, 4096), (64, 12288), (320, 1600), (640, 1024), (1024, 4096), (2048, 2048),
                                 (4096, 4096)])
@pytest.mark.parametrize("m", [2, 4, 8, 16, 32, 33, 64, 300])
def test_bf16_small_weights_speed(mx4, ctx, m, n, k):
    """Where the matrix cores would leave most of the chip idle, the row-per-wave
    kernel runs: no call takes much longer than that one."""
    w = ctx.upload_weight_bf16(np.full(n * k, 0x3c00, np.uint16), n, k)
    check_not_slower(mx4, ctx, w, m, k, n, "bf16 weights")
    w.release()


@pytest.mark.parametrize("n,k", [(16, 1600), (64, 480), (64, 8992), (128, 1600), (256, 3264), (256, 8992), (512, 1600),
                                 (1024, 4288)])
@pytest.mark.parametrize("m", [2, 8, 16, 32, 33, 64, 128, 300])
def test_any_width_small_weights_speed(mx4, ctx, m, n, k):
    """The same for widths off the tuned ones and the generic kernel."""
    w = ctx.synth_weight(n + k, n, k)
    check_not_slower(mx4, ctx, w, m, k, n, "any width")
    w.release()


@pytest.mark.parametrize("n,k,few,more", [(100, 2080, 16, 20), (256, 1056, 16, 32), (64, 1056, 16, 20), (16, 4288, 16, 17)])
def test_small_weights_stay_on_matrix_cores(mx4, ctx, n, k, few, more):
    """Nearly empty steps along K: going from 16 bf16 token rows to the next tile
    of them costs what it costs on the matrix cores (1.2 to 1.35 times the call),
    not what the generic kernel would take (1.5 to 1.9)."""
    w = ctx.synth_weight(n + k, n, k)
    x, y = ctx.to_device(np.full(more * k, 0x3f80, np.uint16)), ctx.buffer(more * n * 4)
    a, b = (call_us(ctx, lambda: ctx.matmul(x, mx4.BF16, m, w, y)) for m in (few, more))
    print(f"n={n} k={k}: m={few} {a:.2f} us, m={more} {b:.2f}", flush=True)
    assert b <= 1.43 * a, (n, k, a, b)
    w.release()


# The same distance on small weights, which kernels without matrix cores take: chains
# of at most eight products and one 32-bit sum of two of them, then 64 bits. The
# partial sums' rounding, (1 + .. + 8) / 8 + 1 = 5.5 in units of the last one's
# variance (2.5e-8 squared: uniform over half a unit of 24 bits, mantissas from 1 to
# 2), and that of the output make 2.5e-8 6.5^0.5 = 0.65e-7 (measured 0.25 to
# 0.7e-7); one chain per lane at these K 1.2e-7 and more for f32 activations.
SMALL_TOL = 0.9e-7


@pytest.mark.parametrize("fp4,m,n,k", [(True, 14, 64, 1600), (True, 28, 128, 1600), (True, 16, 256, 8992),
                                       (True, 32, 128, 8992), (True, 33, 64, 1600), (True, 64, 64, 8992),
                                       (True, 77, 64, 1056), (False, 2, 512, 8192), (False, 3, 1001, 4096),
                                       (False, 8, 333, 4096), (False, 24, 64, 12296), (False, 33, 64, 4096),
                                       (False, 77, 64, 4104)])
def test_small_weights_precision(mx4, ctx, oracle, fp4, m, n, k):
    rng = np.random.default_rng(m + n + k)
    if fp4:
        packed, scales = planted(rng, n, k)
        scales = np.full_like(scales, 120)
        weight, w = ctx.upload_weight(packed, scales, n, k), oracle.dequantize(packed, scales)
    else:
        bits = (f32_bits(rng.standard_normal((n, k)).astype(np.float32)) >> 16).astype(np.uint16)
        weight, w = ctx.upload_weight_bf16(bits, n, k), oracle.bf16_to_f32(bits)
    for xt in (mx4.BF16, mx4.F32):
        xb, x = activations(mx4, ctx, rng, m, k, xt)
        x = x.reshape(m, k).astype(np.float64)
        y = ctx.to_device(np.full(m * n + 64, 7.0, np.float32))
        ctx.matmul(xb, xt, m, weight, y)
        out = y.download(np.float32)
        assert np.all(out[m * n:] == 7.0)
        ref = x @ w.astype(np.float64).T
        err = np.linalg.norm(out[:m * n].reshape(m, n) - ref) / np.linalg.norm(ref)
        print(f"fp4={fp4} m={m} n={n} k={k} xt={xt}: {err:.2e}", flush=True)
        assert err <= SMALL_TOL, (fp4, m, n, k, xt, err)
    weight.release()


@pytest.mark.parametrize("m", [1, 3, 5, 29, 77])
@pytest.mark.parametrize("tiny", ["x", "w"])
def test_subnormal_bf16_operands(mx4, ctx, oracle, tiny, m):
    """bf16 activations and bf16 weights, one of them below the normal range: the
    dot products and matrix cores keep subnormal values."""
    rng = np.random.default_rng(m)
    n, k = 200, 1608
    bits = {}
    for name, rows in (("x", m), ("w", n)):
        values = np.ldexp(rng.standard_normal((rows, k)), -130 if name == tiny else 100).astype(np.float32)
        bits[name] = (f32_bits(values) >> 16).astype(np.uint16)
    weight, y = ctx.upload_weight_bf16(bits["w"], n, k), ctx.buffer(m * n * 4)
    ctx.matmul(ctx.to_device(bits["x"]), mx4.BF16, m, weight, y)
    check_rows(y.download(np.float32).reshape(m, n), oracle.bf16_to_f32(bits["x"]), oracle.bf16_to_f32(bits["w"]),
               f"tiny {tiny}, m={m}")
    weight.release()


def test_group_split_pays(mx4, ctx):
    """A group of short rows and many outputs is not cut along K, where adding
    the slices would cost more than it saves: well below its members, which are
    cut."""
    m, n, k = 300, 1536, 512
    ws = [ctx.synth_weight(i, n, k) for i in (1, 2)]
    x, ys = ctx.to_device(np.ones(m * k, np.float32)), [ctx.buffer(m * n * 4) for _ in ws]
    group = call_us(ctx, lambda: ctx.matmul_group(x.ptr, mx4.F32, m, ws, [y.ptr for y in ys]))
    apart = call_us(ctx, lambda: [ctx.matmul(x, mx4.F32, m, w, y) for w, y in zip(ws, ys)])
    print(f"group {group:.1f} us, apart {apart:.1f}", flush=True)
    assert group <= 0.75 * apart, (group, apart)
    for w in ws:
        w.release()


def some(rng, count, most):
    """All of range(count), or its first and last few and a draw."""
    if count <= most:
        return np.arange(count)
    third = most // 3
    return np.unique(np.r_[0:third, count - third:count, rng.choice(count, third)])


def run_instance(mx4, ctx, oracle, fp4, x_bf16, m, rows, k):
    """One call (a group's for more than one weight) against sums in 64 bits:
    every output written, none past the end, sampled ones within ROW_TOL, once on
    plain activations of full mantissas and once, f32, with an inf in one token
    row and a NaN in another (which show there and nowhere else)."""
    rng = np.random.default_rng(m + sum(rows) + k)
    ws, values = [], []
    for n in rows:
        cols = some(rng, n, 96)
        if fp4:
            packed, scales = planted(rng, n, k)
            ws.append(wrapped(ctx, packed, scales, n % 4))
            values.append((cols, oracle.dequantize(packed[cols], scales[cols])))
        else:
            bits = rng.integers(0x3c00, 0x3f80, (n, k), dtype=np.uint16) | (rng.integers(0, 2, (n, k), dtype=np.uint16) << 15)
            ws.append(ctx.upload_weight_bf16(bits, n, k))
            values.append((cols, oracle.bf16_to_f32(bits[cols])))
    xt = mx4.BF16 if x_bf16 else mx4.F32
    ys = [ctx.buffer((m * n + 64) * 4) for n in rows]
    for odd in (False, True) if xt == mx4.F32 else (False,):
        xb, x = activations(mx4, ctx, rng, m, k, xt)
        toks = some(rng, m, 48)
        if odd:
            x[toks[1], k // 2], x[toks[-2], k - 1] = np.inf, np.nan
            xb = ctx.to_device(np.concatenate([x.reshape(-1), np.full(2 * k, np.nan, np.float32)]))
        for y, n in zip(ys, rows):
            y.upload(np.full(m * n + 64, 7.0, np.float32))
        if len(rows) == 1:
            ctx.matmul(xb, xt, m, ws[0], ys[0])
        else:
            ctx.matmul_group(xb.ptr, xt, m, ws, [y.ptr for y in ys])
        for y, n, (cols, w) in zip(ys, rows, values):
            out = y.download(np.float32)
            what = f"fp4={fp4} x_bf16={x_bf16} m={m} rows={rows} n={n} k={k} odd={odd}"
            assert np.all(out[m * n:] == 7.0), f"{what}: written past the output"
            out = out[:m * n].reshape(m, n)
            got = out[np.ix_(toks, cols)]
            plain = np.ones(len(toks), bool)
            if odd:
                plain[[1, -2]] = False
                assert np.all(np.isnan(got[-2])), what
                with np.errstate(all="ignore"):
                    ref = (x[toks[1]].astype(np.float64) * w.astype(np.float64)).sum(1)
                assert np.array_equal(np.isnan(got[1]), np.isnan(ref)) and np.array_equal(np.isposinf(got[1]), np.isposinf(ref)), what
                bad = np.delete(out, [toks[1], toks[-2]], 0)
            else:
                bad = out
            assert np.all(np.isfinite(bad)) and np.count_nonzero(bad == 7.0) <= 2, what
            check_rows(got[plain], x[toks][plain], w, what)
    for w in ws:
        w.release()


@pytest.mark.parametrize("m,rows,k", sorted({s for (kind, _), shapes in GEMM_SHAPES.items() if kind == "exact" for s in shapes}))
def test_any_width_gemm_instances(mx4, ctx, oracle, m, rows, k):
    """Every any-width instance of the exact GEMM, alone and over a group, unsplit
    and split with short last slices, at ragged rows and columns."""
    for x_bf16 in (True, False):
        if (m, rows, k) in GEMM_SHAPES["exact", x_bf16]:
            run_instance(mx4, ctx, oracle, True, x_bf16, m, rows, k)


@pytest.mark.parametrize("m,rows,k", sorted({s for (kind, _), shapes in GEMM_SHAPES.items() if kind == "bf16" for s in shapes}))
def test_bf16_gemm_instances(mx4, ctx, oracle, m, rows, k):
    for x_bf16 in (True, False):
        if (m, rows, k) in GEMM_SHAPES["bf16", x_bf16]:
            run_instance(mx4, ctx, oracle, False, x_bf16, m, rows, k)


@pytest.mark.parametrize("fp4,x_bf16,m,rows,k", list(SKINNY_SHAPES))
def test_any_width_skinny_instances(mx4, ctx, oracle, fp4, x_bf16, m, rows, k):
    run_instance(mx4, ctx, oracle, fp4, x_bf16, m, rows, k)
