"""GPU parity of the kernels that take any width or format, at the sizes where
they can go wrong: edges of tiles, remainders, the smallest and largest of
their ranges. Bars as in test_gpu_parity (assert_close)."""
import numpy as np
import pytest

from test_gpu_parity import ctx, mx4  # noqa: F401  (fixtures)

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
