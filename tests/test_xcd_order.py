"""The block and item orders over the XCDs cover every logical index exactly
once (a host restatement of xcd_block and xcd_item / eval_grid)."""
import pytest

XCDS, WAVES = 8, 4


def xcd_block(b, n, chunk):
    xcd, local = b % XCDS, b // XCDS
    if chunk > 0:
        if b >= n // (XCDS * chunk) * (XCDS * chunk):
            return b
        return (local // chunk * XCDS + xcd) * chunk + local % chunk
    per, rem = n // XCDS, n % XCDS
    return xcd * per + min(xcd, rem) + local


def items(ni, icap, chunk):
    per = -(-icap // (XCDS * chunk)) * chunk if chunk else -(-icap // XCDS) + 1
    out = []
    for b in range(-(-per // WAVES) * XCDS):
        for w in range(WAVES):
            x, j = b % XCDS, b // XCDS * WAVES + w
            if chunk:
                first, last = (j // chunk * XCDS + x) * chunk + j % chunk, ni
            else:
                first, last = ni * x // XCDS + j, ni * (x + 1) // XCDS
            if first < last:
                out.append(first)
    return out


@pytest.mark.parametrize("chunk", [0, 1, 4, 32])
@pytest.mark.parametrize("n", [1, 7, 8, 31, 32, 33, 255, 256, 257, 1000, 4099])
def test_orders_are_bijections(n, chunk):
    assert sorted(xcd_block(b, n, chunk) for b in range(n)) == list(range(n))
    if chunk % WAVES == 0:
        for icap in (n, n + 1, n + 65):
            assert sorted(items(n, icap, chunk)) == list(range(n))
