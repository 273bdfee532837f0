"""The operand-ordered Q8_0 kernels (q8_mid.hip) against the oracle, bit for bit: an exact integer dot per 32-element
block, (wScale * aScale) * dot and the ascending block sum (RT/Q8DotKernel.cs:352-445), per-head sums added in order
(RT/CachedMultiHeadAttention.cs:689-710).

The shapes lie at the edges of the kernels and of the rule between them: 2 .. 130 rows around multiples of 16, planes of
1, 2, 3, 4, 5 and 513 blocks (whole and partial groups of four, one group to more than a round of eight waves), outputs off
the 16- and 64-row tiles, the split kernel on four and eight waves and the panel kernel at each of its heights. Scales hold
subnormals, and a last weight row of infinite and NaN scales, which no other output may show.
"""
import sys

import numpy as np
import pytest

from qdata import normal

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
ov = pytest.importorskip("overfit_amd")

DEV = "cuda:0"


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _planes(rng, n, k):
    q = rng.integers(-128, 128, size=(n, k), dtype=np.int8)
    s = rng.uniform(1e-4, 1e-2, size=(n, k // 32)).astype(np.float32)
    s[::3] *= np.float32(1e-40)  # subnormal
    s[-1, 0::2], s[-1, 1::2] = np.inf, np.nan
    return q, s


def _x(rng, rows, k):
    x = normal(rng, (rows, k))
    x[::5] *= np.float32(1e-30)
    x[rows - 1, -32:] = 0.0
    return x


def _check(y, ref, what):
    y = y.cpu().numpy().reshape(ref.shape)
    nan = np.isnan(ref)
    same = (y.view(np.uint32) == ref.view(np.uint32)) | (nan & np.isnan(y))
    bad = int(np.count_nonzero(~same))
    assert bad == 0, f"{what}: {bad}/{y.size} outputs differ from the oracle"


# test_kernel_choice.py checks that the automatic choice takes the kernels of this file for every shape.
PROJECT = [
    (33, 32, 17),      # one block: a group of four with three absent
    (33, 160, 40),     # five blocks: the second group of one
    (17, 96, 4090),    # two tiles, four waves, as many workgroups as CUs
    (2, 16416, 33),    # past the decode kernel at two rows; 129 groups, rounds of eight waves
    (33, 640, 31),     # three tiles, the second workgroup's upper one absent
    (130, 288, 48),    # nine tiles on the split kernel
    (16, 512, 4113),   # more 16-row tiles than CUs, one activation tile: four waves
    (65, 416, 4100),   # panel of 32 rows
    (150, 96, 4031),   # panel of 48
    (120, 544, 14330),  # panel of 64
    (512, 64, 1030),
]


@pytest.mark.parametrize("rows,k,n", PROJECT + [(9, 32, 17), (16, 160, 40), (120, 160, 14330)])  # the last three stay
def test_project_bit_exact(orc, rows, k, n):
    print("[case] q8 mid", rows, k, n, flush=True, file=sys.stderr)
    rng = np.random.default_rng(rows + k + n)
    q, s = _planes(rng, n, k)
    w = ov.Q8Weight(q.reshape(-1), s.reshape(-1), k, n)
    x, bias = _x(rng, rows, k), normal(rng, n)
    for b in (None, bias):
        y = ov.project(w, t(x).view(-1), rows=rows, bias=None if b is None else t(b))
        torch.cuda.synchronize()
        _check(y, orc.q8_project_batched(x, rows, q, s, k, n, b), f"bias={b is not None}")


@pytest.mark.parametrize("rows,H,hd,dm", [
    (9, 3, 32, 40),    # one block a head; fewer groups than four waves
    (6, 5, 160, 33),   # two groups a head, the second of one block
    (20, 11, 96, 64),  # three blocks; eight waves step past a head
    (16, 7, 64, 4113),  # four waves
    (33, 9, 256, 48),
    (65, 3, 128, 4100),  # panel of 32 rows
    (150, 5, 96, 4031),  # panel of 48
    (120, 2, 160, 14330),  # panel of 64
    (150, 3, 64, 4031),  # two of a group's four blocks computed
    (65, 2, 32, 4100),   # one
])
def test_heads_bit_exact(orc, rows, H, hd, dm):
    print("[case] q8 mid heads", rows, H, hd, dm, flush=True, file=sys.stderr)
    rng = np.random.default_rng(rows + H + hd + dm)
    planes = [_planes(rng, dm, hd) for _ in range(H)]
    ws = [ov.Q8Weight(q.reshape(-1), s.reshape(-1), hd, dm) for q, s in planes]
    x, bias = _x(rng, rows, H * hd), normal(rng, dm)
    for b in (None, bias):
        y = ov.project_heads_q8_0(ws, t(x), rows=rows, bias=None if b is None else t(b))
        torch.cuda.synchronize()
        ref = orc.q8_project_heads(x, rows, [q for q, _ in planes], [s for _, s in planes], hd, dm, b)
        _check(y, ref, f"bias={b is not None}")


def test_scale_products_of_any_exponent(orc):
    """One block a row, so that an output is one (wScale * aScale) * dot: the matrix unit's scale products against the
    oracle's float multiplication for 512 x 2040 pairs of scales with random sign, exponent and fraction, subnormal,
    infinite and NaN ones among them, and products past either end of the range."""
    print("[case] q8 mid scale products", flush=True, file=sys.stderr)
    rng = np.random.default_rng(31)
    rows, k, n = 512, 32, 2040
    bits = rng.integers(0, 1 << 32, size=n, dtype=np.uint64).astype(np.uint32)
    bits[:64] &= np.uint32(0x807FFFFF)  # subnormal
    s = bits.view(np.float32).reshape(n, 1)
    s[64:68, 0] = np.inf, -np.inf, np.nan, 0.0
    q = rng.integers(-128, 128, size=(n, k), dtype=np.int8)
    q[:, 0] = np.where(q[:, 0] == 0, 1, q[:, 0])
    x = np.zeros((rows, k), np.float32)  # a row's largest element gives its scale
    exponents = rng.integers(1, 255, size=rows, dtype=np.uint32) << 23
    x[:, 0] = (exponents | rng.integers(0, 1 << 23, size=rows, dtype=np.uint32)).view(np.float32)
    x[:, 1:] = x[:, :1] * rng.uniform(-1, 1, size=(rows, k - 1)).astype(np.float32)
    w = ov.Q8Weight(q.reshape(-1), s.reshape(-1), k, n)
    y = ov.project(w, t(x).view(-1), rows=rows)
    torch.cuda.synchronize()
    _check(y, orc.q8_project_batched(x, rows, q, s, k, n, None), "scale products")
