"""The split and panel MFMA kernels (mfma_split.hip) against the oracle, bit for bit: every output is an exact integer
dot per super-block and the reference's fp32 sum over the row (RT/Q4KDotKernel.cs:944-951, RT/Q6KDotKernel.cs:114-115).

They take batches whose activation is quantised by the call, by a rule on rows and shapes; the shapes here lie on both
sides of its tile edges: 3 .. 150 rows around multiples of 16 and 64, output counts off the 16-row tiles, one
super-block to one more than the small-M kernel takes, four and eight waves, odd Q6_K super-block counts (rows that start
2, 4, .. 14 bytes past a 16-byte boundary), a last block that ends inside a 16-byte piece. test_kernel_choice.py checks
that the rule sends each list to the kernel that it names.
"""
import sys

import numpy as np
import pytest

from qdata import normal, random_q4k_blocks, random_q6k_blocks, set_subnormal_scales

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
ov = pytest.importorskip("overfit_amd")

DEV = "cuda:0"


def case(*what):
    print("[case]", *what, flush=True, file=sys.stderr)


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _weight(rng, fmt, n, k):
    nb = n * (k // 256)
    if fmt == "q4k":
        blocks = set_subnormal_scales(random_q4k_blocks(rng, nb))
        return blocks, ov.Q4KWeight(blocks.reshape(-1), k, n)
    blocks = set_subnormal_scales(random_q6k_blocks(rng, nb), q6=True)
    return blocks, ov.Q6KWeight(blocks.reshape(-1), k, n)


def _check(y, ref, what):
    y = y.cpu().numpy().reshape(ref.shape)
    bad = int(np.count_nonzero(y.view(np.uint32) != ref.view(np.uint32)))
    assert bad == 0, f"{what}: {bad}/{y.size} outputs differ from the oracle"


def _ref(orc, fmt, x, rows, blocks, k, n, bias):
    return (orc.q4k_project_batched if fmt == "q4k" else orc.q6k_project_batched)(x, rows, blocks, k, n, bias)


SPLIT = [
    (17, 256, 33),     # one super-block: three of four waves idle
    (3, 16640, 17),    # past the small-M kernel's inputs, from 3 rows; an incomplete last round of eight waves
    (5, 4352, 250),    # 17 super-blocks
    (16, 4096, 48),    # exactly one tile, two rounds of eight waves
    (17, 1792, 65),    # two tiles, four waves
    (33, 2304, 97),    # three tiles, two rounds
    (64, 2560, 16),    # four tiles
    (65, 3328, 31),    # two workgroups of three tiles, the last rows of the second absent
    (130, 768, 1000),  # nine tiles over three workgroups, four waves with one idle
]
SPLIT_FUSED = [(2, 4352, [7000, 48, 130]), (40, 1024, [256, 64, 70, 16])]


@pytest.mark.parametrize("fmt", ["q4k", "q6k"])
@pytest.mark.parametrize("rows,k,n", SPLIT + [(9, 256, 33), (16, 2048, 48)])  # the last two stay on the small-M kernel
def test_split_projection_bit_exact(orc, fmt, rows, k, n):
    case("split", fmt, rows, k, n)
    rng = np.random.default_rng(rows * 7919 + k + n)
    blocks, w = _weight(rng, fmt, n, k)
    x, bias = normal(rng, (rows, k)), normal(rng, n)
    _check(ov.project(w, t(x), t(bias), rows=rows), _ref(orc, fmt, x, rows, blocks, k, n, bias), "bias")
    _check(ov.project(w, t(x), rows=rows), _ref(orc, fmt, x, rows, blocks, k, n, None), "no bias")


@pytest.mark.parametrize("rows,k,shapes", SPLIT_FUSED + [(2, 4352, [128, 48, 50])])
def test_split_fused_projections_bit_exact(orc, rows, k, shapes):
    """Several weights in one launch, none a multiple of the tile (2 rows of 17 super-blocks: the launch that the multi-row
    decode kernel's mostly empty last item would slow down; with few outputs it stays there)."""
    case("split fused", rows, k, shapes)
    rng = np.random.default_rng(rows + k)
    made = [_weight(rng, "q4k", n, k) for n in shapes]
    x = normal(rng, (rows, k))
    bias = normal(rng, shapes[1])
    ys = ov.project_multi([w for _, w in made], t(x), rows=rows,
                          biases=[t(bias) if i == 1 else None for i in range(len(shapes))])
    for i, (y, (blocks, _)) in enumerate(zip(ys, made)):
        _check(y, _ref(orc, "q4k", x, rows, blocks, k, shapes[i], bias if i == 1 else None), f"job {i}")


def test_prepared_weight_keeps_the_kernel_that_reads_its_copy(orc):
    """200 rows of 512 inputs on the automatic choice: without its MFMA-ready copy the weight takes the split kernel, with it
    the tiled one. Which ran shows in the scratch of a fresh context (operand-ordered planes are laid out in whole 16-row
    tiles, row-major ones hold the bsums twice); the bits are the same."""
    case("prepared")
    rng = np.random.default_rng(12)
    rows, k, n = 200, 512, 2048
    blocks = set_subnormal_scales(random_q6k_blocks(rng, n * (k // 256)), q6=True).reshape(-1)
    x = normal(rng, (rows, k))
    ref = _ref(orc, "q6k", x, rows, blocks, k, n, None)
    live = {}
    for kind, prepare, kernel in (("plain", False, "auto"), ("prepared", True, "auto"), ("tiled", False, "tiled")):
        ctx = ov.Context(0)
        ctx.set_batched_kernel(kernel)
        w = ov.Q6KWeight(blocks, k, n, ctx=ctx)
        if prepare:
            w.prepare_mfma()
        _check(ov.project(w, t(x).view(-1), rows=rows), ref, kind)
        live[kind] = ctx.scratch_bytes()[0]
        del w
        ctx.close()
    assert live["prepared"] == live["tiled"] != live["plain"], live


@pytest.mark.parametrize("down", ["q4k", "q6k"])
@pytest.mark.parametrize("d,ff,rows", [(512, 2304, 35), (8960, 1280, 59)])  # down on the split kernel, on the panel kernel
def test_ffn_intermediate_matches_separate_calls(down, d, ff, rows):
    """The FFN's intermediate, quantised in the down kernel's operand order, against the same FFN with another kernel
    forced, which reads it row by row: the same quants, so the same bits."""
    case("ffn", down, d, ff, rows)
    rng = np.random.default_rng(5)
    gate, up = _weight(rng, "q4k", ff, d)[1], _weight(rng, "q4k", ff, d)[1]
    w = _weight(rng, down, d, ff)[1]
    x = t(normal(rng, (rows, d), 0.02))
    y = ov.ffn_swiglu(gate, up, w, x, rows)
    ctx = ov.default_context()
    ctx.set_batched_kernel("tiled")
    try:
        ref = ov.ffn_swiglu(gate, up, w, x, rows)
    finally:
        ctx.set_batched_kernel("auto")
    assert torch.equal(y.view(torch.int32), ref.view(torch.int32))


PANEL = [
    (5, 512, [12300]),           # tall, one tile: the weights' last 64-row group partial
    (17, 256, [12289]),          # one super-block, two tiles
    (48, 768, [6200, 6200]),     # an odd number of super-blocks, a gate/up pair
    (64, 512, [12288]),          # four full tiles
    (70, 1280, [4096, 512, 520]),  # not tall: two activation tiles of three, the last rows absent
    (59, 1280, [9130]),          # not tall, one activation tile of four, an odd number of short super-blocks
    (150, 768, [14330]),           # three activation tiles of four, the last of two and ragged; the last weight rows absent
    (250, 1280, [4000, 520]),      # four of four, an odd number of 210-byte blocks a row
]


@pytest.mark.parametrize("fmt", ["q4k", "q6k"])
@pytest.mark.parametrize("rows,k,shapes", PANEL)
def test_panel_projection_bit_exact(orc, fmt, rows, k, shapes):
    """The panel kernel (tall matrices; from 65 rows others): tile edges in both directions, one to five super-blocks."""
    case("panel", fmt, rows, k, shapes)
    rng = np.random.default_rng(rows * 31 + k)
    made = [_weight(rng, fmt, n, k) for n in shapes]
    x = normal(rng, (rows, k))
    biases = [normal(rng, n) if i == 0 else None for i, n in enumerate(shapes)]
    ys = ov.project_multi([w for _, w in made], t(x), rows=rows, biases=[None if b is None else t(b) for b in biases])
    for i, (y, (blocks, _)) in enumerate(zip(ys, made)):
        _check(y, _ref(orc, fmt, x, rows, blocks, k, shapes[i], biases[i]), f"job {i}")


PANEL_OF_FIVE = [
    (75, 256, 27990),    # five activation tiles a workgroup, the last rows of the fifth and the last weight rows absent
    (80, 512, 28100),    # five full tiles
    (150, 512, 28672),   # two workgroups of five
]


@pytest.mark.parametrize("rows,k,n", PANEL_OF_FIVE)
def test_panel_of_five_tiles_bit_exact(orc, rows, k, n):
    case("panel of five", rows, k, n)
    rng = np.random.default_rng(rows + k + n)
    blocks, w = _weight(rng, "q4k", n, k)
    x, bias = normal(rng, (rows, k)), normal(rng, n)
    y = ov.project(w, t(x).view(-1), rows=rows, bias=t(bias))
    _check(y, _ref(orc, "q4k", x, rows, blocks, k, n, bias), "panel of five")


@pytest.mark.parametrize("gate,down", [("q4k", "q4k"), ("q4k", "q6k"), ("q6k", "q6k")])
@pytest.mark.parametrize("E,k,rows,first", [
    (4, 2, 26, 8),                   # 13 pairs an expert: panel kernel where a projection cannot stream (Q6_K)
    (3, 2, 33, 16), (8, 3, 90, 16),  # 16 to 64: panel kernel both ways
    (6, 2, 150, 90),                 # the same, expert 0 with a second, ragged 64-row tile
    (4, 1, 300, 16),                 # 75: gate/up on the tiled kernel, down on the panel kernel
    (2, 2, 130, 16),                 # 129: Q4_K down on the tiled kernel too
])
def test_expert_groups_match_small_batches(E, k, rows, first, gate, down):
    """Expert groups on the panel and 64-row-tiled kernels (16 and more pairs an expert) against the same tokens in batches
    that the stream and small-M kernels take: every projection is bit-identical, and so are the outputs. Slots with an
    expert out of range or repeated add nothing; expert 0 gets a run of tokens, so that groups end on and off the tiles."""
    case("experts", E, k, rows, gate, down)
    rng = np.random.default_rng(E * 100 + rows)
    d, ff = 512, 768
    gw, up = ([_weight(rng, gate, ff, d)[1] for _ in range(E)] for _ in range(2))
    dw = [_weight(rng, down, d, ff)[1] for _ in range(E)]
    x = normal(rng, (rows, d), 0.02)
    idx = rng.integers(0, E, (rows, k)).astype(np.int32)
    idx[:first, 0] = 0
    idx[5, k - 1] = E + 3
    idx[rows - 1, 0] = -1
    wt = rng.random((rows, k)).astype(np.float32)
    y = ov.moe_ffn(gw, up, dw, t(x), rows, k, t(idx), t(wt)).reshape(rows, d)
    step = max(1, 8 * E // k - 1)
    for r in range(0, rows, step):
        m = min(step, rows - r)
        ref = ov.moe_ffn(gw, up, dw, t(x[r:r + m]), m, k, t(idx[r:r + m]), t(wt[r:r + m])).reshape(m, d)
        assert torch.equal(y[r:r + m].view(torch.int32), ref.view(torch.int32)), f"tokens {r} .. {r + m - 1}"


@pytest.mark.parametrize("E,k,rows", [(8, 2, 33), (64, 8, 190), (3, 1, 257), (5, 3, 1000), (2, 2, 1024), (2, 1, 1025)])
def test_plan_of_many_tokens(E, k, rows):
    """The one-launch router and grouping plan (65 entries to 1024 tokens, 8 slots) against batches of up to 64 entries,
    planned in one wave, and against the separate router; 1025 tokens take the general plan. Expert FFNs of one super-block
    each way, bit-identical outputs."""
    case("plan", E, k, rows)
    rng = np.random.default_rng(E + rows)
    d = ff = 256
    gate, up, down = ([_weight(rng, "q4k", d, ff)[1] for _ in range(E)] for _ in range(3))
    x, logits = normal(rng, (rows, d), 0.02), normal(rng, (rows, E))
    y, idx, wt = ov.moe_ffn_routed(gate, up, down, t(x), rows, t(logits), k)
    idx0 = torch.empty(rows * k, dtype=torch.int32, device=DEV)
    wt0 = torch.empty(rows * k, device=DEV)
    ov.MoeRouter.SelectTopK(t(logits), k, idx0, wt0, rows=rows)
    assert torch.equal(idx, idx0) and torch.equal(wt.view(torch.int32), wt0.view(torch.int32))
    # the caller's indices, one repeated and one out of range
    idx = idx.reshape(rows, k).clone()
    wt = wt.reshape(rows, k)
    if k > 1:
        idx[rows // 2, 1] = idx[rows // 2, 0]
    idx[rows - 1, k - 1] = E
    y2 = ov.moe_ffn(gate, up, down, t(x), rows, k, idx.reshape(-1), wt.reshape(-1)).reshape(rows, d)
    step = 64 // k
    for r in range(0, rows, step):
        m = min(step, rows - r)
        ref = ov.moe_ffn(gate, up, down, t(x[r:r + m]), m, k, idx[r:r + m].reshape(-1).contiguous(),
                         wt[r:r + m].reshape(-1).contiguous()).reshape(m, d)
        assert torch.equal(y2[r:r + m].view(torch.int32), ref.view(torch.int32)), f"tokens {r} .. {r + m - 1}"
    same = torch.ones(rows, dtype=torch.bool, device=DEV)
    same[rows // 2] = k == 1
    same[rows - 1] = False
    assert torch.equal(y.reshape(rows, d)[same].view(torch.int32), y2[same].view(torch.int32))
