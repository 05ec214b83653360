"""The tiled GEMM's plan (block tile and K slices for a shape) on the CPU: the built library's own, at 256
CUs."""
import numpy as np

from common import run_cpp

ROOM = 64 << 20  # the slices' workspace of a Gpu
# Block tiles of launch.h by number: features, tokens, threads.
TILES = {1: (256, 256, 512), 2: (256, 128, 512), 3: (128, 128, 256), 4: (64, 64, 256), 5: (16, 16, 64)}


def plans(tmp_path, shapes, room=ROOM):
    out = run_cpp(tmp_path, "tile_plan.cpp", "".join(f"{r} {c} {n} {room}\n" for r, c, n in shapes))
    return [tuple(int(v) for v in line.split()) for line in out.splitlines()]


def test_a_planned_grid_is_one_that_hip_launches(tmp_path):
    """Operands up to 4 GiB and outputs up to the card's memory: a grid of at most 2^32 - 1 threads, in
    slices that K and the workspace hold."""
    shapes = []
    for cols in (8, 24, 64, 1024, 4096):
        for lr in np.arange(2, 28.2, 0.5):
            for ln in np.arange(1, 28.2, 0.5):
                rows, n = int(2 ** lr) // 4 * 4, int(2 ** ln)
                if rows >= 4 and rows * cols < 1 << 31 and n * cols < 1 << 31 and rows * n < 140 << 30:
                    shapes.append((rows, cols, n))
    for (rows, cols, n), (tile, slices) in zip(shapes, plans(tmp_path, shapes)):
        bf, bt, threads = TILES[tile]
        assert -(-rows // bf) * -(-n // bt) * slices * threads < 1 << 32, (rows, cols, n, tile, slices)
        assert slices == 1 or (slices <= -(-cols // 64) and slices * n * rows * 4 <= ROOM), (rows, cols, n, tile, slices)


def test_the_gpu_tests_shapes_reach_every_tile_that_the_plan_uses(tmp_path):
    """The tiles, in one piece and in slices, that the plan picks for the projections of the Qwen3 shapes by
    2 to 2048 rows are among those it picks for the GEMM tests of test_gpu_kernels.py."""
    from bench import QWEN3_0_6B, QWEN3_8B, QWEN3_32B
    from test_gpu_kernels import PLANNED, PREFILL, PREFILL_N
    shapes = []
    for m in (QWEN3_0_6B, QWEN3_8B, QWEN3_32B):
        h, i, d = m["hidden_size"], m["intermediate_size"], m["head_dim"]
        q, kv = m["num_attention_heads"] * d, m["num_key_value_heads"] * d
        shapes += [(r, c, n) for r, c in ((q + 2 * kv, h), (h, q), (2 * i, h), (h, i)) for n in range(2, 2049)]
    used = {(t, s > 1) for t, s in plans(tmp_path, shapes)}
    tested = {(t, s > 1) for t, s in plans(tmp_path, PLANNED + [(r, c, PREFILL_N) for _, r, c in PREFILL])}
    assert used <= tested, used - tested
