"""Times every tile kernel of one GEMM format against the kernel the library picks, on a grid of shapes,
and writes the per-shape table that the library's choice of tile consults.

    python -m hipkittens_amd.tile_sweep fp8|bf16|mxfp4            report on the 110-shape grid
    python -m hipkittens_amd.tile_sweep fp8|bf16|mxfp4 --emit     sweep the larger grid, rewrite the format's
                                                                  entries of csrc/tile_table.inc, then rebuild
    python -m hipkittens_amd.tile_sweep fp8|bf16|mxfp4 --draw N   report on N drawn shapes (what a rule fitted to a
                                                                  grid does between the grid's points)

For each shape it prints the GPU time (a HIP graph of 20 launches between two events, the launches rotating
over copies of B that exceed the memory-side cache, as a model's weights do; best of three replays, in two passes over the kernels, forwards and backwards) of the default choice (variant -1; with at
most 64 rows of A that can be the skinny kernel, csrc/gemm_skinny.h, instead of a tile kernel), of the 256x256,
128x128, 64x64, 192x256 and 256x192 tile kernels, and of the call with a workspace where the library would split K
without the skinny kernel, and marks the shapes where the default is more than 5 % behind the best tile kernel.

The choice of tile (`pick_gemm_tile`, csrc/gemm_small_tile.h) is a rule plus a generated table of exceptions,
the counterpart of the reference's tuned.yaml (analysis/baselines/gemm/utils/tuned.yaml: one tuned solution
per shape). `--emit` measures the five tile kernels on every shape of the larger grid and records the
shapes where the rule's choice (`hk_gemm_tile_shape(..., consult_table=0)`) is more than 3 % slower than
the fastest tile, keyed as the library looks them up: format, ceil(M / 64), ceil(N / 64), K-steps. The
table applies on devices with the CU count it was measured on; run it again after changing a tile kernel
or on another device, and rebuild the library.
"""
import math
import random
import re
import sys
from pathlib import Path

import torch

from . import _lib
from . import tk_kernel as tk

M_GRID = (16, 128, 256, 512, 768, 1024, 1536, 2048, 3072, 4096, 8192)
NK_GRID = ((1024, 1024), (2048, 2048), (4096, 4096), (8192, 8192), (4096, 14336), (14336, 4096),
           (2880, 2880), (7168, 2048), (2048, 7168), (5120, 5120))
# the grid of --emit: the report's grid and the shapes between its points
M_GRID_EMIT = (16, 64, 128, 192, 256, 384, 512, 640, 768, 1024, 1280, 1536, 2048, 2560, 3072, 4096, 6144, 8192)
NK_GRID_EMIT = NK_GRID + ((1536, 1536), (3072, 3072), (6144, 6144), (5760, 2880), (2880, 5760), (4096, 7168),
                          (7168, 4096), (1024, 8192), (8192, 1024), (2560, 10240),
                          (28672, 4096), (32768, 8192), (65536, 2880))   # (wide outputs: vocabulary projections)
FORMATS = {"fp8": 0, "bf16": 1, "mxfp4": 2}
TABLE_PATH = Path(__file__).resolve().parent / "csrc" / "tile_table.inc"
EMIT_MARGIN = 1.03


def _time_us(fn, iters=20):
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        fn()
        with torch.cuda.graph(graph, stream=stream):
            for _ in range(iters):
                fn()
    torch.cuda.synchronize()
    best = float("inf")
    for _ in range(3):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        graph.replay()
        e1.record()
        torch.cuda.synchronize()
        best = min(best, e0.elapsed_time(e1) / iters)
    return best * 1000.0


# B is the weight matrix of a layer: in a model it comes from HBM every time, because between two uses of it the
# other layers' weights have passed through the 256 MB memory-side cache. Timing one and the same B again and again
# would find it in that cache whenever it fits, and would tune the choice of tile for a case that does not occur.
# The calls therefore rotate over copies of B that together exceed the cache more than four times (A, the
# activations, stays).
ROTATE_BYTES = 1.2e9
ROTATE_MAX = 32


def _copies(b_bytes):
    return 1 if b_bytes >= 256e6 else min(ROTATE_MAX, int(ROTATE_BYTES // b_bytes) + 1)


def _problem(fmt, M, N, K, dev):
    C = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    turn = [0]

    def rotating(items):
        def nxt():
            turn[0] = (turn[0] + 1) % len(items)
            return items[turn[0]]
        return nxt

    lib = _lib.load_library()

    def pinned(st):
        _lib.check(st, "tile_sweep")

    if fmt == "fp8":
        A = torch.randn(M, K, device=dev).to(torch.float8_e4m3fn)
        B = rotating([torch.randn(N, K, device=dev).to(torch.float8_e4m3fn) for _ in range(_copies(N * K))])

        def run(tile=None, ws=None):
            if tile is None:
                return tk.dispatch_fp8_gemm(A, B(), C, 1.0, 1.0, workspace=ws)
            pinned(lib.hk_fp8_gemm_tile(A.data_ptr(), B().data_ptr(), C.data_ptr(), M, N, K, 1.0, 1.0, tile, tk._stream(A)))

        return run, tk.fp8_gemm_workspace_bytes(M, N, K)
    if fmt == "bf16":
        A = torch.randn(M, K, device=dev, dtype=torch.bfloat16)
        B = rotating([torch.randn(N, K, device=dev, dtype=torch.bfloat16) for _ in range(_copies(2 * N * K))])

        def run(tile=None, ws=None):
            if tile is None:
                return tk.dispatch_bf16_gemm(A, B(), C, workspace=ws)
            pinned(lib.hk_bf16_gemm_tile(A.data_ptr(), B().data_ptr(), C.data_ptr(), M, N, K, tile, tk._stream(A)))

        return run, tk.bf16_gemm_workspace_bytes(M, N, K)
    A = torch.randint(0, 256, (M, K // 2), dtype=torch.uint8, device=dev)
    As = torch.randint(120, 130, (M, K // 32), dtype=torch.uint8, device=dev)
    B = rotating([(torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, device=dev),
                   torch.randint(120, 130, (N, K // 32), dtype=torch.uint8, device=dev))
                  for _ in range(_copies(N * (K // 2 + K // 32)))])

    def run(tile=None, ws=None):
        b, bs = B()
        if tile is None:
            return tk.dispatch_mxfp4_gemm(A, As, b, bs, C, workspace=ws)
        pinned(lib.hk_mxfp4_gemm_tile(A.data_ptr(), As.data_ptr(), K // 32, b.data_ptr(), bs.data_ptr(), K // 32, C.data_ptr(),
                                      M, N, K, tile, tk._stream(A)))

    return run, tk.mxfp4_gemm_workspace_bytes(M, N, K)


def _k_steps(fmt, K):
    row_bytes = {"fp8": K, "bf16": 2 * K, "mxfp4": K // 2}[fmt]
    return (row_bytes + 127) // 128


def _write_table(fmt, entries, cus):
    """Replaces the entries of `fmt` in csrc/tile_table.inc; the other formats' entries stay."""
    code = FORMATS[fmt]
    kept = []
    for m in re.finditer(r"\{(\d+), (\d+), (\d+), (\d+), (\d+)\},", TABLE_PATH.read_text()):
        e = tuple(int(x) for x in m.groups())
        if e[0] != code and e[0] != 255:
            kept.append(e)
    rows = sorted(set(kept) | {(code,) + e for e in entries})
    lines = [
        "// Generated by `python -m hipkittens_amd.tile_sweep FORMAT --emit` (one run per format; each run rewrites its",
        "// format's entries). Shapes on which the rule of pick_gemm_tile (gemm_small_tile.h) was measured more than 3 % behind",
        "// another tile kernel: {format, ceil(M / 64), ceil(N / 64), K-steps, tile}; 192256 and 256192: the ring kernel's shorter",
        "// tiles.",
        f"constexpr int kTileTableCus = {cus};   // CU count of the device the sweeps ran on",
        "static constexpr TileTableEntry kTileTable[] = {",
        "    {255, 0, 0, 0, 0},   // (keeps the array non-empty)",
    ]
    lines += [f"    {{{e[0]}, {e[1]}, {e[2]}, {e[3]}, {e[4]}}}," for e in rows]
    lines.append("};")
    TABLE_PATH.write_text("\n".join(lines) + "\n")
    return len(rows)


# the tile kernels as hk_gemm_tile_shape names them: rows * 1000 + columns
TILES = (256256, 128128, 64064, 192256, 256192)


def _table_tile(tile):
    """A tile as the table names it: 256, 128 and 64 for the square ones."""
    return tile % 1000 if tile // 1000 == tile % 1000 else tile


def _drawn(n, rng):
    """Shapes over the range of the grids, log-uniform, in whole multiples of 64 columns and 128 elements of K mostly."""
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    while n:
        M, N, K = log(1, 8192), -(-log(512, 65536) // 64) * 64, -(-log(512, 16384) // 128) * 128
        N -= rng.choice((0, 0, 0, 16, 40))
        if M * N * K <= 6144 ** 3 and N * K <= 5e8:
            n -= 1
            yield M, N, K


def measure(run):
    """GPU time, us, of the default choice (None) and of every tile kernel. Every kernel is timed in two passes, the second
    in reverse order, and the faster one counts: single timings of one and the same kernel differ by 2-6 % with their
    position in the sequence (cold operands first, a warm chip last)."""
    order = (None,) + TILES
    t = {v: _time_us(lambda: run(v)) for v in order}
    for v in reversed(order):
        t[v] = min(t[v], _time_us(lambda: run(v)))
    return t


def _entries(measured):
    """Table entries from [(key, the rule's tile, {tile: us})]. A key stands for every shape with the same counts of blocks and
    K-steps (16 and 64 rows among them): it is listed where the rule is behind by the margin on one of its shapes, with the
    tile that is, and only if that tile is not the slower one on another."""
    by_key = {}
    for key, rule, t in measured:
        by_key.setdefault(key, []).append((rule, t))
    out = set()
    for key, shapes in by_key.items():
        rule, t = max(shapes, key=lambda s: s[1][s[0]] / min(s[1].values()))
        best = min(t, key=t.get)
        if t[rule] > EMIT_MARGIN * t[best] and all(s[best] <= 1.01 * s[r] for r, s in shapes):
            out.add(key + (_table_tile(best),))
    return out


def main(argv):
    args = [a for a in argv[1:] if not a.startswith("--")]
    flags = [a for a in argv[1:] if a.startswith("--")]
    draw = int(args.pop()) if flags == ["--draw"] and len(args) == 2 else 0
    if len(args) != 1 or args[0] not in FORMATS or flags not in ([], ["--emit"], ["--draw"]) or (flags == ["--draw"]) != (draw > 0):
        print(__doc__)
        return 2
    if not torch.cuda.is_available():
        raise RuntimeError("tile_sweep needs a GPU")
    fmt, dev, emit = args[0], "cuda:0", "--emit" in flags
    lib = _lib.load_library()
    grid = lambda ms, nks: [(M, N, K) for M in ms for N, K in nks]
    shapes = grid(M_GRID_EMIT, NK_GRID_EMIT) if emit else list(_drawn(draw, random.Random())) if draw else grid(M_GRID, NK_GRID)
    behind = rule_behind = 0
    measured = []
    for M, N, K in shapes:
        run, ws_bytes = _problem(fmt, M, N, K, dev)
        t = measure(run)
        best = min(TILES, key=lambda v: t[v])
        rule = int(lib.hk_gemm_tile_shape(FORMATS[fmt], M, N, K, 0))
        line = f"{fmt} {M} {N} {K}: default {t[None]:.1f} us, rule {rule} {t[rule]:.1f} |" + "".join(f" {v}: {t[v]:.1f}" for v in TILES)
        if ws_bytes and not emit:
            ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
            line += f" | split-K {_time_us(lambda: run(None, ws)):.1f}"
        if t[None] > 1.05 * t[best]:
            behind += 1
            line += "  <-- default more than 5 % behind"
        rule_behind += t[rule] > 1.05 * t[best]
        choice = int(lib.hk_gemm_tile_shape(FORMATS[fmt], M, N, K, 1))
        # (up to 64 rows the default can be the skinny kernel, which a time of its own shows: no tile to list there)
        if M > 64 or abs(t[None] / t[choice] - 1.0) <= 0.05:
            measured.append((((M + 63) // 64, (N + 63) // 64, _k_steps(fmt, K)), rule, {v: t[v] for v in TILES}))
        print(line, flush=True)
    print(f"{fmt}: more than 5 % behind the best tile kernel on {behind} (default) / {rule_behind} (rule alone) of {len(shapes)} shapes")
    if emit:
        entries = _entries(measured)
        cus = torch.cuda.get_device_properties(0).multi_processor_count
        n = _write_table(fmt, entries, cus)
        print(f"{len(entries)} entries for {fmt}; {TABLE_PATH} now holds {n}: rebuild the library "
              f"(python -m hipkittens_amd.build)")
    return 0


if __name__ == "__main__":
    sys.exit(main(sys.argv))
