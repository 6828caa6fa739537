"""Render the tile tables of `feather_ops/tiles.py` into `csrc/feather_tiles.h`, or `--check` it is current.

Mirrors the reference's `tools/gen_tiles.py:36-69` flow (render / --check) for the gfx950 table. The tiles
module is loaded by path so this runs without torch or a built extension.
"""

import argparse
import importlib.util
import pathlib
import sys

HERE = pathlib.Path(__file__).resolve().parent
TILES = HERE / "feather_ops" / "tiles.py"
HEADER = HERE / "csrc" / "feather_tiles.h"


def load_tiles():
    spec = importlib.util.spec_from_file_location("_feather_tiles", TILES)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def render() -> str:
    tables = load_tiles()
    lines = [
        "// Generated by feather-ops_amd/gen_tiles.py from feather_ops/tiles.py. Do not edit.",
        "#pragma once",
        "",
        "// X(warps_m, warps_n, unroll_k, repeat_m, repeat_n, prefetch)",
    ]
    for macro, tiles in (("SCALED_MM_TILES", tables.SCALED_MM_TILES), ("GRAD_TILES", tables.GRAD_TILES)):
        lines.append(f"#define FEATHER_{macro}(X) \\")
        lines += [f"    X({', '.join(str(v) for v in tile)}) \\" for tile in tiles]
        lines.append("")
    return "\n".join(lines) + "\n"


def main() -> int:
    parser = argparse.ArgumentParser()
    parser.add_argument("--check", action="store_true", help="fail if the header is stale")
    args = parser.parse_args()
    text = render()
    if args.check:
        current = HEADER.read_text() if HEADER.exists() else ""
        if current != text:
            print(f"{HEADER} is stale: run python {pathlib.Path(__file__).name}", file=sys.stderr)
            return 1
        return 0
    if not HEADER.exists() or HEADER.read_text() != text:
        HEADER.write_text(text)
    return 0


if __name__ == "__main__":
    sys.exit(main())
