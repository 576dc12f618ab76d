"""The GEMM's compiled tiles by the names MVLM_GEMM_TILE takes, read from the
launch table in gemm_mfma.hip: a name that is not in it forces nothing."""
import os
import re

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mvlm_amd", "csrc", "gemm_mfma.hip")


def _tiles():
    text = open(SOURCE).read()
    table = text[text.index("static const TileCfg kTiles[] = {"):]
    auto = int(re.search(r"constexpr int kAutoTiles = (\d+);", table).group(1))
    names = []
    for kind, args in re.findall(r"MVLM_(TILE|PINGPONG)\(([^)]*)\)", table[:table.index("};")]):
        v = [int(a) for a in args.split(",")[:6] if "." not in a]
        if kind == "PINGPONG":
            na, nb, ua, slots = v[:4]
            names.append(f"{na * ua}x{nb * 128}s{slots}w8")
        else:
            bm, bn, bk, stages, wm, wn = v
            names.append(f"{bm}x{bn}s{stages}w{wm * wn}" + (f"k{bk}" if bk != 64 else ""))
    return names, names[:auto]


COMPILED, AUTOMATIC = _tiles()
