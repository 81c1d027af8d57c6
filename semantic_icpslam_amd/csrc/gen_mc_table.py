"""Writes mc_table.inc: the marching-cubes triangle table the reference
meshes with (triangleTableHost, Mapping/Constant.h:39-296, the classic
published table), as one string of hexadecimal edge indices per sign case.

MeshScene's triangle lists can only equal the reference's with the same
table, so the table is carried over; this build derives the edge table and
the vertex counts from it and the corner signs instead of copying them.
Run once where the reference is mounted:

    python semantic_icpslam_amd/csrc/gen_mc_table.py /root/reference/Mapping/Constant.h
"""
import os
import re
import sys

# Corner pairs of the 12 cube edges in the reference's numbering
# (MeshScene.cu:200-291).
EDGE = [(0, 1), (1, 2), (2, 3), (3, 0), (4, 5), (5, 6), (6, 7), (7, 4), (0, 4), (1, 5), (2, 6),
        (3, 7)]


def read_table(path):
    src = open(path).read()
    start = src.index("triangleTableHost[256][16]")
    body = src[src.index("=", start): src.index("};", start)]
    vals = [int(x) for x in re.findall(r"-?\d+", body)]
    if len(vals) != 256 * 16:
        raise SystemExit(f"expected 4096 entries, found {len(vals)}")
    rows = [vals[16 * c: 16 * c + 16] for c in range(256)]
    for c, row in enumerate(rows):
        n = row.index(-1) if -1 in row else 16
        if n % 3 or any(v != -1 for v in row[n:]) or not all(0 <= v < 12 for v in row[:n]):
            raise SystemExit(f"case {c}: malformed row {row}")
        cut = {j for j, (a, b) in enumerate(EDGE) if ((c >> a) & 1) != ((c >> b) & 1)}
        if set(row[:n]) != cut:
            raise SystemExit(f"case {c}: triangles do not use exactly the cut edges")
    return [row[: row.index(-1) if -1 in row else 16] for row in rows]


def main():
    if len(sys.argv) != 2:
        raise SystemExit(__doc__)
    rows = read_table(sys.argv[1])
    out = os.path.join(os.path.dirname(os.path.abspath(__file__)), "mc_table.inc")
    with open(out, "w") as f:
        f.write("// Generated by gen_mc_table.py from the reference's triangle table\n"
                "// (Mapping/Constant.h:39-296): per sign case, the edge indices of its\n"
                "// triangles in hexadecimal, three per triangle.\n"
                "static constexpr const char* kMcTriangles[256] = {\n")
        for c in range(0, 256, 8):
            f.write("    " + " ".join('"%s",' % "".join("%x" % v for v in rows[k])
                                      for k in range(c, c + 8)) + "\n")
        f.write("};\n")
    print("wrote", out)


if __name__ == "__main__":
    main()
