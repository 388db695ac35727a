"""The rules of trk_rules.h (table indexes of a draw, launch shapes, budgets),
compiled by the host compiler and evaluated here: no GPU needed."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def evaluate(tmp_path, body):
    """The numbers, line by line, that `body` prints with the rules in scope."""
    src, exe = tmp_path / "probe.cpp", tmp_path / "probe"
    src.write_text("#include <cmath>\n#include <cstdio>\n#include <initializer_list>\n#include \"trk_rules.h\"\n#include \"trk_philox.h\"\n"
                   "using namespace trk;\nint main() {\n" + body + "\nreturn 0; }\n")
    subprocess.run(["g++", "-std=c++17", "-ffp-contract=off", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "trekis-3_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    return [[float(x) for x in line.split()] for line in out.splitlines()]


def test_bucket_of_a_draw_stays_in_its_row(tmp_path):
    """The largest draw is 1: its bucket is the last one, and so is every
    bucket's upper end kept within the row of kShiBuckets + 1 entries."""
    rows = evaluate(tmp_path, """
        const uint64_t top = (1ull << 53) - 1;
        for (uint64_t u : {(uint64_t)0, top / 64, top / 2, top - 1, top}) {
            const double RN = ((double)u + 0.5) * 0x1.0p-53;
            printf("%.17g %d %d\\n", RN, shi_bucket(RN), kShiBuckets);
        }
        for (int b = 0; b < kShiBuckets; ++b)
            for (double RN : {b / (double)kShiBuckets, std::nextafter((b + 1) / (double)kShiBuckets, 0.0)})
                printf("%.17g %d %d\\n", RN, shi_bucket(RN), kShiBuckets);
    """)
    assert rows[4][0] == 1.0
    for RN, b, n in rows:
        assert 0 <= b < n and b / n <= RN <= (b + 1) / n


def test_transport_shape_uses_the_whole_gpu(tmp_path):
    """Every particle of a round fits its launch's lanes or is taken later by a
    full grid; no launch has more workgroups or threads than may be resident;
    and from 64 particles per SIMD on, the launch has a workgroup on at least
    four fifths of the CUs, with the waves spread evenly."""
    for cus, full in ((256, 768), (304, 768), (80, 512)):
        edges = [64 * 4 * cus, full * cus]
        ns = [1, 2, 3, 63, 64, 65, 4 * cus, 4 * cus + 1] + [e + d for e in edges for d in (-65, -64, -1, 0, 1, 64, 65)]
        ns += [int(64 * 4 * cus * 1.03 ** k) for k in range(60)] + [10 ** 7, 10 ** 9 + 7]
        rows = evaluate(tmp_path, "for (int64_t n : {%s}) {\nconst TransportShape s = transport_shape(n, %d, %d);\n"
                        'printf("%%lld %%lld %%d %%d\\n", (long long)n, (long long)s.blocks, s.threads, s.lane_cap);\n}'
                        % (", ".join(f"(int64_t){n}" for n in ns), cus, full))
        for n, blocks, threads, cap in rows:
            assert 1 <= blocks <= cus and threads % 64 == 0 and 64 <= threads <= full and 1 <= cap <= 64
            waves = threads / 64
            assert blocks * waves * cap >= min(n, full * cus), n
            if n >= 64 * 4 * cus:
                # one wave less per workgroup would not do, so at most a fifth of the CUs has none
                assert blocks >= 0.8 * cus, (n, blocks)
                assert (waves - 1) * 64 * cus < n, (n, waves)
