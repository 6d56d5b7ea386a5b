"""best_segments (tf-approximate_amd/csrc/depthwise_segments.h) on the host: the choices of searches over every segment
count, for the costs that the depthwise window kernels have, without looking at every count."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "depthwise_segments.h"
#include <cstdio>
#include <initializer_list>
using namespace axc;

int main()
{
    // images x bands, workgroups per channel group, wavefronts' tasks per round, columns of the filter
    for (long nb : {1L, 3L, 64L, 1217L, 400000L})
        for (int wgs : {1, 8, 85, 256})
            for (int round : {16, 32, 128})
                for (int kw : {1, 5})
                    for (int ow : {1, 2, 3, 7, 8, 13, 56, 100, 224, 1021, 32767}) {
                        if (ow == 32767 && (wgs != 85 || round != 128))
                            continue;
                        int tries = 0;
                        auto cost = [&](const int count, const int length) {
                            ++tries;
                            const int64_t tasks = (int64_t)nb * count, per_wg = (tasks + wgs - 1) / wgs;
                            return tasks < (int64_t)1 << 31 ? (per_wg + round - 1) / round * (length + kw) : (int64_t)-1;
                        };
                        const Segments got = best_segments(ow, cost);
                        if (tries > 2 + 2 * 182 || (int64_t)tries * tries > 4 * (int64_t)ow + 8) {
                            printf("%d tries for %d columns\n", tries, ow);
                            return 1;
                        }
                        int count = 1, length = ow;
                        int64_t best = -1;
                        for (int ns = 1; ns <= ow; ++ns) {
                            const int sl = (ow + ns - 1) / ns, ne = (ow + sl - 1) / sl;
                            const int64_t c = cost(ne, sl);
                            if (c >= 0 && (best < 0 || c < best)) {
                                best = c;
                                count = ne;
                                length = sl;
                            }
                        }
                        if (got.count != count || got.length != length) {
                            printf("nb %ld wgs %d round %d kw %d ow %d: %d x %d, not %d x %d\n", nb, wgs, round, kw, ow, got.count,
                                   got.length, count, length);
                            return 1;
                        }
                    }
    // the 3x3 kernel's rule: 8 to 24 columns, fewer while every task has a wavefront
    for (long nb : {1L, 3L, 64L, 1217L, 400000L})
        for (int wgs : {1, 8, 85, 256})
            for (int ow = 1; ow < 260; ++ow) {
                auto per_wg = [&](const int count) { return ((int64_t)nb * count + wgs - 1) / wgs; };
                const Segments got = best_segments(ow, [&](const int count, const int length) {
                    if (length > 24 || (count > 1 && length < 8 && per_wg(count) > 16))
                        return (int64_t)-1;
                    return (per_wg(count) + 15) / 16 * (length + 3);
                });
                int count = 1, length = ow;
                int64_t best = -1;
                for (int ns = 1; ns <= ow; ++ns) {
                    const int sl = (ow + ns - 1) / ns, ne = (ow + sl - 1) / sl;
                    if (ns > 1 && sl < 8 && per_wg(ne) > 16)
                        break;
                    if (sl > 24 && (ow + ns) / (ns + 1) >= 8)
                        continue;
                    const int64_t c = (per_wg(ne) + 15) / 16 * (sl + 3);
                    if (best < 0 || c < best) {
                        best = c;
                        count = ne;
                        length = sl;
                    }
                }
                if (got.count != count || got.length != length) {
                    printf("3x3 nb %ld wgs %d ow %d: %d x %d, not %d x %d\n", nb, wgs, ow, got.count, got.length, count, length);
                    return 1;
                }
            }
    const Segments none = best_segments(9, [](int, int) { return (int64_t)-1; });
    return none.count == 1 && none.length == 9 ? 0 : 1;
}
"""


def test_same_choice_as_every_count_in_fewer_tries(tmp_path):
    src, exe = tmp_path / "segments.cpp", tmp_path / "segments"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "tf-approximate_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    res = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
