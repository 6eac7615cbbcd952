"""Where int4_head_rows_kernel keeps its rows in LDS (async-gpu_amd/csrc/int4_head_layout.h), compiled by itself: no GPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_operands_are_read_from_what_was_staged(tmp_path):
    """Every place of every batch that the ring asks for, the last batch's beyond the last group among them, lies inside the rows' bytes; every group's operand is
    where its pieces were put, and no two pieces share a place."""
    src, exe = tmp_path / "layout.cpp", tmp_path / "layout"
    src.write_text('''
#include <cstdio>
#include <vector>
#include "int4_head_layout.h"
template <int SETS> int check(int rows, int K) {
    const int groups = K / 32, bytes = (int)hr_rows_bytes(rows, K), pieces = SETS > 0 ? 1 : 3, sets = SETS > 0 ? SETS : 1;
    std::vector<int> put(bytes / 16, -1);
    for (int run = 0; run < K / 8; ++run)
        for (int row = 0; row < rows; ++row)
            for (int piece = 0; piece < 3; ++piece) {
                const int at = hr_piece_at<SETS>(groups, run, row, piece);
                if (at < 0 || at + 16 > bytes || at % 16 || put[at / 16] != -1) return std::printf("staged: rows %d K %d run %d row %d\\n", rows, K, run, row);
                put[at / 16] = (run * 16 + row) * 3 + piece;
            }
    for (int g = 0; g < groups; g += HR_AHEAD)
        for (int u = 0; u < HR_AHEAD; ++u)
            for (int set = 0; set < sets; ++set)
                for (int piece = 0; piece < pieces; ++piece)
                    for (int lane = 0; lane < 64; ++lane) {
                        const int kq = lane >> 4, c16 = lane & 15, at = hr_operand_at<SETS>(groups, g, u, set, piece, kq, c16);
                        if (at < 0 || at + 16 > bytes || at % 16) return std::printf("read: rows %d K %d group %d at %d of %d\\n", rows, K, g + u, at, bytes);
                        const int row = SETS > 0 ? 4 * set + c16 / 4 : c16, pc = SETS > 0 ? c16 % 4 : piece;
                        if (g + u < groups && row < rows && pc < 3 && put[at / 16] != ((4 * (g + u) + kq) * 16 + row) * 3 + pc)
                            return std::printf("other: rows %d K %d group %d row %d\\n", rows, K, g + u, row);
                    }
    return 0;
}
int main() {
    int bad = 0;
    for (int rows = 2; rows <= 16; ++rows)
        for (int K = 32; K <= 2048; K += 32) bad |= hr_sets(rows) == 1 ? check<1>(rows, K) : hr_sets(rows) == 2 ? check<2>(rows, K) : check<0>(rows, K);
    return bad ? 1 : 0;
}
''')
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "async-gpu_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout[:2000]
