"""Pairs of a read's buckets (CPU: csrc/bucket_rows.hpp compiled for the host with the compiler's alignment
check, which ends the program at a load that is promised more than its address has): rows of
any number of maps, odd ones too, whose rows start on 8-byte boundaries only."""
import subprocess

from rabbitqcplus_amd import build

PROGRAM = '''#include "bucket_rows.hpp"
#include <cstdio>
#include <cstdlib>
int main(){
    for(int M = 1; M <= 48; M++){
        const int reads = 5;
        uint2* rows = static_cast<uint2*>(aligned_alloc(64, (size_t(reads) * M * sizeof(uint2) + 63) / 64 * 64));
        for(int i = 0; i < reads * M; i++) rows[i] = make_uint2(uint32_t(3 * i + 1), uint32_t(7 * i + 2));
        for(int r = 0; r < reads; r++){
            for(int u = 0; u < M + 4; u += 2){
                const uint4 x = bucketPair(rows + r * M, u, M);
                const uint2 a = u < M ? rows[r * M + u] : make_uint2(0u, 0u);
                const uint2 b = u + 1 < M ? rows[r * M + u + 1] : make_uint2(0u, 0u);
                if(x.x != a.x || x.y != a.y || x.z != b.x || x.w != b.y) return 1;
            }
        }
        free(rows);
    }
    std::puts("ok");
    return 0;
}
'''


def test_pairs_of_any_row(tmp_path):
    (tmp_path / "rows.hip").write_text(PROGRAM)
    exe = str(tmp_path / "rows")
    subprocess.run([build.HIPCC, "-O1", "-std=c++17", "--offload-host-only", "-Xarch_host", "-fsanitize=alignment",
                    "-Xarch_host", "-fsanitize-trap=alignment", f"-I{build.CSRC}", str(tmp_path / "rows.hip"), "-o", exe],
                   check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout == "ok\n", run.returncode
