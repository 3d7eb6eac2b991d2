"""The order of attn_prompt_kernel's row tiles (stack_attn_order.h): every tile of every head is one workgroup's, whatever the levels, the workgroups in each and the CUs are; where two share a
CU, a light tile shares a heavy one's."""
import os
import subprocess

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'trtllm-llama_amd', 'csrc', 'kernels', 'stack_attn_order.h')
CHECK = r'''
#include "%s"
#include <cstdio>
#include <vector>
using namespace tllm::kernels;
int main()
{
    for (int cus : {1, 7, 64, 256, 304})
        for (int per = 1; per <= 640; ++per)
            for (int tiles = 1; tiles <= 40; ++tiles)
            {
                const int turn = prompt_turn(tiles, per, cus);
                std::vector<int> seen(tiles, 0);
                for (int at = 0; at < tiles; ++at)
                {
                    const int level = prompt_level(at, turn, tiles);
                    if (level < 0 || level >= tiles || seen[level]++)
                        return std::printf("tiles %%d, per %%d, cus %%d: level %%d of %%d\n", tiles, per, cus, level, at), 1;
                    if (at < turn && level != at)
                        return std::printf("tiles %%d, per %%d, cus %%d: %%d is not the heaviest left\n", tiles, per, cus, at), 1;
                }
                if ((int64_t) tiles * per > 2 * cus)
                    continue;
                for (int at = turn; at + 1 < tiles; ++at) // the later, the heavier
                    if (prompt_level(at + 1, turn, tiles) != prompt_level(at, turn, tiles) - 1)
                        return std::printf("tiles %%d, per %%d, cus %%d: order behind %%d\n", tiles, per, cus, turn), 1;
            }
    return 0;
}
'''


def test_every_tile_is_one_workgroups(tmp_path):
    source, program = tmp_path / 'levels.cpp', str(tmp_path / 'levels')
    source.write_text(CHECK % HEADER)
    subprocess.run(['g++', '-std=c++17', '-O1', '-Wall', str(source), '-o', program], check=True)
    r = subprocess.run([program], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
