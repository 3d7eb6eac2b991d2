// The order of attn_prompt_kernel's row tiles (stack_attn.hip): blockIdx.x / per counts levels, `per` (entries x heads) workgroups each, level 0 the heaviest tiles.  Plain C++, for host and
// device.
#pragma once
#include <cstdint>

namespace tllm
{
namespace kernels
{
// Up to two workgroups to a CU, workgroup i + CUs shares i's: from this level on the lightest come first.
constexpr int prompt_turn(int tiles, int64_t per, int64_t cus)
{
    return tiles * per <= 2 * cus ? (int) (cus / per) : tiles;
}
constexpr int prompt_level(int at, int turn, int tiles)
{
    return at < turn ? at : turn + tiles - 1 - at;
}
} // namespace kernels
} // namespace tllm
