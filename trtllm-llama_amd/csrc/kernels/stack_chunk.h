// Launchers of the chunked recurrences (stack_chunk.hip) for the row-by-row launchers beside them.
#pragma once
#include "stack_kernels.h"

namespace tllm
{
namespace kernels
{
constexpr int CHUNK_ROWS = 16;
// chunk slots of a step: every entry's chunks have places of their own (ent_first / 16 + entry + chunk)
inline int stack_chunk_slots(int tokens, int entries)
{
    return tokens / CHUNK_ROWS + entries + 1;
}
// 0: launched, -1: launch error, 1: not served (shape, row counts, scratch)
int launch_stack_chunk_hgrn2(const StackHgrnParams& p, hipStream_t stream);
int launch_stack_chunk_delta(const StackDeltaParams& p, hipStream_t stream);
int launch_stack_chunk_ssm(const StackSsmParams& p, hipStream_t stream);
} // namespace kernels
} // namespace tllm
