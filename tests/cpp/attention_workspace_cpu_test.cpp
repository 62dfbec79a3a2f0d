// The attention workspace (csrc/kernels/dispatch.hpp): one sized for the cache's
// length holds the split of every shorter context, and never shrinks as the
// context grows; a whole prefill's is what its launch uses.
#include "../../qwen3-runtime-byyourself_amd/csrc/kernels/dispatch.hpp"
#include "test_util.hpp"

#include <string>

using test::require;

namespace
{
    void body()
    {
        using namespace q3k;
        const int32_t heads[][2] = {{16, 8}, {32, 8}, {40, 8}, {64, 8}, {2, 1}, {4, 1}, {5, 1}, {8, 1}, {32, 1}};
        int64_t split = 0;
        for (const auto &h : heads)
            for (const int64_t B : {1, 2, 5, 16, 40, 64})
                for (const int64_t S : {1, 2, 7, 33, 100, 260, 512, 1024, 2048})
                {
                    int64_t before = 0;
                    for (int64_t cached = S; cached <= 32768; cached += cached / 32 + 1)
                    {
                        const std::string what = std::to_string(h[0]) + "/" + std::to_string(h[1]) + " heads, B " +
                                                 std::to_string(B) + ", S " + std::to_string(S) + ", " +
                                                 std::to_string(cached) + " keys";
                        const int64_t bytes = attention_workspace_bytes(B, S, h[0], h[1], cached);
                        const AttnSplit p = plan_attention_split(B, S, h[0], h[1], cached);
                        require(bytes >= before, what + ": less workspace than for a shorter context");
                        require((p.splits > 1) == (p.bytes > 0), what + ": a size without a split, or a split without");
                        require(bytes >= p.bytes, what + ": the split needs more than the workspace");
                        require(cached > S || bytes == p.bytes,
                                what + ": a whole prefill asks for what it does not use");
                        before = bytes;
                        split += p.splits > 1;
                    }
                }
        require(split > 1000, "the shapes cover split keys");
    }
} // namespace

int main() { return test::run("attention workspace test", body); }
