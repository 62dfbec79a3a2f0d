// Argmax over the last dimension for gfx950 (src/ops/argmax.cu:28-100 of the
// reference: bf16 rows, NaN counts as -inf, ties go to the smaller index,
// int32 indices).
//
// Every candidate becomes one 64-bit key: the bf16 bits mapped to an
// order-preserving unsigned value (NaN -> -inf, -0 -> +0, since the
// reference's float compare treats them as equal) in the high word and
// ~index in the low word, so "larger value, then smaller index" is a plain
// unsigned max.  One block of 1024 threads per row (rows strided over the
// grid): 128-bit loads of the row's aligned middle, a thread's maximum from the
// bits as packed 16-bit integers (a key per thread, not per element), wave and
// block maxima by DPP and through LDS.  When rows are long (kWholeRowColumns),
// too few to fill the GPU, and the caller gives a workspace, each row is cut
// into slices of whole 8-column vectors: one block per (row, slice) writes the
// slice's best key, and a second kernel takes the maximum over the slices of
// each row (the key order is total, so the result is the same).
#include "q3k_common.hpp"

#include <mutex>
#include <type_traits>

namespace q3k
{
    namespace
    {
        constexpr int kArgmaxBlock = 1024;

        __device__ __forceinline__ uint64_t argmax_key(uint32_t b, uint32_t index)
        {
            if ((b & 0x7fffu) > 0x7f80u)
                b = 0xff80u; // NaN -> -inf
            if (b == 0x8000u)
                b = 0u; // -0 -> +0
            const uint32_t ord = (b & 0x8000u) ? (~b & 0xffffu) : (b | 0x8000u);
            return (static_cast<uint64_t>(ord) << 32) | (0xffffffffu - index);
        }

        // Maximum over the wave's lanes, in every lane: DPP within 16-lane rows,
        // permlane swaps across them (VALU only, no LDS round trip).
        __device__ __forceinline__ uint32_t wave_max(uint32_t v)
        {
            auto max2 = [](uint32_t x, uint32_t y) __attribute__((always_inline)) { return x > y ? x : y; };
            v = max2(v, dpp_u<kDppQuadXor1>(v));
            v = max2(v, dpp_u<kDppQuadXor2>(v));
            v = max2(v, dpp_u<kDppHalfMirror>(v));
            v = max2(v, dpp_u<kDppMirror>(v));
            const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
            v = max2(r[0], r[1]);
            const auto q = __builtin_amdgcn_permlane32_swap(v, v, false, false);
            return max2(q[0], q[1]);
        }
        __device__ __forceinline__ uint64_t wave_max(uint64_t key)
        {
            const uint32_t hi = wave_max(static_cast<uint32_t>(key >> 32));
            const uint32_t lo = static_cast<uint32_t>(key >> 32) == hi ? static_cast<uint32_t>(key) : 0u;
            return (static_cast<uint64_t>(hi) << 32) | wave_max(lo);
        }

        // The 16-byte aligned middle of columns [begin, end) of row r: vectors
        // from column `first`, `count` of them; up to seven columns lie on either
        // side, column side(t) with thread t < 16 (-1: none).
        struct Middle
        {
            int64_t begin, end, first, count;
            __device__ __forceinline__ Middle(const uint16_t *r, int64_t b, int64_t e) : begin(b), end(e)
            {
                const int64_t odd = (reinterpret_cast<uintptr_t>(r + b) / 2) % 8;
                first = odd == 0 ? b : b + 8 - odd < e ? b + 8 - odd : e;
                count = (e - first) / 8;
            }
            __device__ __forceinline__ int64_t side(int t) const
            {
                const int64_t c = t < 8 ? begin + t : first + 8 * count + t - 8;
                return t < 16 && c < (t < 8 ? first : end) ? c : -1;
            }
        };

        constexpr int kUnroll = 5; // most vectors a thread has in flight
        typedef int16_t i16x2 __attribute__((ext_vector_type(2)));
        __device__ __forceinline__ uint32_t max_i16x2(uint32_t a, uint32_t b)
        {
            return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(i16x2, a), __builtin_bit_cast(i16x2, b)));
        }

        // Two bf16 with NaN as -inf.
        __device__ __forceinline__ uint32_t without_nan(uint32_t d)
        {
            const i16x2 inf = {0x7f80, 0x7f80};
            const uint32_t nan = __builtin_bit_cast(uint32_t, (inf - __builtin_bit_cast(i16x2, d & 0x7fff7fffu)) >> 15);
            return (nan & 0xff80ff80u) | (~nan & d);
        }

        // Largest of a vector's eight 16-bit integers.
        __device__ __forceinline__ int32_t max_of(uint32_t d0, uint32_t d1, uint32_t d2, uint32_t d3)
        {
            const uint32_t m = max_i16x2(max_i16x2(d0, d1), max_i16x2(d2, d3));
            const int32_t lo = static_cast<int16_t>(m & 0xffffu), hi = static_cast<int32_t>(m) >> 16;
            return lo > hi ? lo : hi;
        }

        // The largest value a thread has scanned, in its scan's own integers, and the
        // vector that holds its first occurrence.
        struct Scan
        {
            int32_t best;
            int32_t at;
            Vec8 vec;
            __device__ __forceinline__ void take(int32_t x, int32_t i, const Vec8 &v)
            {
                if (x > best)
                {
                    best = x;
                    at = i;
                    vec = v;
                }
            }
        };

        // 16 bits of bf16 as integers in order among positive values, everything else
        // below: the plain bits, signed.
        __device__ __forceinline__ int32_t positive_of(uint32_t bits)
        {
            return static_cast<int16_t>(without_nan(bits) & 0xffffu);
        }
        // In order among the others: 0x7fff less the magnitude's bits, so the zeros are
        // 0x7fff, -inf 0x7f and NaN below.
        __device__ __forceinline__ int32_t negative_of(uint32_t bits) { return static_cast<int32_t>(~bits & 0x7fffu); }

        // This thread's best key over columns [begin, end) of row r, or 0 (below every
        // candidate): the best of all threads' is the row's.
        //
        // The 16-byte aligned middle of the range goes UNROLL vectors a thread at a
        // time, all loaded before any is used; of the vectors seen only the one
        // holding the first maximum is kept.  A wave that sees a positive value in its
        // first vectors scans for those alone: a packed instruction for two columns (a
        // 64-bit key per element made the kernel VALU-bound, 64 x 151936: 7.5 us of
        // kernel, 12 instructions an element).  A wave that sees none scans for both,
        // and each of its threads takes the negative maximum if it finds nothing
        // positive; where that is -inf all its columns are -inf or NaN, and the first
        // of them is the one.  Nothing is read twice: a second pass with a key per
        // element over rows without a positive value or with a NaN took as long again
        // as one and a half reads (no positive value, 1 / 64 / 256 rows of 151936: 5.7 /
        // 6.8 / 13.6 us, 19.7 / 21.2 / 30.0 with the second pass; ordinary rows 4.6 / 6.2 /
        // 13.2 either way).
        template <int UNROLL>
        __device__ __forceinline__ uint64_t thread_best(const uint16_t *r, int64_t begin, int64_t end)
        {
            const Middle mid(r, begin, end);
            const int32_t nv = static_cast<int32_t>(mid.count); // below 2^28
            const Vec8 *rv = reinterpret_cast<const Vec8 *>(r + mid.first);
            int32_t tid = threadIdx.x;
            __asm__ volatile("" : "+v"(tid)); // nothing of a row is kept in registers for the next one
            const int64_t side = mid.side(tid);
            if (__ballot(tid < nv || side >= 0) == 0)
                return 0; // a short row: nothing for this wave
            const uint32_t side_bits = side >= 0 ? r[side] : 0u; // beside the vectors
            Scan p{0, 0, {}}, n{-1, 0, {}};
            bool negative = true; // the wave has seen no positive value in its first vectors
            for (int32_t i0 = 0; i0 < nv; i0 += UNROLL * kArgmaxBlock)
            {
                // past the end a thread reads the last vector once more
                Vec8 v[UNROLL];
                auto index = [&](int u) __attribute__((always_inline)) {
                    const int32_t i = i0 + tid + u * kArgmaxBlock;
                    return i < nv ? i : nv - 1;
                };
#pragma unroll
                for (int u = 0; u < UNROLL; ++u)
                    v[u] = load8<false>(rv + index(u));
                int32_t x[UNROLL], top = 0;
                auto maxima = [&]() __attribute__((always_inline)) {
#pragma unroll
                    for (int u = 0; u < UNROLL; ++u)
                    {
                        x[u] = max_of(v[u].d[0], v[u].d[1], v[u].d[2], v[u].d[3]);
                        top = x[u] > top ? x[u] : top;
                    }
                };
                maxima();
                if (__ballot(top > p.best) != 0)
                {
                    if (__ballot(top > 0x7f80) != 0)
                    {
#pragma unroll
                        for (int u = 0; u < UNROLL; ++u)
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                v[u].d[j] = without_nan(v[u].d[j]);
                        top = 0;
                        maxima();
                    }
#pragma unroll
                    for (int u = 0; u < UNROLL; ++u)
                        p.take(x[u], index(u), v[u]);
                }
                if (i0 == 0)
                    negative = __ballot(p.best > 0) == 0;
                if (negative)
#pragma unroll
                    for (int u = 0; u < UNROLL; ++u)
                    {
                        constexpr uint32_t kMagnitude = 0x7fff7fffu;
                        n.take(max_of(~v[u].d[0] & kMagnitude, ~v[u].d[1] & kMagnitude, ~v[u].d[2] & kMagnitude,
                                      ~v[u].d[3] & kMagnitude),
                               index(u), v[u]);
                    }
            }
            // the column of a scan's best, the side column included
            auto column = [&](Scan &s, bool any, auto value) __attribute__((always_inline)) {
                uint32_t at = 0;
                if (any)
                {
                    int e = 7;
#pragma unroll
                    for (int j = 7; j >= 0; --j)
                        e = value(j % 2 == 0 ? s.vec.d[j / 2] & 0xffffu : s.vec.d[j / 2] >> 16) == s.best ? j : e;
                    at = static_cast<uint32_t>(mid.first + 8 * static_cast<int64_t>(s.at) + e);
                }
                const int32_t x = value(side_bits);
                if (side >= 0 && (x > s.best || (x == s.best && static_cast<uint32_t>(side) < at)))
                {
                    s.best = x;
                    at = static_cast<uint32_t>(side);
                }
                return at;
            };
            const uint32_t p_at = column(p, p.best > 0, [](uint32_t b) __attribute__((always_inline)) { return positive_of(b); });
            if (p.best > 0)
                return argmax_key(static_cast<uint32_t>(p.best), p_at);
            if (!negative)
                return 0;
            const uint32_t n_at = column(n, n.best >= 0, [](uint32_t b) __attribute__((always_inline)) { return negative_of(b); });
            if (n.best > 0x7f)
                return argmax_key(0x8000u + static_cast<uint32_t>(0x7fff - n.best), n_at);
            if (n.best < 0)
                return 0; // no columns
            const int64_t first = mid.first + 8 * static_cast<int64_t>(tid < nv ? tid : nv - 1);
            return argmax_key(0xff80u, static_cast<uint32_t>(nv > 0 && (side < 0 || first < side) ? first : side));
        }

        // The best key of columns [begin, end) of row r, in every thread of wave 0;
        // the shared memory (a key a wave) is free again when the call returns.
        constexpr int kArgmaxWaves = kArgmaxBlock / kWave;
        template <int UNROLL>
        __device__ __forceinline__ uint64_t block_best(const uint16_t *r, int64_t begin, int64_t end, uint64_t *wave_key)
        {
            const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
            uint64_t best = wave_max(thread_best<UNROLL>(r, begin, end));
            if (lane == 0)
                wave_key[wave] = best;
            __syncthreads();
            if (wave == 0)
                best = wave_max(lane < kArgmaxWaves ? wave_key[lane] : uint64_t{0});
            __syncthreads();
            return best;
        }

        __device__ __forceinline__ int32_t key_index(uint64_t key)
        {
            return static_cast<int32_t>(0xffffffffu - static_cast<uint32_t>(key));
        }

        template <int UNROLL>
        __global__ __launch_bounds__(kArgmaxBlock) void argmax_kernel(const uint16_t *__restrict__ x,
                                                                      int32_t *__restrict__ out, int64_t rows,
                                                                      int64_t stride, int64_t n)
        {
            __shared__ uint64_t wave_key[kArgmaxWaves];
            for (int64_t row = blockIdx.x; row < rows; row += gridDim.x)
            {
                const uint64_t best = block_best<UNROLL>(x + row * stride, 0, n, wave_key);
                if (threadIdx.x == 0)
                    out[row] = key_index(best);
            }
        }

        // One block per (row, slice): part[row * slices + slice] = the best
        // key of columns [slice * slice_len, min(n, (slice + 1) * slice_len)).
        template <int UNROLL>
        __global__ __launch_bounds__(kArgmaxBlock) void argmax_slice_kernel(const uint16_t *__restrict__ x,
                                                                            uint64_t *__restrict__ part,
                                                                            int64_t stride, int64_t n,
                                                                            int32_t slices, int64_t slice_len)
        {
            __shared__ uint64_t wave_key[kArgmaxWaves];
            const int32_t row = static_cast<int32_t>(blockIdx.x) / slices;
            const int64_t begin = (static_cast<int32_t>(blockIdx.x) % slices) * slice_len;
            const int64_t end = begin + slice_len < n ? begin + slice_len : n;
            const uint64_t best = block_best<UNROLL>(x + row * stride, begin, end, wave_key);
            if (threadIdx.x == 0)
                part[blockIdx.x] = best;
        }

        // One wave per row: the maximum of its slice keys (slices <= 64).
        __global__ __launch_bounds__(kBlock) void argmax_merge_kernel(const uint64_t *__restrict__ part,
                                                                      int32_t *__restrict__ out, int64_t rows,
                                                                      int32_t slices)
        {
            const int64_t row = static_cast<int64_t>(blockIdx.x) * (kBlock / kWave) + threadIdx.x / kWave;
            if (row >= rows)
                return;
            const int lane = threadIdx.x % kWave;
            const uint64_t best = wave_max(lane < slices ? part[row * slices + lane] : uint64_t{0});
            if (lane == 0)
                out[row] = key_index(best);
        }

        // Rows are cut into slices when fewer than kTargetBlocks blocks would
        // run; a slice keeps at least kMinSlice columns (8 per thread).
        constexpr int64_t kTargetBlocks = 512;
        constexpr int64_t kMinSlice = 8 * kArgmaxBlock;
        constexpr int kMaxSlices = kWave;

        // Rows up to kWholeRowColumns long are searched whole, a block each: one launch.
        // Of at most kFewRows rows that holds up to kWholeFewRowsColumns only: their
        // slices, on CUs that would idle, then take less than the second launch.  (Whole
        // / slices in us, stream: 1 row of 200000 5.3 / 5.5, 230000 5.9 / 5.5, 262144 6.4 /
        // 5.5; 8 of 200000 5.6 / 5.6, 262144 6.7 / 5.4; 32 of 200000 6.6 / 6.9, 230000 7.7 /
        // 6.9.  40 of 230000 7.8 / 8.4, 262144 8.3 / 8.7, 300000 9.4 / 9.0; 64 of 151936 6.2 /
        // 7.5, 262144 9.1 / 9.2, 300000 10.0 / 9.8; 256 of 151936 13.2 / 15.1, 262144 27.6 /
        // 27.4.)
        constexpr int64_t kWholeRowColumns = int64_t{1} << 18;
        constexpr int64_t kWholeFewRowsColumns = 5 * 8 * kUnroll * kArgmaxBlock; // 204800: five rounds of loads
        constexpr int64_t kFewRows = 32;

        struct SlicePlan
        {
            int32_t slices = 1;
            int64_t slice_len = 0;
            int64_t bytes = 0;
        };

        SlicePlan plan_slices(int64_t rows, int64_t n)
        {
            SlicePlan p;
            if (rows <= 0 || rows >= kTargetBlocks || n <= (rows <= kFewRows ? kWholeFewRowsColumns : kWholeRowColumns))
                return p;
            int64_t want = (kTargetBlocks + rows - 1) / rows;
            if (want > n / kMinSlice)
                want = n / kMinSlice;
            if (want > kMaxSlices)
                want = kMaxSlices;
            if (want < 2)
                return p;
            const int64_t len = ((n + want - 1) / want + 7) / 8 * 8;
            const int64_t slices = (n + len - 1) / len;
            if (slices < 2 || rows > INT32_MAX / slices)
                return p;
            p.slices = static_cast<int32_t>(slices);
            p.slice_len = len;
            p.bytes = rows * slices * static_cast<int64_t>(sizeof(uint64_t));
            return p;
        }
    } // namespace
} // namespace q3k

namespace q3k
{
    namespace
    {
        // Shared checks of both argmax entry points (src/ops/argmax.cu:104-161).
        int validate_argmax(const uint16_t *x, const int32_t *out, int64_t rows, int64_t row_stride,
                            int64_t search_size)
        {
            if (rows < 0)
                return set_error(Q3K_ERR_INVALID_ARGUMENT, "argmax row count cannot be negative");
            if (row_stride <= 0)
                return set_error(Q3K_ERR_INVALID_ARGUMENT, "argmax reduction dimension must be positive");
            if (row_stride > INT32_MAX)
                return set_error(Q3K_ERR_INVALID_ARGUMENT, "argmax reduction dimension exceeds Int32 index range");
            if (search_size <= 0 || search_size > row_stride)
                return set_error(Q3K_ERR_INVALID_ARGUMENT, "valid reduction size is outside the last dimension");
            if (rows == 0)
                return Q3K_OK;
            if (x == nullptr || out == nullptr)
                return set_error(Q3K_ERR_INVALID_ARGUMENT, "argmax received a null pointer");
            if (!aligned_to(x, 2) || !aligned_to(out, 4))
                return set_error(Q3K_ERR_INVALID_ARGUMENT, "argmax pointers must be aligned to their element size");
            if (rows > INT64_MAX / row_stride)
                return set_error(Q3K_ERR_OVERFLOW, "argmax input size overflows");
            return Q3K_OK;
        }

        // Calls launch with the vectors a thread has in flight over `columns`: up to kUnroll,
        // as many as fill the fewest rounds (past the end each further one costs a thread
        // about twenty instructions: 64 rows of 1000 2.9 us, 3.3 with five; 1 of 20000 3.0
        // and 3.2; 42 of 86600, three rounds of four, 4.5 and 4.7 with five; 600 of 1000
        // 4.0, with the waves that have no columns going through the motions as well 5.1).
        template <typename F>
        void with_unroll(int64_t columns, F launch)
        {
            static_assert(kUnroll == 5, "instances");
            const int64_t vectors = (columns + 8 * kArgmaxBlock - 1) / (8 * kArgmaxBlock);
            const int64_t rounds = (vectors + kUnroll - 1) / kUnroll;
            switch ((vectors + rounds - 1) / rounds)
            {
            case 1: return launch(std::integral_constant<int, 1>{});
            case 2: return launch(std::integral_constant<int, 2>{});
            case 3: return launch(std::integral_constant<int, 3>{});
            case 4: return launch(std::integral_constant<int, 4>{});
            default: return launch(std::integral_constant<int, 5>{});
            }
        }

        // Launches for checked arguments: the sliced kernels when `part`
        // (8-byte aligned, room for plan.bytes) is given and the plan slices,
        // else one block per row.
        int launch_argmax(const uint16_t *x, int32_t *out, int64_t rows, int64_t row_stride, int64_t search_size,
                          const SlicePlan &plan, uint64_t *part, hipStream_t s)
        {
            if (plan.slices > 1 && part != nullptr)
            {
                with_unroll(plan.slice_len, [&](auto unroll) {
                    argmax_slice_kernel<decltype(unroll)::value>
                        <<<dim3(static_cast<unsigned>(rows * plan.slices)), dim3(kArgmaxBlock), 0, s>>>(
                            x, part, row_stride, search_size, plan.slices, plan.slice_len);
                });
                const int64_t per_block = kBlock / kWave;
                argmax_merge_kernel<<<dim3(static_cast<unsigned>((rows + per_block - 1) / per_block)), dim3(kBlock), 0,
                                      s>>>(part, out, rows, plan.slices);
                return check_launch("argmax_last_dimension");
            }
            const unsigned grid = static_cast<unsigned>(rows < 65535 ? rows : 65535);
            with_unroll(search_size, [&](auto unroll) {
                argmax_kernel<decltype(unroll)::value>
                    <<<dim3(grid), dim3(kArgmaxBlock), 0, s>>>(x, out, rows, row_stride, search_size);
            });
            return check_launch("argmax_last_dimension");
        }

        // The slice results of q3k_argmax_bf16_noalloc: a fixed array in
        // device memory, one copy per GPU, held until the process ends.  The
        // slice plan needs rows * slices * 8 bytes with rows * slices < 1024
        // (rows < 512, slices <= ceil(512 / rows)), so 8 KiB covers every
        // input; the array has twice that.  Every entry a call reads is
        // written by the same call first, so nothing needs clearing.
        constexpr int64_t kArgmaxScratchBytes = 16384;
        constexpr int kMaxScratchDevices = 64;
        std::mutex g_scratch_mutex;
        void *g_scratch_address[kMaxScratchDevices];  // per device, from hipGetSymbolAddress
    } // namespace

    static __device__ __align__(256) uint64_t scratch[kArgmaxScratchBytes / sizeof(uint64_t)];

    namespace
    {
        // The device address of `scratch` on the current GPU, looked up on
        // the first call per GPU (the host-side name is not a device address).
        int scratch_address(void **address)
        {
            int device = 0;
            if (hipGetDevice(&device) != hipSuccess)
                return set_error(Q3K_ERR_HIP, "argmax: no current GPU");
            if (device < 0 || device >= kMaxScratchDevices)
                return set_error(Q3K_ERR_INVALID_ARGUMENT, "argmax scratch supports GPUs 0 .. %d", kMaxScratchDevices - 1);
            std::lock_guard<std::mutex> lock(g_scratch_mutex);
            if (g_scratch_address[device] == nullptr)
            {
                void *p = nullptr;
                const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
                if (e != hipSuccess || p == nullptr)
                    return set_error(Q3K_ERR_HIP, "argmax scratch lookup failed on GPU %d: %s", device,
                                     hipGetErrorString(e));
                g_scratch_address[device] = p;
            }
            *address = g_scratch_address[device];
            return Q3K_OK;
        }
    } // namespace
} // namespace q3k

extern "C" int q3k_argmax_bf16(const uint16_t *x, int32_t *out, int64_t rows, int64_t row_stride,
                               int64_t search_size, void *workspace, int64_t workspace_bytes,
                               q3k_stream_t stream)
{
    using namespace q3k;
    if (const int st = validate_argmax(x, out, rows, row_stride, search_size))
        return st;
    if (workspace_bytes < 0)
        return set_error(Q3K_ERR_INVALID_ARGUMENT, "argmax workspace size cannot be negative");
    if (rows == 0)
        return Q3K_OK;
    const SlicePlan plan = plan_slices(rows, search_size);
    const bool sliced = plan.slices > 1 && workspace != nullptr && workspace_bytes >= plan.bytes &&
                        aligned_to(workspace, 8);
    return launch_argmax(x, out, rows, row_stride, search_size, plan,
                         sliced ? static_cast<uint64_t *>(workspace) : nullptr, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int q3k_argmax_bf16_noalloc(const uint16_t *x, int32_t *out, int64_t rows, int64_t row_stride,
                                       int64_t search_size, q3k_stream_t stream)
{
    using namespace q3k;
    if (const int st = validate_argmax(x, out, rows, row_stride, search_size))
        return st;
    if (rows == 0)
        return Q3K_OK;
    const SlicePlan plan = plan_slices(rows, search_size);
    uint64_t *part = nullptr;
    if (plan.slices > 1)
    {
        if (plan.bytes > kArgmaxScratchBytes)
            return set_error(Q3K_ERR_INVALID_ARGUMENT,
                             "argmax needs %lld bytes of scratch, more than the library's fixed %lld",
                             static_cast<long long>(plan.bytes), static_cast<long long>(kArgmaxScratchBytes));
        void *address = nullptr;
        if (const int st = scratch_address(&address))
            return st;
        part = static_cast<uint64_t *>(address);
    }
    return launch_argmax(x, out, rows, row_stride, search_size, plan, part, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int64_t q3k_argmax_workspace_bytes(int64_t rows, int64_t search_size)
{
    return q3k::plan_slices(rows, search_size).bytes;
}
