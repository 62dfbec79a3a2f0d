// Internal control of the small-block device cache behind qwen3::Buffer.
#pragma once

#include <cstddef>

namespace qwen3::detail
{
    // While an instance lives, device Buffers made on this thread get fresh
    // device memory instead of a block kept for reuse.  For writers on a
    // stream other than the default one (the weight upload): a reused block
    // may still be read by work queued on the default stream, and a fresh
    // one cannot be.
    class FreshDeviceBlocks
    {
    public:
        FreshDeviceBlocks() noexcept;
        ~FreshDeviceBlocks();
        FreshDeviceBlocks(const FreshDeviceBlocks &) = delete;
        FreshDeviceBlocks &operator=(const FreshDeviceBlocks &) = delete;
    };

    // Device memory of one op's launches on the default stream, from the same
    // cache, which also keeps the larger ones of these (up to 16 MiB; 64 MiB per
    // device in all): a decode attention of 34 sequences of 64 / 8 heads needs
    // 6.8 MB in every layer of every token.
    class DeviceWorkspace
    {
    public:
        DeviceWorkspace(std::size_t bytes, int device);
        ~DeviceWorkspace();
        DeviceWorkspace(const DeviceWorkspace &) = delete;
        DeviceWorkspace &operator=(const DeviceWorkspace &) = delete;
        [[nodiscard]] void *data() const noexcept { return data_; } // null for 0 bytes

    private:
        void *data_;
        std::size_t bytes_;
        int device_;
    };
} // namespace qwen3::detail
