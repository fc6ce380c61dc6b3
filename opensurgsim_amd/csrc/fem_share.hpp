// Admission of solves whose workgroups wait for each other (fem_resident.hip) to one GPU.
#pragma once

#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <mutex>

namespace femgpu {

// Such solves run side by side only while all of their workgroups have a CU: two grids that share too few could each hold
// CUs that the other's workgroups wait for. Workgroups go round-robin over the XCDs, whatever CUs are free there, so a solve of
// n workgroups takes ceil(n / 8) CUs of an XCD. First come, first served, so that a large solve is not kept out by small ones.
class ChipShare {
public:
    static constexpr int kXcds = 8;
    // Waits for `workgroups` CUs of `num_cus`; a solve that asks for more than there are is admitted alone. Held until release() or
    // the end.
    class Use {
    public:
        Use() = default;
        Use(ChipShare& chip, int workgroups, int num_cus) : chip_(&chip), cus_((workgroups + kXcds - 1) / kXcds) {
            const int all = std::max(1, num_cus / kXcds);
            std::unique_lock<std::mutex> lock(chip.mutex_);
            const uint64_t mine = chip.arrived_++;
            chip.turn_.wait(lock, [&] { return chip.admitted_ == mine && (chip.used_ == 0 || chip.used_ + cus_ <= all); });
            ++chip.admitted_;
            chip.used_ += cus_;
            chip.turn_.notify_all();
        }
        Use(Use&& other) noexcept : chip_(other.chip_), cus_(other.cus_) { other.chip_ = nullptr; }
        Use& operator=(Use&& other) noexcept {
            release();
            std::swap(chip_, other.chip_);
            std::swap(cus_, other.cus_);
            return *this;
        }
        ~Use() { release(); }
        void release() {
            if (!chip_) return;
            {
                std::lock_guard<std::mutex> lock(chip_->mutex_);
                chip_->used_ -= cus_;
            }
            chip_->turn_.notify_all();
            chip_ = nullptr;
        }

    private:
        ChipShare* chip_ = nullptr;
        int cus_ = 0;
    };

private:
    std::mutex mutex_;
    std::condition_variable turn_;
    uint64_t arrived_ = 0, admitted_ = 0;
    int used_ = 0;  // CUs of every XCD
};

}  // namespace femgpu
