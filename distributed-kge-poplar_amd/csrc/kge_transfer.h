// Bulk transfers between the caller's host arrays and the device, through pinned memory.
//
// The caller's arrays are pageable, so their bytes pass through pinned slots that the kernels
// address directly (a kernel gathers table rows and stores them to the slot across PCIe: no
// device-side staging buffer, no separate copy).  What bounds a large transfer then is the host's
// own memcpy between slot and array, most of all the first touch of a fresh array's pages, so it
// is split over a few threads and runs beside the next slot's kernel.
#pragma once

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <exception>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace kge {

// A handful of threads that all run one function at a time, woken once per transfer.  Created by
// the first large transfer of its owner, joined with it.  Where the system has no more threads to
// give there are fewer of them, or none: the callers go by size().
class CopyThreads {
   public:
    explicit CopyThreads(int n) {
        threads_.reserve(n);
        try {
            for (int i = 0; i < n; ++i) threads_.emplace_back([this, i] { loop(i); });
        } catch (const std::exception&) {
        }
    }
    ~CopyThreads() {
        {
            std::lock_guard<std::mutex> lock(mu_);
            quit_ = true;
        }
        wake_.notify_all();
        for (auto& t : threads_) t.join();
    }
    CopyThreads(const CopyThreads&) = delete;
    CopyThreads& operator=(const CopyThreads&) = delete;
    int size() const { return (int)threads_.size(); }
    void start(std::function<void(int)> fn) {
        {
            std::lock_guard<std::mutex> lock(mu_);
            fn_ = std::move(fn);
            running_ = (int)threads_.size();
            ++job_;
        }
        wake_.notify_all();
    }
    void wait() {
        std::unique_lock<std::mutex> lock(mu_);
        done_.wait(lock, [this] { return running_ == 0; });
    }

   private:
    void loop(int i) {
        long seen = 0;
        for (;;) {
            {
                std::unique_lock<std::mutex> lock(mu_);
                wake_.wait(lock, [&] { return quit_ || job_ != seen; });
                if (quit_) return;
                seen = job_;
            }
            fn_(i);
            std::lock_guard<std::mutex> lock(mu_);
            if (--running_ == 0) done_.notify_all();
        }
    }
    std::mutex mu_;
    std::condition_variable wake_, done_;
    std::function<void(int)> fn_;
    std::vector<std::thread> threads_;
    long job_ = 0;
    int running_ = 0;
    bool quit_ = false;
};

// The copies of one transfer: chunk k of `n_chunks` is bytes [k * chunk, ...) of the caller's array
// and lies in slot k % n_slots.  allow(k) lets the threads work on chunk k, wait(k) returns when it
// is copied; the calling thread takes a share of every chunk inside wait().
//
// A slot's kernel takes some 40 us, a thread's wake-up about as long: whoever waits looks on for kLook,
// giving its core to others meanwhile, and sleeps only after that, so that a transfer that stalls, or a
// host with fewer cores than threads, is not kept busy by the waiting.
class SlottedCopy {
   public:
    // to_slot: array -> slots, else slots -> array.  threads: null for a copy by the calling thread alone
    SlottedCopy(char* array, char* slots, size_t total, size_t chunk, int n_slots, bool to_slot, CopyThreads* threads)
        : array_(array), slots_(slots), total_(total), chunk_(chunk), n_slots_(n_slots), to_slot_(to_slot),
          threads_(threads), parts_(threads ? threads->size() + 1 : 1),
          left_(new std::atomic<int>[n_chunks()]) {
        for (size_t k = 0; k < n_chunks(); ++k) left_[k].store(parts_ - 1, std::memory_order_relaxed);
        if (threads_) threads_->start([this](int i) {
            for (size_t k = 0; k < n_chunks(); ++k) {
                await(may_, [&] { return allowed_.load(std::memory_order_acquire) > k || stop_.load(std::memory_order_relaxed); });
                if (allowed_.load(std::memory_order_acquire) <= k) return;  // stopped
                copy_part(k, i + 1);
                if (left_[k].fetch_sub(1, std::memory_order_acq_rel) == 1) signal(copied_);
            }
        });
    }
    ~SlottedCopy() {
        stop_.store(true);
        signal(may_);
        if (threads_) threads_->wait();
    }
    SlottedCopy(const SlottedCopy&) = delete;
    SlottedCopy& operator=(const SlottedCopy&) = delete;
    size_t n_chunks() const { return (total_ + chunk_ - 1) / chunk_; }
    void allow(size_t k) {
        allowed_.store(k + 1, std::memory_order_release);
        signal(may_);
    }
    void wait(size_t k) {
        copy_part(k, 0);
        await(copied_, [&] { return left_[k].load(std::memory_order_acquire) == 0; });
    }

   private:
    static constexpr std::chrono::microseconds kLook{200};
    template <class Ready>
    void await(std::condition_variable& cv, Ready&& ready) {
        const auto until = std::chrono::steady_clock::now() + kLook;
        while (!ready()) {
            if (std::chrono::steady_clock::now() >= until) {
                std::unique_lock<std::mutex> lock(mu_);
                cv.wait(lock, ready);
                return;
            }
            std::this_thread::yield();
        }
    }
    // (what was waited for is stored before: a waiter that is about to sleep holds the mutex until it does)
    void signal(std::condition_variable& cv) {
        if (!threads_) return;
        { std::lock_guard<std::mutex> lock(mu_); }
        cv.notify_all();
    }
    void copy_part(size_t k, int part) {
        const size_t n = std::min(chunk_, total_ - k * chunk_);
        // a chunk's parts end on whole pages of the array, wherever it starts: no two threads touch the
        // same new page of a chunk
        const uintptr_t base = (uintptr_t)(array_ + k * chunk_);
        auto cut = [&](int q) -> size_t {
            const uintptr_t page = (base + n * q / parts_) & ~(uintptr_t)4095;
            return q == parts_ ? n : page > base ? page - base : 0;
        };
        const size_t a = cut(part), b = cut(part + 1);
        if (a >= b) return;
        char* arr = array_ + k * chunk_ + a;
        char* slot = slots_ + (k % n_slots_) * chunk_ + a;
        if (to_slot_) std::memcpy(slot, arr, b - a);
        else std::memcpy(arr, slot, b - a);
    }
    char *array_, *slots_;
    size_t total_, chunk_;
    int n_slots_;
    bool to_slot_;
    CopyThreads* threads_;
    int parts_;
    std::unique_ptr<std::atomic<int>[]> left_;
    std::atomic<size_t> allowed_{0};
    std::atomic<bool> stop_{false};
    std::mutex mu_;
    std::condition_variable may_, copied_;
};

}  // namespace kge
