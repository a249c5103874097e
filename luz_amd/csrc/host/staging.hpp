// Copies between the caller's ordinary host memory and the device through pinned slots.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

namespace luzgpu
{
	// One transfer engine per context (a context is used by one thread at a time).
	//
	// The runtime copies unpinned memory through its own staging on one thread, which is slow
	// where the destination's pages are touched for the first time. Here kWorkers threads copy
	// between the caller's memory and kSlots pinned slots while the copy engine moves the slots
	// before or after. An FP64 1080p image up and down again (50 MB each way): 4.6 ms through the
	// runtime, 2.6 ms here; into fresh pages 6.6 and 3.6 ms; three workers and four slots do as
	// well as six and six. The threads live for one transfer and cost about 0.1 ms to start, so
	// transfers below kStagedBytes (0.2 ms) and pointers that HIP knows (pinned, managed or
	// device memory) go to the runtime.
	class	HostStaging
	{
		static constexpr size_t	kSlotBytes = size_t(2) << 20;
		static constexpr int	kSlots = 4;
		static constexpr int	kWorkers = 3;
		static constexpr size_t	kStagedBytes = size_t(4) << 20;

		char*	pinned = nullptr;
		hipEvent_t	events[kSlots] = {};

		// What the workers of a transfer share: `allowed` chunks may be copied, `done[slot]`
		// counts the pieces copied of the chunk in a slot, over all its chunks.
		struct	Transfer
		{
			std::atomic<size_t>	allowed{0};
			std::atomic<size_t>	done[kSlots] = {};
			std::vector<std::thread>	workers;

			static constexpr size_t	kStop = ~size_t(0);

			~Transfer()
			{
				allowed.store(kStop);	// only an error leaves workers waiting
				allowed.notify_all();
				for (std::thread& t : workers) t.join();
			}

			void	allow(size_t chunks)
			{
				allowed.store(chunks, std::memory_order_release);
				allowed.notify_all();
			}

			// until every piece of chunk c has been copied
			void	wait(size_t c, size_t pieces)
			{
				std::atomic<size_t>& d = done[c % kSlots];
				const size_t want = (c / kSlots + 1) * pieces;
				for (size_t v = d.load(std::memory_order_acquire); v < want; v = d.load(std::memory_order_acquire))
				{
					d.wait(v, std::memory_order_acquire);
				}
			}
		};

		bool	ready()
		{
			if (pinned) return true;
			if (hipHostMalloc(reinterpret_cast<void**>(&pinned), kSlots * kSlotBytes, hipHostMallocDefault) != hipSuccess)
			{
				(void)hipGetLastError();
				pinned = nullptr;
				return false;
			}
			for (hipEvent_t& e : events)
			{
				if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess)
				{
					(void)hipGetLastError();
					release();
					return false;
				}
			}
			return true;
		}

		void	release()
		{
			for (hipEvent_t& e : events)
			{
				if (e) (void)hipEventDestroy(e);
				e = nullptr;
			}
			if (pinned) (void)hipHostFree(pinned);
			pinned = nullptr;
		}

		static bool	ordinary(const void* p)
		{
			hipPointerAttribute_t a{};
			if (hipPointerGetAttributes(&a, p) != hipSuccess)
			{
				(void)hipGetLastError();
				return true;
			}
			return a.type == hipMemoryTypeUnregistered;
		}

		// Starts the workers: worker k copies piece k of every allowed chunk. Returns how many
		// there are.
		size_t	start(Transfer& t, char* host, size_t bytes, bool upload)
		{
			const size_t chunks = (bytes + kSlotBytes - 1) / kSlotBytes;
			std::atomic<size_t>* total = &pieces;
			total->store(0);
			t.workers.reserve(kWorkers);
			char* slots = pinned;
			for (int k = 0; k < kWorkers; k++)
			{
				try
				{
					t.workers.emplace_back([&t, host, bytes, upload, chunks, slots, total, k] {
						total->wait(0);
						const size_t n = total->load();
						for (size_t c = 0; c < chunks; c++)
						{
							for (size_t a = t.allowed.load(std::memory_order_acquire); a <= c; a = t.allowed.load(std::memory_order_acquire))
							{
								t.allowed.wait(a, std::memory_order_acquire);
							}
							if (t.allowed.load() == Transfer::kStop) return;
							const size_t size = std::min(kSlotBytes, bytes - c * kSlotBytes), step = ((size + n - 1) / n + 63) & ~size_t(63);
							const size_t at = std::min(size, step * static_cast<size_t>(k)), len = std::min(step, size - at);
							char* mine = host + c * kSlotBytes + at;
							char* slot = slots + (c % kSlots) * kSlotBytes + at;
							if (upload) std::memcpy(slot, mine, len);
							else std::memcpy(mine, slot, len);
							t.done[c % kSlots].fetch_add(1, std::memory_order_release);
							t.done[c % kSlots].notify_one();
						}
					});
				}
				catch (const std::exception&)
				{
					break;	// no more threads to be had: those that started do the work
				}
			}
			total->store(t.workers.empty() ? Transfer::kStop : t.workers.size());
			total->notify_all();
			return t.workers.size();
		}

		std::atomic<size_t>	pieces{0};

	public:
		HostStaging() = default;
		HostStaging(const HostStaging&) = delete;
		HostStaging& operator=(const HostStaging&) = delete;
		~HostStaging() { release(); }

		// Host to device on `st`; `host` may be reused on return.
		hipError_t	upload(void* device, const void* host, size_t bytes, hipStream_t st)
		{
			if (bytes < kStagedBytes || !ordinary(host) || !ready()) return hipMemcpyAsync(device, host, bytes, hipMemcpyHostToDevice, st);
			const size_t chunks = (bytes + kSlotBytes - 1) / kSlotBytes;
			for (hipEvent_t e : events)
			{
				if (const hipError_t err = hipEventSynchronize(e); err != hipSuccess) return err;
			}
			Transfer t;
			const size_t n = start(t, const_cast<char*>(static_cast<const char*>(host)), bytes, true);
			if (n == 0) return hipMemcpyAsync(device, host, bytes, hipMemcpyHostToDevice, st);
			t.allow(kSlots);
			for (size_t c = 0; c < chunks; c++)
			{
				t.wait(c, n);
				const size_t size = std::min(kSlotBytes, bytes - c * kSlotBytes);
				if (const hipError_t err = hipMemcpyAsync(static_cast<char*>(device) + c * kSlotBytes, pinned + (c % kSlots) * kSlotBytes, size,
						hipMemcpyHostToDevice, st); err != hipSuccess) return err;
				if (const hipError_t err = hipEventRecord(events[c % kSlots], st); err != hipSuccess) return err;
				if (c == 0) continue;	// the slot of chunk c - 1 is free once it has been sent
				if (const hipError_t err = hipEventSynchronize(events[(c - 1) % kSlots]); err != hipSuccess) return err;
				t.allow(c + kSlots);
			}
			return hipSuccess;
		}

		// Device to host on `st`; the data is there once `st` has been synchronized.
		hipError_t	readback(void* host, const void* device, size_t bytes, hipStream_t st)
		{
			if (bytes < kStagedBytes || !ordinary(host) || !ready())
			{
				return hipMemcpyAsync(host, device, bytes, hipMemcpyDeviceToHost, st);
			}
			const size_t chunks = (bytes + kSlotBytes - 1) / kSlotBytes;
			auto send = [&](size_t c) {
				const size_t size = std::min(kSlotBytes, bytes - c * kSlotBytes);
				if (const hipError_t err = hipMemcpyAsync(pinned + (c % kSlots) * kSlotBytes, static_cast<const char*>(device) + c * kSlotBytes,
						size, hipMemcpyDeviceToHost, st); err != hipSuccess) return err;
				return hipEventRecord(events[c % kSlots], st);
			};
			for (size_t c = 0; c < std::min<size_t>(chunks, kSlots); c++)
			{
				if (const hipError_t err = send(c); err != hipSuccess) return err;
			}
			Transfer t;
			const size_t n = start(t, static_cast<char*>(host), bytes, false);
			if (n == 0) return hipMemcpyAsync(host, device, bytes, hipMemcpyDeviceToHost, st);
			for (size_t c = 0; c < chunks; c++)
			{
				if (const hipError_t err = hipEventSynchronize(events[c % kSlots]); err != hipSuccess) return err;
				t.allow(c + 1);
				if (c == 0) continue;
				t.wait(c - 1, n);
				if (c - 1 + kSlots < chunks)
				{
					if (const hipError_t err = send(c - 1 + kSlots); err != hipSuccess) return err;
				}
			}
			t.wait(chunks - 1, n);
			return hipSuccess;
		}
	};
}
