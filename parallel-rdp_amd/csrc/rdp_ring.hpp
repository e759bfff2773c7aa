// Command ring of one processor (CommandRing, command_ring.cpp:31-134):
// rdp_mi_enqueue_command copies complete commands in, and the processor's
// ring thread decodes them, a chunk at a time.  Long lists are handed
// over in chunks, so decoding starts with the first and copying (block moves,
// not word by word) never waits for the whole ring.  Private
// meta commands ride in the same ring so they stay ordered with the RDP
// commands (Op::MetaSignalTimeline and Op::MetaFlush, rdp_common.hpp:41-42).
// Host code only, without the GPU's headers.
#pragma once

#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace rdp_mi {

constexpr uint32_t kMetaSignal = 1, kMetaFlush = 2;
// 256 KB stay in the two cores' caches.  (A ring that holds a whole frame, 1 MB,
// and word vectors kept from frame to frame cost 130 us of a 640x480 two-cycle
// frame, 515 against 385 us, on a busy host: each frame then walks memory that
// has left the caches, where the allocator hands out what was just freed.)
constexpr size_t kRingWords = 1u << 16;
constexpr size_t kRingChunk = 1u << 12;

// Waits for something another thread or the GPU finishes within a frame poll
// before they sleep: waking a thread whose core has gone idle took 50 us and more
// here, two or three times a frame.  Callers poll for kWaitPollUs, a ring thread
// without work for kRingPollUs; only kWaitPollers and kRingPollers of them at a
// time, so that many processors do not keep every core busy.
constexpr int64_t kWaitPollUs = 1000, kRingPollUs = 400;
constexpr int kWaitPollers = 4, kRingPollers = 2;
inline std::atomic<int> g_wait_pollers{ 0 }, g_ring_pollers{ 0 };
template <typename Pred>
bool poll_for(int64_t us, Pred done)
{
	const auto t0 = std::chrono::steady_clock::now();
	for (;;) {
		for (int i = 0; i < 64; i++) {
			if (done()) return true;
			__builtin_ia32_pause();
		}
		if (std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(us)) return false;
	}
}

// The same where fewer than `most` threads poll already; otherwise one look.
template <typename Pred>
bool poll_among(std::atomic<int> &pollers, int most, int64_t us, Pred done)
{
	const bool polls = ++pollers <= most;
	const bool ok = polls ? poll_for(us, done) : done();
	--pollers;
	return ok;
}

// Waits for `ready` (atomics changed under g's mutex, announced through cv) for
// timeout_us at most, the time it polls included; UINT64_MAX: as long as it takes.
// g holds its mutex on return.
template <typename Ready>
bool wait_ready(std::unique_lock<std::mutex> &g, std::condition_variable &cv, uint64_t timeout_us, Ready ready)
{
	const auto start = std::chrono::steady_clock::now();
	const int64_t us = (int64_t)std::min<uint64_t>(timeout_us, 1ull << 50);
	poll_among(g_wait_pollers, kWaitPollers, std::min(us, kWaitPollUs), ready);
	g.lock();
	if (timeout_us != UINT64_MAX) return cv.wait_until(g, start + std::chrono::microseconds(us), ready);
	cv.wait(g, ready);
	return true;
}

class CommandRing {
public:
	// Copy complete commands (n <= kRingWords words) in; waits for space.
	void push(const uint32_t *w, size_t n)
	{
		std::lock_guard<std::mutex> pg(push_lock);
		if (write_count + n > read_count + kRingWords)
			wait_for([&] { return write_count + n <= read_count + kRingWords; });
		const size_t pos = (size_t)(write_count & (kRingWords - 1)), flat = std::min(n, kRingWords - pos);
		memcpy(words.get() + pos, w, flat * 4);
		memcpy(words.get(), w + flat, (n - flat) * 4);
		write_count += n;
		if (sleeping) {
			std::lock_guard<std::mutex> g(lock);
			cv.notify_one();
		}
	}

	// Wait until everything pushed so far has been decoded (CommandRing::drain,
	// command_ring.cpp:63-69).
	void drain()
	{
		const uint64_t end = write_count;
		wait_for([&] { return read_count >= end; });
	}

	// Whether the ring holds commands not decoded yet.
	bool busy() const { return read_count != write_count; }

	// The ring thread's loop (CommandRing::thread_loop, command_ring.cpp:86-134)
	// until finish() and an empty ring.  sink.decode(words, n, pending) takes
	// complete commands off the front of n words, returns how many words they are,
	// and says whether work waits to be handed to the device; when it does and no
	// command arrives for 500 us, sink.idle(pending) hands it over (the
	// reference's MetaIdle).
	template <typename Sink>
	void run(Sink &&sink)
	{
		std::vector<uint32_t> local(kRingChunk);
		bool pending = false;
		auto has_work = [this] { return write_count != read_count || stop; };
		for (;;) {
			bool idle = false;
			if (!has_work()) {
				if (!pending) poll_among(g_ring_pollers, kRingPollers, kRingPollUs, has_work);
				std::unique_lock<std::mutex> g(lock);
				sleeping = true;
				if (pending)
					idle = !cv.wait_for(g, std::chrono::microseconds(500), has_work);
				else
					cv.wait(g, has_work);
				sleeping = false;
			}
			if (idle) {
				sink.idle(pending);
				continue;
			}
			const uint64_t at = read_count;
			size_t n = (size_t)(write_count - at);
			if (n == 0) break;  // finish() was called, ring empty
			// The first commands, about kRingChunk words of them, so that producers get
			// their space back while decoding goes on, from a flat copy in the thread's
			// own memory (14 us of 715 KB).
			n = std::min(n, kRingChunk);
			const size_t pos = (size_t)(at & (kRingWords - 1)), flat = std::min(n, kRingWords - pos);
			memcpy(local.data(), words.get() + pos, flat * 4);
			memcpy(local.data() + flat, words.get(), (n - flat) * 4);
			read_count += sink.decode(local.data(), n, pending);
			if (waiters) {
				std::lock_guard<std::mutex> g(lock);
				progress.notify_all();
			}
		}
	}

	template <typename Loop>
	void start(Loop loop)
	{
		thr = std::thread(loop);
	}
	// Decode what is left and end the thread; nothing is pushed afterwards.
	void finish()
	{
		{
			std::lock_guard<std::mutex> g(lock);
			stop = true;
			cv.notify_all();
		}
		if (thr.joinable()) thr.join();
	}

private:
	// Waits until the ring thread has come as far as `reached` asks.
	template <typename Pred>
	void wait_for(Pred reached)
	{
		if (poll_among(g_wait_pollers, kWaitPollers, kWaitPollUs, reached)) return;
		std::unique_lock<std::mutex> g(lock);
		waiters++;
		progress.wait(g, reached);
		waiters--;
	}

	std::unique_ptr<uint32_t[]> words{ new uint32_t[kRingWords] };
	// Words copied in, words decoded.  A chunk changes hands through these alone:
	// under a common lock, the two threads put each other to sleep up to 18 times
	// a frame.  `lock` is for sleeping and waking; a thread announces that it
	// sleeps before it looks at the counts a last time, and the other one looks
	// for that after it has changed them.
	std::atomic<uint64_t> write_count{ 0 }, read_count{ 0 };
	std::atomic<bool> sleeping{ false };  // the ring thread
	std::atomic<int> waiters{ 0 };        // producers and drains
	std::mutex push_lock;                 // one producer at a time
	std::mutex lock;
	std::condition_variable cv;           // data for the ring thread
	std::condition_variable progress;     // space for producers, completion for drains
	std::thread thr;
	std::atomic<bool> stop{ false };
};

// A processor's failed submissions (under its lock).  The ring thread's have no
// caller to return to: the first one's code and message go to the next timeline
// signal; the count and the last one's tell a caller whether one failed since it
// last looked.
struct SubmitLog {
	int first = 0, last = 0;
	std::string first_msg, last_msg;
	uint64_t failures = 0;

	void failed(int err, const std::string &msg)
	{
		if (!first) {
			first = err;
			first_msg = msg;
		}
		last = err;
		last_msg = msg;
		failures++;
	}
};

// Submits everything pushed so far and returns 0 or the code of a submission
// that failed meanwhile, on whichever thread.  A ring thread still decoding submits
// its own passes, with their words in its core's caches; `flush` does it
// otherwise.  g holds the processor's lock on return.
template <typename Flush>
int flush_ring(CommandRing *ring, std::unique_lock<std::mutex> &g, const SubmitLog &log, Flush flush)
{
	g.lock();
	const uint64_t seen = log.failures;
	g.unlock();
	if (ring && ring->busy()) {
		const uint32_t w[1] = { kMetaFlush << 24 };
		ring->push(w, 1);
		ring->drain();
	}
	g.lock();
	if (int err = flush()) return err;
	return log.failures != seen ? log.last : 0;
}

}  // namespace rdp_mi
