// The command ring (parallel-rdp_amd/csrc/rdp_ring.hpp) alone, on the CPU, for
// test_ring.py, which builds it with ThreadSanitizer too.  A command of this
// probe is len | producer << 8 | number << 12, then len - 1 words of its number.
// Each mode prints "ok", or what went wrong.
#include <stdio.h>
#include <stdlib.h>
#include <time.h>

#include <random>

#include "../parallel-rdp_amd/csrc/rdp_ring.hpp"

using namespace rdp_mi;

#ifdef __SANITIZE_THREAD__
// g++ 11's ThreadSanitizer does not know this call, which timed waits use, and takes
// the mutex to be held throughout; it knows pthread_cond_timedwait.
extern "C" int pthread_cond_clockwait(pthread_cond_t *c, pthread_mutex_t *m, clockid_t clock, const timespec *until)
{
	timespec from, now;
	clock_gettime(clock, &from);
	clock_gettime(CLOCK_REALTIME, &now);
	const int64_t ns = (until->tv_sec - from.tv_sec + now.tv_sec) * 1000000000ll + until->tv_nsec - from.tv_nsec + now.tv_nsec;
	const timespec at = { (time_t)(ns / 1000000000), (long)(ns % 1000000000) };
	return pthread_cond_timedwait(c, m, &at);
}
#endif

namespace {

struct Sink {
	uint32_t next[16] = {};
	uint64_t commands = 0, idles = 0;
	bool held = false;                          // as with passes waiting for the device
	std::atomic<uint32_t> delay_us{ 0 };  // of every chunk
	std::atomic<bool> bad{ false };

	size_t decode(const uint32_t *w, size_t n, bool &pending)
	{
		if (const uint32_t us = delay_us) std::this_thread::sleep_for(std::chrono::microseconds(us));
		size_t i = 0;
		while (i < n) {
			const uint32_t len = w[i] & 0xff, who = (w[i] >> 8) & 15, number = w[i] >> 12;
			if (len == 0 || len > 44) {
				bad = true;
				return n;
			}
			if (i + len > n) break;
			if (number != next[who]) bad = true;
			for (uint32_t k = 1; k < len; k++)
				if (w[i + k] != number) bad = true;
			next[who] = number + 1;
			commands++;
			i += len;
		}
		pending = held = commands & 1;
		return i;
	}
	void idle(bool &pending)
	{
		idles++;
		pending = held = false;
	}
};

struct RefSink {
	Sink &s;
	size_t decode(const uint32_t *w, size_t n, bool &pending) { return s.decode(w, n, pending); }
	void idle(bool &pending) { s.idle(pending); }
};

// `count` commands of producer `who`, pushed in runs of up to `most` words.
void produce(CommandRing &r, uint32_t who, uint32_t count, size_t most, uint32_t seed)
{
	std::mt19937 rng(seed);
	std::vector<uint32_t> run;
	for (uint32_t k = 0; k < count; k++) {
		const uint32_t len = 1 + rng() % 44;
		if (run.size() + len > most) {
			r.push(run.data(), run.size());
			run.clear();
			if (rng() % 64 == 0) std::this_thread::sleep_for(std::chrono::microseconds(rng() % 900));
		}
		run.push_back(len | who << 8 | k << 12);
		run.insert(run.end(), len - 1, k);
	}
	if (!run.empty()) r.push(run.data(), run.size());
}

int fail(const char *what)
{
	printf("%s\n", what);
	fflush(stdout);
	_Exit(1);  // threads may still run
}

int check(const Sink &s, const uint32_t *counts, int producers)
{
	if (s.bad) return fail("a command arrived broken or out of order");
	for (int i = 0; i < producers; i++)
		if (s.next[i] != counts[i]) return fail("commands are missing");
	printf("ok\n");
	return 0;
}

}  // namespace

int main(int argc, char **argv)
{
	const int mode = argc > 1 ? atoi(argv[1]) : 0;
	const uint32_t count = argc > 2 ? (uint32_t)atoi(argv[2]) : 20000;
	CommandRing r;
	Sink s;
	r.start([&] { r.run(RefSink{ s }); });
	if (mode == 0) {
		// Two producers and a third thread that drains, over many turns of the ring.
		const uint32_t counts[2] = { count, count };
		std::atomic<bool> done{ false };
		std::thread a([&] { produce(r, 0, count, kRingChunk, 1); }), b([&] { produce(r, 1, count, 44, 2); });
		std::thread d([&] {
			while (!done) r.drain();
		});
		a.join();
		b.join();
		r.drain();
		const bool left = r.busy();
		done = true;
		d.join();
		r.finish();
		if (left) return fail("busy after a drain");
		return check(s, counts, 2);
	}
	if (mode == 1) {
		// A full ring: every chunk takes longer than a waiting producer polls.
		s.delay_us = (uint32_t)(2 * kWaitPollUs);
		const uint32_t counts[2] = { count, count };
		std::thread a([&] { produce(r, 0, count, kRingChunk, 3); }), b([&] { produce(r, 1, count, kRingWords, 4); });
		a.join();
		b.join();
		r.finish();
		return check(s, counts, 2);
	}
	if (mode == 2) {
		// Ends with commands left in the ring: all of them are decoded first.
		s.delay_us = 3000;
		const uint32_t counts[1] = { count };
		produce(r, 0, count, kRingChunk, 5);
		r.finish();
		return check(s, counts, 1);
	}
	if (mode == 3) {
		// Single commands with pauses around the times the threads poll and sleep;
		// what waits for the device is handed over by the idle call.
		const uint32_t counts[1] = { count };
		for (uint32_t k = 0; k < count; k++) {
			const uint32_t w[2] = { 2 | k << 12, k };
			r.push(w, 2);
			if (k % 3 == 0) r.drain();
			std::this_thread::sleep_for(std::chrono::microseconds(k % 8 * 130));
		}
		std::this_thread::sleep_for(std::chrono::milliseconds(20));
		r.finish();
		if (count > 8 && !s.idles) return fail("no idle call");
		if (s.held) return fail("work left waiting");
		return check(s, counts, 1);
	}
	if (mode == 4) {
		// Submissions that fail, by the ring thread while it decodes or by the caller:
		// each flush reports its own, and one that works reports none.
		r.finish();
		struct Failing {
			std::mutex &lock;
			SubmitLog &log;
			std::atomic<int> &code;
			size_t decode(const uint32_t *w, size_t n, bool &pending)
			{
				std::this_thread::sleep_for(std::chrono::milliseconds(20));
				std::lock_guard<std::mutex> g(lock);
				for (size_t i = 0; i < n; i++)
					if (w[i] == kMetaFlush << 24 && code) log.failed(code, "ring");
				pending = false;
				return n;
			}
			void idle(bool &) {}
		};
		CommandRing q;
		std::mutex lock;
		SubmitLog log;
		std::atomic<int> code{ 0 };
		q.start([&] { q.run(Failing{ lock, log, code }); });
		const uint32_t w[1] = { 0 };
		const int codes[] = { 0, -3, -3, 0, -5, 0, 0, -3 };
		for (int want : codes) {
			code = want;
			q.push(w, 1);  // the ring thread is busy for 20 ms
			std::unique_lock<std::mutex> g(lock, std::defer_lock);
			const int got = flush_ring(&q, g, log, [] { return 0; });
			if (got != want || !g.owns_lock()) return fail("a failure on the ring thread is lost or made up");
		}
		for (int want : codes) {  // the ring is empty: the caller submits
			std::unique_lock<std::mutex> g(lock, std::defer_lock);
			const int got = flush_ring(want == -5 ? nullptr : &q, g, log, [&] {
				if (want) log.failed(want, "caller");
				return want;
			});
			if (got != want || !g.owns_lock()) return fail("a failure of the caller's own flush is lost or made up");
		}
		q.finish();
		if (log.first != -3 || log.first_msg != "ring" || log.last_msg != "caller" || log.failures != 8) return fail("the log");
		printf("ok\n");
		return 0;
	}
	if (mode == 5) {
		// Timed waits end at their timeout, the polled time included (the shortest of
		// ten: another thread may hold the core), and at once when what they wait for
		// or an error is there.
		r.finish();
		std::mutex m;
		std::condition_variable cv;
		std::atomic<uint64_t> done{ 0 };
		std::atomic<int> error{ 0 };
		auto ready = [&] { return done >= 1 || error != 0; };
		auto timed = [&](uint64_t us, bool want) {
			int64_t best = INT64_MAX;
			for (int i = 0; i < 10; i++) {
				const auto t0 = std::chrono::steady_clock::now();
				std::unique_lock<std::mutex> g(m, std::defer_lock);
				if (wait_ready(g, cv, us, ready) != want || !g.owns_lock()) fail("the wrong answer");
				const auto t = std::chrono::steady_clock::now() - t0;
				best = std::min<int64_t>(best, std::chrono::duration_cast<std::chrono::microseconds>(t).count());
			}
			return best;
		};
		for (uint64_t us : { 0ull, 300ull, 1000ull, 1500ull, 4000ull }) {
			const int64_t t = timed(us, false);
			if (t < (int64_t)us) return fail("a wait ended early");
			if (t > (int64_t)us + 700) return fail("a wait overran its timeout");
		}
		error = -3;
		if (timed(UINT64_MAX, true) > 300) return fail("an error is there and the wait goes on");
		error = 0;
		std::thread late([&] {
			std::this_thread::sleep_for(std::chrono::milliseconds(30));
			std::lock_guard<std::mutex> g(m);
			done = 1;
			cv.notify_all();
		});
		std::vector<std::thread> others;  // more waiters than may poll
		for (int i = 0; i < 12; i++)
			others.emplace_back([&] {
				std::unique_lock<std::mutex> g(m, std::defer_lock);
				if (!wait_ready(g, cv, UINT64_MAX, ready)) fail("the wrong answer");
			});
		late.join();
		for (auto &t : others) t.join();
		if (g_wait_pollers != 0) return fail("pollers left");
		printf("ok\n");
		return 0;
	}
	return fail("unknown mode");
}
