// The end of a synchronous call, apart from HIP (runtime.hip wait_call;
// tests/c/call_wait_model.cpp runs it on the host).
#pragma once

#include <cstdint>

namespace vk {

// Whether a synchronous call ends by a watched word: only in a run of calls
// that the program does not follow by synchronising the device itself.  A call
// that ends by the word is over sooner, but the runtime has not seen its
// kernels finish, and the next synchronisation of the stream or the device
// makes up for all of them: measured on MI355X, us, k calls of one small kernel
// and such a synchronisation, by the word / by hipStreamSynchronize: k = 1 8.7
// + 8.8 / 11.3 + 0.2, 2 17 + 9 / 23 + 0.2, 4 39 + 25 / 46 + 0.2, 8 79 + 26 / 92
// + 0.2, 16 158 + 28 / 185 + 0.2.
// So calls block until `need` of them have come one after the other.  Then they
// watch, until one comes late, or two of the last kBlocked take kMoreNs longer
// to come than any did while calls blocked: at least what a synchronisation
// between them costs then and did not before.  After that twice as many block.
struct CallRun {
	static constexpr int64_t kLateNs = 50000, kMoreNs = 7000;
	static constexpr uint32_t kBlocked = 16, kMostBlocked = 1024, kSettled = 64;

	// A call that waits at `now` (ns): true if it may watch.
	bool watch(int64_t now) {
		const int64_t gap = now - ended;
		if (!length || gap > kLateNs) {
			start();
		} else if (length <= need) {
			usual = gap > usual ? gap : usual;
		} else if (gap > usual + kMoreNs) {
			if (slow_at && length - slow_at < kBlocked) {
				need = 2 * need < kMostBlocked ? 2 * need : kMostBlocked;
				start();
			} else {
				slow_at = length;
			}
		} else if (length - (slow_at ? slow_at : need) >= kSettled) {
			need = kBlocked;
		}
		length += length < 0xffffffff;
		return length > need;
	}
	void end(int64_t now) {
		ended = now;
	}

private:
	void start() {
		length = slow_at = 0;
		usual = 0;
	}
	int64_t ended = 0;  // when the last call returned
	int64_t usual = 0;  // longest gap while the run's calls blocked
	uint32_t length = 0, need = kBlocked;  // of the run; blocked calls of one
	uint32_t slow_at = 0;  // the last slow call, 0: none
};

// Returns once a call's work is done.  mark() enqueues behind it what done()
// watches for, and is false if that was not enqueued; more() bounds the watch;
// block() waits in the runtime and returns a vkhel_status.  Whatever fails,
// nothing but done() or block() lets the call return: its work is on the stream
// already, and its caller reads the results.
template <class Mark, class Done, class More, class Block>
int watch_or_block(Mark mark, Done done, More more, Block block) {
	if (mark()) {
		do {
			if (done())
				return 0;
		} while (more());
	}
	return block();
}

}  // namespace vk
