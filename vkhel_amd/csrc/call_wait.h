// The end of a synchronous call, apart from HIP (runtime.hip wait_call;
// tests/c/call_wait_model.cpp runs it on the host).
#pragma once

namespace vk {

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
