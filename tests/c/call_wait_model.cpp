// The end of a synchronous call (vkhel_amd/csrc/call_wait.h) with a stand-in
// for the device: whatever the completion mark does, the call returns only
// after its work is done.
#include <cstdio>

#include "call_wait.h"

// A call whose mark is enqueued or not, whose work ends at the `ends`-th look
// (0: only in block()), watched for `looks` looks.
static bool returns_complete(bool enqueued, int ends, int looks, int want_blocks) {
	int seen = 0, blocks = 0;
	bool complete = false;
	const int rc = vk::watch_or_block([&] { return enqueued; },
			[&] { return complete = enqueued && ends && ++seen >= ends; },
			[&] { return --looks > 0; },
			[&] { blocks++; complete = true; return 0; });
	const bool ok = rc == 0 && complete && blocks == want_blocks;
	printf("enqueued=%d ends=%d: rc=%d complete=%d blocks=%d %s\n", enqueued, ends,
			rc, complete, blocks, ok ? "ok" : "WRONG");
	return ok;
}

int main() {
	bool ok = returns_complete(true, 1, 8, 0);
	ok &= returns_complete(true, 8, 8, 0);
	ok &= returns_complete(true, 0, 8, 1);
	ok &= returns_complete(false, 0, 8, 1);
	puts(ok ? "model ok" : "model wrong");
	return ok ? 0 : 1;
}
