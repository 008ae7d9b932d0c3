// The end of a synchronous call (vkhel_amd/csrc/call_wait.h) with a stand-in
// for the device: whatever the completion mark does, the call returns only
// after its work is done.
#include <cstdio>
#include <initializer_list>

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

// A program of `passes` passes: `calls` calls each, `gap` us of its own before a
// call and `between` more before a pass, and a synchronisation of the device
// behind each pass if `sync`.  Times of a call and of the synchronisation are
// the measured ones (call_wait.h).
struct Total {
	double us;
	long watched, calls;
};

template <class Watch, class End>
static Total program(int passes, int calls, double gap, double between, bool sync,
		Watch watch, End end) {
	double now = 1e6;
	long watched = 0;
	int unseen = 0;  // calls whose kernels the runtime has not seen finish
	for (int p = 0; p < passes; p++) {
		now += between;
		for (int c = 0; c < calls; c++) {
			now += gap;
			const bool w = watch((int64_t) (now * 1000));
			now += w ? 9.7 : 11.5;
			unseen = w ? unseen + 1 : 0;
			watched += w;
			end((int64_t) (now * 1000));
		}
		if (sync) {
			now += !unseen ? 0.2 : unseen <= 2 ? 8.8 : 25;
			unseen = 0;
		}
	}
	return Total{now - 1e6, watched, (long) passes * calls};
}

static bool check(int calls, double gap, double between, bool sync) {
	const int passes = 4000 / calls;
	vk::CallRun run;
	const Total rule = program(passes, calls, gap, between, sync,
			[&](int64_t now) { return run.watch(now); }, [&](int64_t now) { run.end(now); });
	const Total block = program(passes, calls, gap, between, sync,
			[](int64_t) { return false; }, [](int64_t) {});
	// a few calls alone: nothing watched; with synchronisations no slower than
	// blocking; without, all but the first calls watch
	const bool ok = between > 100 && calls <= 16 ? rule.watched == 0
		: sync || between > 100 ? rule.us < 1.03 * block.us
		: rule.watched > 0.95 * rule.calls;
	printf("%d calls, gap %.0f, between %.0f, sync %d: %ld of %ld watched, %.0f us, "
			"%.0f blocking %s\n", calls, gap, between, sync, rule.watched, rule.calls,
			rule.us, block.us, ok ? "ok" : "WRONG");
	return ok;
}

int main() {
	bool run = true;
	for (const int calls : {1, 2, 4, 5, 8, 16, 40})
		for (const double gap : {3.0, 6.0})
			for (const double between : {0.0, 10.0, 1000.0})
				for (const bool sync : {false, true})
					run &= check(calls, gap, between, sync);
	if (!run)
		return puts("model wrong"), 1;

	bool ok = returns_complete(true, 1, 8, 0);
	ok &= returns_complete(true, 8, 8, 0);
	ok &= returns_complete(true, 0, 8, 1);
	ok &= returns_complete(false, 0, 8, 1);
	puts(ok ? "model ok" : "model wrong");
	return ok ? 0 : 1;
}
