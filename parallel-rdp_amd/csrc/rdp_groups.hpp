// Groups of rounds that share their setup, TMEM and bin launches: which round
// begins one, and where its scratch goes.  Host code only.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace rdp_mi {

// Limits of a group: scratch (a frame of 8192 small triangles takes about 25 MB)
// and passes, whose index in the group has 15 bits of a span or bin work item; and
// rounds, since each one's uploads are compared with what the rasters of all the
// rounds before it in the group write.
constexpr size_t kGroupScratchBytes = 64u << 20;
constexpr uint32_t kGroupMaxPasses = 1u << 12, kGroupMaxRounds = 64;

// Walks a submission's rounds in order.
struct GroupWalk {
	// Every round its own scratch and a group of its own (rounds of many passes).
	bool own = false;
	size_t scratch = 0;   // end of the scratch taken so far: the next round's begins here
	uint32_t passes = 0, rounds = 0;  // of the group so far
	bool any = false;

	// Whether the next round begins a group.  Groups run one after another and
	// share one scratch region, so a group that begins starts at 0 again; but an
	// upscaled pass reads the TMEM snapshots its native pass (the round before) left
	// in its scratch.  A round with one stays in its group when the scratch is full,
	// and where its passes or rounds end the group it begins one behind the scratch taken.
	bool next(uint32_t round_passes, size_t round_scratch, bool upscaled)
	{
		const bool too_many = passes + round_passes > kGroupMaxPasses || rounds >= kGroupMaxRounds;
		const bool full = scratch + round_scratch > kGroupScratchBytes;
		const bool begins = own || !any || too_many || (full && !upscaled);
		if (begins) {
			passes = rounds = 0;
			if (!own && !upscaled) scratch = 0;
		}
		any = true;
		passes += round_passes;
		rounds++;
		return begins;
	}
};

}  // namespace rdp_mi
