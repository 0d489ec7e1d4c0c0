// Space of the block lists (16-byte entries): a fixed region for the low bins, then the high bins',
// each with 16 lists as long as the bin's own (its list positions). Plain arithmetic, shared by
// the kernels and the host.
#pragma once

#include <stdint.h>

namespace lucid {

// Block slots hold entry offsets in 32 bits, so the lists end there (64 GiB).
constexpr uint64_t kMaxListEntries = (uint64_t)1 << 32;

// The cursor counts list positions of high bins in 32 bits: the fixed bins' to begin with, then
// promoted ones are added (fewer than 2^23: each has less than 1024 positions, and there are at
// most 5120 bins). It starts low enough never to wrap; such a frame does not fit anyway.
constexpr uint32_t list_cursor_start(uint32_t positions) {
	return positions < 0xff800000u ? positions : 0xff800000u;
}

// First entry of the high bin that found the cursor at `cursor`, and the entries that all lists
// before it take.
constexpr uint64_t list_entry(uint64_t low_entries, uint32_t cursor) {
	return low_entries + 16ull * cursor;
}

constexpr bool lists_fit(uint64_t low_entries, uint32_t cursor, uint32_t positions, uint64_t cap) {
	return list_entry(low_entries, cursor) + 16ull * positions <= cap;
}

// Capacity after an overflow of `cap` entries, from the cursor that the frame left; 0 if no
// capacity will do. Twice the old one, so that a scene that grows a little every frame overflows
// seldom (the frames of an asynchronous loop that overflow are lost).
constexpr uint64_t grown_list_cap(uint64_t low_entries, uint32_t cursor, uint64_t cap) {
	const uint64_t need = list_entry(low_entries, cursor);
	if(need > kMaxListEntries)
		return 0;
	const uint64_t more = cap * 2;
	return need > more ? need : more < kMaxListEntries ? more : kMaxListEntries;
}

} // namespace lucid
