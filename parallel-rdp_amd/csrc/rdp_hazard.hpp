// Host-side bounds of what a pass's raster can write, what a TMEM upload can read
// and what a clear overwrites whole, as RDRAM byte ranges.  They decide whether a
// round's TMEM replay may run before the rasters of earlier rounds, and with
// host-coherent RDRAM which of the caller's pages a submission copies in.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <vector>

#include "rdp_frontend.hpp"
#include "rdp_types.hpp"

namespace rdp_mi {

// RDRAM byte range [lo, hi) before the wrap at the RDRAM size.
struct ByteRange {
	uint64_t lo, hi;
};

// Every RDRAM byte the raster stage of a pass can write: colour image and
// depth image rows 0 .. fb_height-1 of fb_width pixels, word aligned.
inline void pass_write_ranges(const HostPass &hp, std::vector<ByteRange> &out)
{
	if (hp.prims.empty()) return;
	const uint64_t px = (uint64_t)hp.fb_width * hp.fb_height;
	uint64_t base, bytes;
	switch (hp.fb_fmt) {
	case FB_I4:
	case FB_I8: base = hp.fb_addr; bytes = px; break;
	case FB_RGBA5551:
	case FB_IA88: base = hp.fb_addr & ~1u; bytes = 2 * px; break;
	default: base = hp.fb_addr & ~3u; bytes = 4 * px; break;
	}
	out.push_back({ base & ~3ull, (base + bytes + 3) & ~3ull });
	if (hp.depth_addr != hp.fb_addr) {
		const uint64_t d = hp.depth_addr & ~1u;
		out.push_back({ d & ~3ull, (d + 2 * px + 3) & ~3ull });
	}
}

// A bound on the RDRAM bytes a TMEM upload reads: rows 0 .. height-1 of the
// source image (vram_width texels apart, at most 4 bytes each) and, for
// TLUT loads, vram_effective_width entries from vram_addr.  False when the
// record does not allow a bound.
inline bool upload_read_range(const UploadInfo &u, ByteRange &r)
{
	if (u.vram_addr < 0 || u.width < 0 || u.height < 0 || u.vram_width < 0 || u.vram_effective_width < 0) return false;
	const uint64_t w = (uint64_t)std::max(std::max(u.vram_width, u.width), u.vram_effective_width);
	r.lo = (uint64_t)u.vram_addr & ~3ull;
	r.hi = (uint64_t)u.vram_addr + (((uint64_t)u.height + 1) * w + w + 16) * 4 + 64;
	return true;
}

// Rows [y0, y1) of a pass's colour image that its first primitive overwrites
// whole, whatever they held: a FILL rectangle across the full width (fill
// coverage is start_x .. end_x inclusive, rasterizer.comp; a row counts when its
// first sub-scanline is inside the rectangle and the scissor).  Empty unless the
// image is 16 or 32 bits, apart from the depth image (or the same 16-bit one), and
// not interlaced.
inline void cleared_rows(const HostPass &hp, uint32_t &y0, uint32_t &y1)
{
	y0 = y1 = 0;
	if (hp.prims.empty() || hp.scale_log2) return;
	if (hp.fb_fmt != FB_RGBA5551 && hp.fb_fmt != FB_IA88 && hp.fb_fmt != FB_RGBA8888) return;
	const PrimRecord &p = hp.prims[0];
	const DrawState &st = hp.states[p.state_index];
	if (p.opcode != 0x36 || p.variant != kFillVariant || (st.raw_ras_flags & (RAS_INTERLACE_FIELD | RAS_COPY)) ||
	    !(st.raw_ras_flags & RAS_FILL))
		return;
	// A Z clear's image is often the depth image too: then one 16-bit word is
	// both, and the fill sets both.
	const uint64_t px = (uint64_t)hp.fb_width * hp.fb_height, bytes = hp.fb_fmt == FB_RGBA8888 ? 4 * px : 2 * px;
	const bool alias = hp.fb_addr == hp.depth_addr && hp.fb_fmt != FB_RGBA8888;
	if (!alias && (uint64_t)hp.fb_addr < (uint64_t)hp.depth_addr + 2 * px + 8 &&
	    (uint64_t)hp.depth_addr < (uint64_t)hp.fb_addr + bytes + 8)
		return;
	const uint32_t *w = hp.words.data() + p.word_offset;
	const uint32_t xl = (w[0] >> 12) & 0xfff, yl = (w[0] & 0xfff) | 3, xh = (w[1] >> 12) & 0xfff, yh = w[1] & 0xfff;
	const uint32_t xlo = std::max(xh, st.scissor[0]), xhi = std::min(xl, st.scissor[2]);
	if (xlo >= 4 || hp.fb_width < 2 || xhi < 4 * (hp.fb_width - 1)) return;
	const uint32_t lo = std::max(yh, st.scissor[1]), hi = std::min(yl, st.scissor[3]);
	const uint32_t a = (lo + 3) / 4, b = std::min((hi + 3) / 4, hp.fb_height);
	if (a >= b) return;
	y0 = a;
	y1 = b;
}

inline void subtract_range(std::vector<ByteRange> &from, const ByteRange &r)
{
	std::vector<ByteRange> out;
	for (const ByteRange &f : from) {
		if (f.lo < std::min(f.hi, r.lo)) out.push_back({ f.lo, std::min(f.hi, r.lo) });
		if (std::max(f.lo, r.hi) < f.hi) out.push_back({ std::max(f.lo, r.hi), f.hi });
	}
	from.swap(out);
}

// RDRAM a submission of these passes (in order) reads before it has itself
// overwritten it: colour and depth rows and the sources of TMEM uploads, without
// what an earlier clear of the submission, or the pass's own, has overwritten
// whole.  Copying in only these leaves the device's RDRAM as copying in every
// page would.
inline void submission_read_ranges(const std::vector<HostPass> &passes, uint64_t size, std::vector<ByteRange> &out)
{
	out.clear();
	std::vector<ByteRange> known;
	for (const HostPass &hp : passes) {
		std::vector<ByteRange> reads;
		for (const UploadInfo &u : hp.uploads) {
			ByteRange b;
			if (!upload_read_range(u, b)) b = { 0, size };
			reads.push_back(b);
		}
		// Uploads read RDRAM as of the start of the pass, the colour and depth
		// rows are read per tile before the first primitive.
		for (const ByteRange &k : known) subtract_range(reads, k);
		uint32_t y0, y1;
		cleared_rows(hp, y0, y1);
		ByteRange cleared{ 0, 0 };
		if (y0 < y1) {
			const uint64_t px = hp.fb_fmt == FB_RGBA8888 ? 4 : 2, base = (uint64_t)hp.fb_addr / px * px;
			const uint64_t row = px * hp.fb_width;
			// Only whole ranges inside RDRAM (no wrap).
			if (base + y1 * row <= size) cleared = { base + y0 * row, base + y1 * row };
		}
		std::vector<ByteRange> fb;
		pass_write_ranges(hp, fb);
		if (cleared.lo < cleared.hi) subtract_range(fb, cleared);
		for (const ByteRange &k : known) subtract_range(fb, k);
		reads.insert(reads.end(), fb.begin(), fb.end());
		out.insert(out.end(), reads.begin(), reads.end());
		if (cleared.lo < cleared.hi) known.push_back(cleared);
	}
}

// The same for native RDRAM when the pass may be an upscaled one: its raster
// writes the sample planes only, and with a resolve also its native region.
inline void native_write_ranges(const HostPass &hp, std::vector<ByteRange> &out)
{
	if (!hp.scale_log2) {
		pass_write_ranges(hp, out);
		return;
	}
	if (!hp.ssaa_resolve || hp.prims.empty()) return;
	const uint64_t px = (uint64_t)(hp.fb_width >> hp.scale_log2) * hp.domain_height;
	const uint32_t log2 = hp.fb_fmt == FB_RGBA8888 ? 2 : (hp.fb_fmt == FB_RGBA5551 || hp.fb_fmt == FB_IA88) ? 1 : 0;
	const uint64_t base = (hp.fb_addr >> log2) << log2;
	out.push_back({ base & ~3ull, (base + (px << log2) + 3) & ~3ull });
	if (hp.depth_addr != hp.fb_addr) {
		const uint64_t dep = hp.depth_addr & ~1u;
		out.push_back({ dep & ~3ull, (dep + 2 * px + 3) & ~3ull });
	}
}

inline bool ranges_overlap(const ByteRange &a, const ByteRange &b, uint64_t size)
{
	if (a.hi - a.lo >= size || b.hi - b.lo >= size) return true;
	ByteRange pa[2], pb[2];
	auto split = [size](const ByteRange &x, ByteRange *out) {
		const uint64_t lo = x.lo % size, hi = lo + (x.hi - x.lo);
		if (hi <= size) {
			out[0] = { lo, hi };
			return 1;
		}
		out[0] = { lo, size };
		out[1] = { 0, hi - size };
		return 2;
	};
	const int na = split(a, pa), nb = split(b, pb);
	for (int i = 0; i < na; i++)
		for (int j = 0; j < nb; j++)
			if (pa[i].lo < pb[j].hi && pb[j].lo < pa[i].hi) return true;
	return false;
}

}  // namespace rdp_mi
