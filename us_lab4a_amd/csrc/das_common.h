// DAS types and the LDS-tiled kernel template, shared by das.hip and the
// per-storage translation units (das_tile_f32.hip, das_tile_f16.hip,
// das_tile_bf16.hip) that instantiate the tiled kernel, so the three storage
// kinds compile in parallel.
#pragma once

#include "common.h"

#include <type_traits>

namespace mista {
namespace das {

constexpr float kPi = 3.14159265358979323846f;

template<int STORAGE>
__device__ __forceinline__ float2 load_sample(const void* __restrict__ t, uint64_t i)
{
	if constexpr (STORAGE == MISTA_STORAGE_F32) {
		return static_cast<const float2*>(t)[i];
	} else if constexpr (STORAGE == MISTA_STORAGE_F16) {
		return __half22float2(static_cast<const __half2*>(t)[i]);
	} else if constexpr (STORAGE == kStorageReal) {
		return make_float2(static_cast<const float*>(t)[i], 0.0f);
	} else {
		const uint32_t b = static_cast<const uint32_t*>(t)[i];
		return make_float2(__uint_as_float(b << 16), __uint_as_float(b & 0xFFFF0000u));
	}
}

// LDS entry type per storage kind.  lerp2: v0 + k (v1 - v0) per component from the
// raw words of two entries as one LDS read returns them (LdsPair), with FP32
// arithmetic: the difference rounded once, then one fused multiply-add.
template<int STORAGE> struct Entry;
template<uint32_t ESZ> struct LdsPair;
template<> struct LdsPair<8> { using T = float4; };   // two 8-byte entries
template<> struct LdsPair<4> { using T = uint2; };    // two 4-byte entries

template<> struct Entry<MISTA_STORAGE_F32> {
	using T = float2;
	static __device__ __forceinline__ float2 lerp2(float4 e, float k)
	{
		return make_float2(fmaf(k, e.z - e.x, e.x), fmaf(k, e.w - e.y, e.y));
	}
};
template<> struct Entry<MISTA_STORAGE_F16> {
	using T = __half2;
	static __device__ __forceinline__ float2 lerp2(uint2 e, float k)
	{
		// v1 - v0 straight from the FP16 halves: the mixed-precision FMA
		// widens both exactly and rounds 1 * v1 - v0 once to FP32, as the
		// widen-then-subtract form does, in one instruction
		float dx, dy;
		asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,1]" : "=v"(dx) : "v"(e.y), "v"(e.x));
		asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,1] op_sel_hi:[1,0,1]" : "=v"(dy) : "v"(e.y), "v"(e.x));
		const float2 v0 = __half22float2(__builtin_bit_cast(__half2, e.x));
		return make_float2(fmaf(k, dx, v0.x), fmaf(k, dy, v0.y));
	}
};
template<> struct Entry<MISTA_STORAGE_BF16> {
	using T = uint32_t;
	static __device__ __forceinline__ float2 get(T b)
	{
		return make_float2(__uint_as_float(b << 16), __uint_as_float(b & 0xFFFF0000u));
	}
	static __device__ __forceinline__ float2 lerp2(uint2 e, float k)
	{
		const float2 v0 = get(e.x), v1 = get(e.y);
		return make_float2(fmaf(k, v1.x - v0.x, v0.x), fmaf(k, v1.y - v0.y, v0.y));
	}
};
template<> struct Entry<kStorageReal> {
	using T = float;
	static __device__ __forceinline__ float2 lerp2(uint2 e, float k)
	{
		const float v0 = __uint_as_float(e.x), v1 = __uint_as_float(e.y);
		return make_float2(fmaf(k, v1 - v0, v0), 0.0f);
	}
};

// Receive elements whose sums one workgroup forms together, and the group
// that the weights and window words are laid out by: [rx group][tx][kRxGroup].
constexpr uint32_t kRxGroup = 4;

struct DasArgs {
	const void* tensor;   // [ntx][nrx][L] complex, storage type
	const float* delay;   // [num_elements][npix]
	const float* w;       // [rx groups][ntx][kRxGroup]
	float* value;         // [npix]
	float* factor;        // [npix] or null
	float2* partial;      // per-rx sums: [nrx][npix] (rx-parallel form) or [tiles][nrx][tile points]
	uint64_t npix;
	uint32_t first_tx, ntx, nrx, L;
	float offset;
	float cf_factor;      // PCF: gamma / sigma0; SCF: p
	float inv_num;        // 1 / (Ntx * Nrx)
	int signed_value;     // RF samples: value = sum / (Ntx * Nrx), not |sum|
	__device__ __forceinline__ float weight(uint32_t r, uint32_t t) const
	{
		return w[(static_cast<uint64_t>(r / kRxGroup) * ntx + t) * kRxGroup + r % kRxGroup];
	}
};

// Shifted single-pass moments for the two-pass population sigma of
// Statistics.h:34-58 (shift = first value, accumulated in double).
struct Moments {
	double k = 0.0, s1 = 0.0, s2 = 0.0;
	__device__ void add(float x, bool first)
	{
		if (first) k = x;
		const double d = static_cast<double>(x) - k;
		s1 += d;
		s2 = fma(d, d, s2);
	}
	__device__ float sigma(uint32_t n) const
	{
		const double v = (s2 - s1 * s1 / n) / n;
		return static_cast<float>(sqrt(v > 0.0 ? v : 0.0));
	}
};

// Per-rx statistics and the final value/factor of one pixel.
template<int CF>
struct PixelStats {
	float sr = 0.0f, si = 0.0f;
	Moments m0, m1;
	int sign_sum = 0;
	__device__ __forceinline__ void add_rx(float ar, float ai, bool first)
	{
		sr += ar;
		si += ai;
		if constexpr (CF == MISTA_CF_PCF) {
			// PhaseCoherenceFactor::calculate, CoherenceFactor.h:270-288
			const float phi = atan2f(ai, ar);
			const float aux = phi + ((phi < 0.0f) ? kPi : -kPi);
			m0.add(phi, first);
			m1.add(aux, first);
		} else if constexpr (CF == MISTA_CF_SCF) {
			// SignCoherenceFactor::calculate, CoherenceFactor.h:198-215
			sign_sum += (ar >= 0.0f) ? 1 : -1;
		}
	}
	// Multiply-adds are written out (fmaf) wherever the compiler could
	// otherwise contract differently in the gather and the tiled kernel.
	__device__ __forceinline__ void write(const DasArgs& a, uint64_t p) const
	{
		a.value[p] = magnitude(a, sr, si);
		if (!a.factor) return;
		float f = 1.0f;
		if constexpr (CF == MISTA_CF_PCF) {
			const float sf = fminf(m0.sigma(a.nrx), m1.sigma(a.nrx));
			f = fmaxf(0.0f, fmaf(-a.cf_factor, sf, 1.0f));
		} else if constexpr (CF == MISTA_CF_SCF) {
			const float k = static_cast<float>(sign_sum) / static_cast<float>(a.nrx);
			const float mm = 1.0f - sqrtf(fmaf(-k, k, 1.0f));
			f = powf(fabsf(mm), a.cf_factor);
		}
		a.factor[p] = f;
	}
	// value = |sum| / (Ntx * Nrx), or the signed sum for real samples
	static __device__ __forceinline__ float magnitude(const DasArgs& a, float re, float im)
	{
		return a.signed_value ? re * a.inv_num : sqrtf(fmaf(re, re, im * im)) * a.inv_num;
	}
};

// Tile geometry: a tw1 (x) by tw2 (y) by tzh (z) block of grid points, one
// point per lane.  A plane has ny = tw2 = 1; a volume is laid out as
// n1 = nx * ny columns (y fastest) by n2 = nz rows.  Each wave takes a compact
// block of points, x fastest: 8 x 8 of a plane tile, 4 x 4 x 4 of a volume tile
// (every tile is whole blocks).  An LDS read of two 8-byte entries takes 16
// lanes a clock over 32 banks (4-byte entries: 32 lanes), and of the blocks
// measured these collide least: a plane's 16 lanes 8 x 2 wait 10.4 clocks a
// read, 4 x 4 11.3, 16 x 1 12.5, 1 x 16 14.4; a volume's 4 x 4 x 1 3.9, 8 x 2
// 5.9, 16 x 1 5.9 to 9.4 (1024 x 64 volume, DAS 17.6 -> 15.6 ms against
// lanes of 16 x 4 x 1, with 1024-point tiles).  Tiles are numbered depth-band major (all
// tiles of a band of tzh rows are consecutive), so the workgroups resident
// at one time cover a depth band and share signal windows through L2/MALL.
struct TileGeom {
	uint32_t n1, n2, ny, nx;
	uint32_t tw1, tw2, tzh;
	uint32_t tiles_x, tiles_y, tiles_z;
	__device__ __forceinline__ void pixel(uint32_t tile, uint32_t lane_id, uint32_t& col, uint32_t& row, bool& valid) const
	{
		const uint32_t per_band = tiles_x * tiles_y;
		const uint32_t tz = tile / per_band, rem = tile % per_band;
		const uint32_t tx = rem / tiles_y, ty = rem % tiles_y;
		uint32_t lx, ly, lz;
		const uint32_t blk = lane_id / 64, l = lane_id % 64;
		if (tw2 == 1) {
			const uint32_t bx = tw1 / 8;
			lx = (blk % bx) * 8 + l % 8;
			lz = (blk / bx) * 8 + l / 8;
			ly = 0;
		} else {
			const uint32_t bx = tw1 / 4, by = tw2 / 4;
			lx = (blk % bx) * 4 + l % 4;
			ly = (blk / bx % by) * 4 + l / 4 % 4;
			lz = (blk / (bx * by)) * 4 + l / 16;
		}
		const uint32_t ix = tx * tw1 + lx, iy = ty * tw2 + ly, iz = tz * tzh + lz;
		valid = ix < nx && iy < ny && iz < n2;
		// lanes outside the grid shadow an in-tile point
		col = min(ix, nx - 1) * ny + min(iy, ny - 1);
		row = min(iz, n2 - 1);
	}
};

// Window word per (tile, rx, tx):
//   bits 0..23   ws * ESZ: byte offset in the channel of the first staged
//                entry (ws = floor of the tile's lowest position for the pair)
//   bits 24..30  1 KiB slots to copy (0: nothing to stage)
//   bit  31      record-end flag: some lane may have pos < 0 or i + 1 >= L,
//                or the pair has nothing to stage (padded transmit or receive
//                element, window past the record end)
// The lowest and highest positions use the same float expression order as
// the lanes', (offset + d_tx) + d_rx, so by monotonic rounding every lane's
// floor(pos) lies in [ws, floor(hi)], and floor(pos) + 1 in the staged
// slots.  The channel itself (t * nrx + r) is not stored: the kernel forms
// its 64-bit address, so tensors of any size are tiled.
constexpr uint32_t kEdgeBit = 1u << 31;
constexpr uint32_t kWsMask = (1u << 24) - 1u;
constexpr uint32_t kSlotShift = 24;
// Records below this: every ws * ESZ fits the word.  (Prepared records end at 2^20
// samples; longer ones, uploaded, take the record or the gather form.)
constexpr uint32_t kMaxWindowL = 1u << 21;

// Read-only tables (window words, weights) through the constant address
// space: uniform indices then become scalar loads.
typedef __attribute__((address_space(4))) const uint32_t* cu32_t;
typedef __attribute__((address_space(4))) const float* cf32_t;

// One frame's per-rx sums, or those of a run of its tiles (every per-tile
// pointer starts at the run's first tile).
struct TileArgs {
	const void* tensor;       // [ntx][nrx][L] complex, storage type
	const float* td;          // [tiles][nrx + ntx][tile points]: rx delays, then offset + tx delays, in lane order
	const uint32_t* words;    // [tiles][rx groups][ntx][kRxGroup]
	const uint32_t* slots;    // [tiles] 1 KiB slots of the tile's longest window
	const float* w;           // [rx groups][ntx][kRxGroup]
	float2* partial;          // [tiles][nrx][tile points]
	uint32_t ntx, nrx, L;
	uint32_t ntiles, ngrp, ngrp4;   // tiles; workgroups per tile; groups of kRxGroup receive elements
	uint32_t lds, nbmax;      // LDS bytes of the ring; most chunk buffers in it (2..4)
};

// The tiles of up to kMaxBatch frames (possibly of different shapes) in one
// launch: frame j's items are global items first[j] .. first[j+1]-1.  Every
// frame shares the kernel instantiation (storage, tile points, chunk size)
// and the LDS ring's size.
constexpr uint32_t kMaxBatch = 16;
struct TileBatch {
	TileArgs jobs[kMaxBatch];
	uint32_t first[kMaxBatch + 1];
	uint32_t njobs, total;
};

// Zeroed bytes after the analytic tensor: a window is staged as whole 1 KiB
// slots from its first entry, so the last channel's copies may read up to
// (slots per window) KiB past its end; the launcher keeps windows below this.
constexpr uint32_t kMaxSlots = 64;

// Direct global -> LDS copies (LDS DMA).  Each lane moves 16 (4) bytes from
// its own address to lds + 16 (4) * lane; lds must be wave-uniform.  Written
// as asm so that the compiler does not treat the asynchronous LDS write as
// aliasing every later LDS read (it would wait for all copies in flight);
// the kernel waits for them itself with s_waitcnt vmcnt.
// m0 is declared clobbered (it is reserved, hence the silenced warning); the
// kernels using these never rely on m0 themselves.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// The first n of four consecutive 1 KiB slots: global base + voff + k KiB -> LDS
// lds + k KiB, the wave-uniform base in scalar registers, voff = 16 * lane.
// The instruction offset of global_load_lds moves both the global and the
// LDS address (measured on gfx950: offset:1024 with m0 = B lands the source
// bytes [1024, 2048) at LDS B + 1024), so one m0 serves four slots.  One asm
// block: as C++ the cases come out as a ladder of flag registers and branches.
__device__ __forceinline__ void lds_dma16_slots(const void* base, uint32_t voff, uint32_t lds, uint32_t n)
{
	asm volatile(
			"s_mov_b32 m0, %0\n\t"
			"s_cmp_lt_u32 %3, 1\n\t"
			"s_cbranch_scc1 .Ldma_%=\n\t"
			"global_load_lds_dwordx4 %1, %2\n\t"
			"s_cmp_lt_u32 %3, 2\n\t"
			"s_cbranch_scc1 .Ldma_%=\n\t"
			"global_load_lds_dwordx4 %1, %2 offset:1024\n\t"
			"s_cmp_lt_u32 %3, 3\n\t"
			"s_cbranch_scc1 .Ldma_%=\n\t"
			"global_load_lds_dwordx4 %1, %2 offset:2048\n\t"
			"s_cmp_lt_u32 %3, 4\n\t"
			"s_cbranch_scc1 .Ldma_%=\n\t"
			"global_load_lds_dwordx4 %1, %2 offset:3072\n"
			".Ldma_%=:"
			:: "s"(lds), "v"(voff), "s"(base), "s"(n) : "memory", "m0", "scc");
}
// One slot.  The s_nop is the wait state that a load with LDS destination needs
// after a scalar write of M0: the compiler puts it in for its own instructions,
// but does not look inside asm (above, the compare and the branch are it).
__device__ __forceinline__ void lds_dma16_slot(const void* base, uint32_t voff, uint32_t lds)
{
	asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
			:: "s"(lds), "v"(voff), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop

// Wait until at most n (wave-uniform) vector memory operations of this wave
// are outstanding, rounding n down to a power of two: waits at least as long
// as s_waitcnt vmcnt(n), with 7 immediates instead of 64.  The expcnt and
// lgkmcnt fields stay at their maxima (no wait on them).
#define MISTA_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (7 << 4) | (15 << 8) | (((n) >> 4) << 14))
// Written as one asm block of compares and branches: as C++ the if-chain
// comes out restructured into flag registers and several branch blocks that
// every chunk walks through (about 15 scalar instructions for n = 0 instead of
// 3).  Small counts first: with two ring buffers (the common case) n is 0.
__device__ __forceinline__ void wait_vmcnt_at_most(uint32_t n)
{
	asm volatile(
			"s_cmp_lt_u32 %0, 1\n\t"
			"s_cbranch_scc0 .Lvw1_%=\n\t"
			"s_waitcnt vmcnt(0)\n\t"
			"s_branch .Lvwe_%=\n"
			".Lvw1_%=:\n\t"
			"s_cmp_lt_u32 %0, 2\n\t"
			"s_cbranch_scc0 .Lvw2_%=\n\t"
			"s_waitcnt vmcnt(1)\n\t"
			"s_branch .Lvwe_%=\n"
			".Lvw2_%=:\n\t"
			"s_cmp_lt_u32 %0, 4\n\t"
			"s_cbranch_scc0 .Lvw4_%=\n\t"
			"s_waitcnt vmcnt(2)\n\t"
			"s_branch .Lvwe_%=\n"
			".Lvw4_%=:\n\t"
			"s_cmp_lt_u32 %0, 8\n\t"
			"s_cbranch_scc0 .Lvw8_%=\n\t"
			"s_waitcnt vmcnt(4)\n\t"
			"s_branch .Lvwe_%=\n"
			".Lvw8_%=:\n\t"
			"s_cmp_lt_u32 %0, 16\n\t"
			"s_cbranch_scc0 .Lvw16_%=\n\t"
			"s_waitcnt vmcnt(8)\n\t"
			"s_branch .Lvwe_%=\n"
			".Lvw16_%=:\n\t"
			"s_cmp_lt_u32 %0, 32\n\t"
			"s_cbranch_scc0 .Lvw32_%=\n\t"
			"s_waitcnt vmcnt(16)\n\t"
			"s_branch .Lvwe_%=\n"
			".Lvw32_%=:\n\t"
			"s_waitcnt vmcnt(32)\n"
			".Lvwe_%=:"
			:
			: "s"(n)
			: "scc", "memory");
}

// Two consecutive LDS entries as one value of LdsPair's type (4-byte
// entries as their raw words).
__device__ __forceinline__ float4 pack_pair(uint64_t a, uint64_t b)
{
	const float2 u = __builtin_bit_cast(float2, a), v = __builtin_bit_cast(float2, b);
	return make_float4(u.x, u.y, v.x, v.y);
}
__device__ __forceinline__ uint2 pack_pair(uint32_t a, uint32_t b) { return make_uint2(a, b); }

// N LDS reads of two consecutive entries each (byte addresses addr; one
// ds_read2 per pair), written as plain loads and all issued before the
// first result is used: the compiler's wait insertion then waits for read
// q just before its use (lgkmcnt(N-1-q), the reads complete in order), so
// the first pairs' accumulation overlaps the later reads' latency.
template<uint32_t ESZ, int N>
__device__ __forceinline__ void lds_read_pairs(const uint32_t* addr, typename LdsPair<ESZ>::T* out)
{
	using W = typename std::conditional<ESZ == 8, uint64_t, uint32_t>::type;
	typedef __attribute__((address_space(3))) const W* lds_entry_t;
#pragma unroll
	for (int q = 0; q < N; ++q) {
		const lds_entry_t lp = (lds_entry_t)(size_t)addr[q];
		out[q] = pack_pair(lp[0], lp[1]);
	}
}

constexpr uint32_t kTileZeroBytes = 128;

// Chunk buffers of the ring for a tile whose longest window has S slots: as many
// as fit with their buffers of transmit delays (0: not even two).
__host__ __device__ inline uint32_t tile_buffers(uint32_t nbmax, uint32_t lds, uint32_t S, uint32_t rc, uint32_t h, uint32_t npts)
{
	uint32_t nb = nbmax < 4u ? nbmax : 4u;
	while (nb >= 2u && kTileZeroBytes + nb * rc * S * 1024u + (1u + (nb - 1u) / h) * npts * 4u > lds) --nb;
	return nb >= 2u ? nb : 0u;
}

// Per-rx sums of one tile: a workgroup of NT lanes, P points a lane (point k
// of lane l is tile point k * NT + l), forms the sums of RC * H receive
// elements over all transmits.  A chunk = RC receive elements of one transmit:
// RC signal windows, each copied HBM -> LDS with direct loads (only as many
// 1 KiB slots as the pair needs).  Chunk i = transmit i / H, receive elements
// RC * (i % H) ..; a transmit's delays of the tile's points are copied the same
// way, once for its H chunks, with the last chunk of the transmit before, and
// read during that chunk.  Chunks stream through a ring of 2..4 LDS buffers
// (as many as the tile's longest window leaves room for); chunk i + NB - 1 is
// copied while chunk i is computed.
template<int STORAGE, int NT, int P, int RC, int H>
__device__ __forceinline__ void das_tile(const TileArgs& A, const uint32_t tile, const uint32_t grp, unsigned char* smem)
{
	using E = typename Entry<STORAGE>::T;
	constexpr uint32_t ESZ = sizeof(E);
	constexpr uint32_t NW = NT / 64;
	constexpr uint32_t NPTS = NT * P;
	constexpr uint32_t R = RC * H;             // receive elements of the workgroup
	constexpr uint32_t WPW = NW / RC;          // waves that share a window's copy
	constexpr uint32_t DSLOTS = NPTS / 256;    // slots of a transmit's delays
	static_assert(NW % RC == 0 && (RC == 4 || R == 4), "whole waves per window; words of a chunk consecutive");

	const uint32_t tid = threadIdx.x, lane = tid % 64;
	const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / 64);
	const uint32_t nrx = A.nrx, L = A.L, ntx = A.ntx;
	const uint32_t nchunks = ntx * H;
	const float lim = static_cast<float>(L - 1u);
	const uint32_t S = *(cu32_t)(A.slots + tile);
	const uint32_t win = S * 1024u;
	const uint32_t buf_bytes = RC * win;
	const uint32_t NB = tile_buffers(A.nbmax, A.lds, S, RC, H, NPTS);
	const uint32_t ring = NB * buf_bytes;
	const uint32_t ND = 1 + (NB - 1) / H;      // buffers of transmit delays, after the ring
	const uint64_t chan_bytes = static_cast<uint64_t>(L) * ESZ;
	const uint64_t tx_bytes = chan_bytes * nrx;
	const uint32_t rows = nrx + ntx;
	const float* td = A.td + static_cast<uint64_t>(tile) * rows * NPTS;
	// words and weights [groups of kRxGroup][ntx][kRxGroup]: chunk (t, h) at
	// t * kRxGroup + h * hstride
	const uint32_t hstride = RC == kRxGroup ? ntx * kRxGroup : static_cast<uint32_t>(RC);
	const uint32_t g4 = grp * (R / kRxGroup);
	const cu32_t wtab = (cu32_t)(A.words + (static_cast<uint64_t>(tile) * A.ngrp4 + g4) * ntx * kRxGroup);
	const cf32_t weights = (cf32_t)(A.w + static_cast<uint64_t>(g4) * ntx * kRxGroup);
	const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<size_t>((__attribute__((address_space(3))) void*)smem));
	const uint32_t voff = lane * 16;
	// The first bytes stay zero: the entries of lanes outside the record.
	const uint32_t lds_ring = lds0 + kTileZeroBytes;
	if (tid < kTileZeroBytes / 4) reinterpret_cast<uint32_t*>(smem)[tid] = 0u;   // seen after the first chunk's barrier

	// rx delays of this lane's points (receive elements past the last shadow it)
	float drx[R][P];
#pragma unroll
	for (uint32_t q = 0; q < R; ++q)
#pragma unroll
		for (int k = 0; k < P; ++k)
			drx[q][k] = td[static_cast<uint64_t>(min(grp * R + q, nrx - 1)) * NPTS + k * NT + tid];
	// Fence: waited for here, before the first copy.  Left to their first use
	// in the chunk loop, the compiler waits there, in every chunk, for all
	// copies in flight (it does not see the copies).
#pragma unroll
	for (uint32_t q = 0; q < R; ++q)
#pragma unroll
		for (int k = 0; k < P; ++k) asm volatile("" : "+v"(drx[q][k]));

	// Copy cursor: chunk is_t, is_h; its ring buffer and its delays' buffer; the
	// channel of this wave's window.  WPW waves share a window: this one copies
	// the sub-th part of window wj.
	const uint32_t wj = wave / WPW, sub = wave % WPW;
	uint32_t is_t = 0, is_h = 0, is_buf = 0, is_d = 0;
	const unsigned char* is_base = static_cast<const unsigned char*>(A.tensor) + (static_cast<uint64_t>(grp) * R + wj) * chan_bytes;
	const unsigned char* is_src = is_base;   // its channel of chunk is_h
	uint32_t iw = 0;
	// (32-bit byte offsets: scalar loads take them as they are)
	typedef __attribute__((address_space(4))) const char* cbyte_t;
	auto load_issue_word = [&]() { iw = *(cu32_t)((cbyte_t)wtab + (is_t * kRxGroup + is_h * hstride + wj) * 4u); };
	auto issue_delays = [&](uint32_t t) -> uint32_t {   // transmit t's, a slot a wave
		uint32_t count = 0;
#pragma unroll
		for (uint32_t d0 = 0; d0 < DSLOTS; d0 += NW) {
			const uint32_t d = d0 + (NW - 1 - wave);
			if (d0 + NW <= DSLOTS || d < DSLOTS) {
				lds_dma16_slot(td + static_cast<uint64_t>(nrx + t) * NPTS + d * 256u, voff,
						lds_ring + ring + (is_d * DSLOTS + d) * 1024u);
				++count;
			}
		}
		if (++is_d == ND) is_d = 0;
		return count;
	};
	// copies of the cursor's chunk; returns how many copy instructions this wave issued
	auto issue = [&]() -> uint32_t {
		const uint32_t n = (iw >> kSlotShift) & 127u;
		uint32_t count = 0;
		if (sub * 4 < n) {
			const unsigned char* src = is_src + ((iw & kWsMask) + sub * 4096u);
			uint32_t dst = lds_ring + is_buf + wj * win + sub * 4096u;
			for (uint32_t s0 = sub * 4; s0 < n; s0 += 4 * WPW, src += 4096 * WPW, dst += 4096 * WPW) {
				lds_dma16_slots(src, voff, dst, n - s0);
				count += min(n - s0, 4u);
			}
		}
		is_buf += buf_bytes;
		if (is_buf == ring) is_buf = 0;
		is_src += RC * chan_bytes;
		if (++is_h == H) {
			is_h = 0;
			++is_t;
			is_base += tx_bytes;
			is_src = is_base;
			if (is_t < ntx) count += issue_delays(is_t);
		}
		return count;
	};
	(void)issue_delays(0);
	uint32_t c1 = 0, c2 = 0;   // copies of the last chunk issued, of the one before
	for (uint32_t k = 0; k < NB - 1 && k < nchunks; ++k) {
		load_issue_word();
		c2 = c1;
		c1 = issue();
	}
	if (is_t < ntx) load_issue_word();
	// window words and weights of the chunk to compute, one chunk ahead
	uint32_t cw[RC];
	float cwt[RC];
	auto load_chunk = [&](uint32_t off) {
#pragma unroll
		for (uint32_t j = 0; j < RC; ++j) {
			cw[j] = ((cu32_t)((cbyte_t)wtab + off * 4u))[j];
			cwt[j] = ((cf32_t)((cbyte_t)weights + off * 4u))[j];
		}
	};
	load_chunk(0);

	float ar[R][P], ai[R][P];
#pragma unroll
	for (uint32_t q = 0; q < R; ++q)
#pragma unroll
		for (int k = 0; k < P; ++k) ar[q][k] = ai[q][k] = 0.0f;
	typedef __attribute__((address_space(3))) const float* lds_float_t;
	float dt[P], dnext[P];   // this transmit's delays, the next one's
	uint32_t rd_d = 0;       // buffer of the next delays to read
	auto read_delays = [&]() {
		const lds_float_t dl = (lds_float_t)(size_t)(lds_ring + ring + rd_d * (DSLOTS * 1024u) + tid * 4u);
#pragma unroll
		for (int k = 0; k < P; ++k) dnext[k] = dl[k * NT];
		if (++rd_d == ND) rd_d = 0;
	};

	// the first transmit's delays: waited for with everything issued so far
	MISTA_VMCNT(0);
	__syncthreads();
	read_delays();
	uint32_t bbase = 0;   // ring offset of the buffer of the chunk being computed
	for (uint32_t t = 0; t < ntx; ++t) {
#pragma unroll
		for (int h = 0; h < H; ++h) {
			uint32_t w_[RC];
			float wt[RC];
#pragma unroll
			for (uint32_t j = 0; j < RC; ++j) {
				w_[j] = cw[j];
				wt[j] = cwt[j];
			}
			// copies issued after this chunk: those of the NB - 2 chunks that follow
			wait_vmcnt_at_most((NB > 2 ? c1 : 0u) + (NB > 3 ? c2 : 0u));
			__syncthreads();
			c2 = c1;
			c1 = is_t < ntx ? issue() : 0u;
			if (h == 0) {
#pragma unroll
				for (int k = 0; k < P; ++k) dt[k] = dnext[k];
			}
			// Register fence: this chunk's positions are computed here, not
			// ahead of the barrier for all H chunks.
#pragma unroll
			for (int k = 0; k < P; ++k) asm volatile("" : "+v"(dt[k]));
			uint32_t any_edge = 0;
#pragma unroll
			for (uint32_t j = 0; j < RC; ++j) any_edge |= w_[j];
			const uint32_t lb = lds_ring + bbase;
			// Positions and LDS addresses.  A chunk in which some lane may lie
			// outside 0 <= pos < L - 1 (or with nothing staged for a pair)
			// sends those lanes to the zero entries: they add zero.  The range
			// test is one unsigned compare of the bit patterns: positions are
			// never -0, and negative values and NaN compare above L - 1's.
			constexpr int N = RC * P;
			uint32_t addr[N];
			float kf[N];
#pragma unroll
			for (uint32_t j = 0; j < RC; ++j) {
				const uint32_t base = lb + j * win - (w_[j] & kWsMask);
#pragma unroll
				for (int k = 0; k < P; ++k) {
					const float pos = dt[k] + drx[h * RC + j][k];
					kf[j * P + k] = __builtin_amdgcn_fractf(pos);
					addr[j * P + k] = static_cast<uint32_t>(pos) * ESZ + base;
				}
			}
			if (any_edge & kEdgeBit) {
#pragma unroll
				for (uint32_t j = 0; j < RC; ++j) {
					const uint32_t limj = (w_[j] >> kSlotShift) & 127u ? __float_as_uint(lim) : 0u;
#pragma unroll
					for (int k = 0; k < P; ++k) {
						const float pos = dt[k] + drx[h * RC + j][k];
						if (!(__float_as_uint(pos) < limj)) addr[j * P + k] = lds0;
					}
				}
			}
			typename LdsPair<ESZ>::T v[N];
			lds_read_pairs<ESZ, N>(addr, v);
			if (h == H - 1) read_delays();
#pragma unroll
			for (uint32_t j = 0; j < RC; ++j)
#pragma unroll
				for (int k = 0; k < P; ++k) {
					const uint32_t q = h * RC + j;
					const float2 s = Entry<STORAGE>::lerp2(v[j * P + k], kf[j * P + k]);
					ar[q][k] = fmaf(s.x, wt[j], ar[q][k]);
					if constexpr (STORAGE != kStorageReal) ai[q][k] = fmaf(s.y, wt[j], ai[q][k]);
				}
			// ... and its sums are finished before the next chunk
#pragma unroll
			for (uint32_t q = h * RC; q < (h + 1) * RC; ++q)
#pragma unroll
				for (int k = 0; k < P; ++k) asm volatile("" : "+v"(ar[q][k]), "+v"(ai[q][k]));
			// the next chunks' scalars, after this chunk's LDS reads (a scalar
			// load in flight would hold up their wait): in flight during the
			// next barrier
			if (is_t < ntx) load_issue_word();
			if (h + 1 < H) load_chunk(t * kRxGroup + (h + 1) * hstride);
			else if (t + 1 < ntx) load_chunk((t + 1) * kRxGroup);
			bbase += buf_bytes;
			if (bbase == ring) bbase = 0;
		}
	}
	float2* out = A.partial + (static_cast<uint64_t>(tile) * nrx + grp * R) * NPTS + tid;
#pragma unroll
	for (uint32_t q = 0; q < R; ++q)
		if (grp * R + q < nrx)
#pragma unroll
			for (int k = 0; k < P; ++k) out[static_cast<uint64_t>(q) * NPTS + k * NT] = make_float2(ar[q][k], ai[q][k]);
}

// Item (tile, rx group) of a launch of n items, XCD-aware: workgroups are
// dealt round-robin to the 8 XCDs (block b runs on XCD b % 8), so XCD x gets
// one contiguous run of the items.
__device__ __forceinline__ uint32_t xcd_item()
{
	const uint32_t T = gridDim.x, q8 = T / 8, rm8 = T % 8, xcd = blockIdx.x % 8;
	return xcd * q8 + min(xcd, rm8) + blockIdx.x / 8;
}

// One frame: its arguments arrive as the kernel's own, which the compiler
// keeps in scalar registers.
template<int STORAGE, int NT, int P, int RC, int H>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 8)))
das_tile_kernel(const TileArgs A)
{
	extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
	const uint32_t item = xcd_item();
	das_tile<STORAGE, NT, P, RC, H>(A, item % A.ntiles, item / A.ntiles, smem);
}

// A batch of frames in one launch, their items concatenated: the hardware
// dispatcher starts each workgroup as a CU frees up, so frames of uneven cost
// balance by themselves.  (A separate kernel: a frame's arguments picked from
// the table by a run-time index are reloaded from memory at their uses.)
template<int STORAGE, int NT, int P, int RC, int H>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 8)))
das_tile_batch_kernel(const TileBatch B)
{
	extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
	const uint32_t g = xcd_item();
	uint32_t j = 0;
	while (j + 1 < B.njobs && B.first[j + 1] <= g) ++j;
	const uint32_t item = g - B.first[j];
	das_tile<STORAGE, NT, P, RC, H>(B.jobs[j], item % B.jobs[j].ntiles, item / B.jobs[j].ntiles, smem);
}

template<int STORAGE, int NT, int P, int RC, int H>
void launch_tile_t(const TileBatch& B, hipStream_t s)
{
	const TileArgs& A = B.jobs[0];   // the ring's size is shared by the batch
	auto go = [&](auto kern, const auto& args) {
		HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
				static_cast<int>(A.lds)));
		hipLaunchKernelGGL(kern, dim3(B.total), dim3(NT), A.lds, s, args);
	};
	if (B.njobs == 1) go(das_tile_kernel<STORAGE, NT, P, RC, H>, A);
	else go(das_tile_batch_kernel<STORAGE, NT, P, RC, H>, B);
}

// Tiled launch for one storage kind (instantiated in das_tile_<storage>.hip).
template<int STORAGE>
void launch_tile_storage(const TileBatch& B, uint32_t npts, uint32_t r, uint32_t rc, uint32_t nt, hipStream_t s)
{
	if (npts == 256) launch_tile_t<STORAGE, 256, 1, 4, 1>(B, s);
	else if (npts == 512 && r == 16) launch_tile_t<STORAGE, 512, 1, 4, 4>(B, s);
	else if (npts == 512 && r == 8) launch_tile_t<STORAGE, 256, 2, 4, 2>(B, s);
	else if (npts == 512) launch_tile_t<STORAGE, 256, 2, 4, 1>(B, s);
	else if (npts == 1024 && r == 8) launch_tile_t<STORAGE, 512, 2, 4, 2>(B, s);
	else if (npts == 1024) launch_tile_t<STORAGE, 512, 2, 4, 1>(B, s);
	else if (nt == 512) launch_tile_t<STORAGE, 512, 4, 2, 2>(B, s);
	else if (rc == 2) launch_tile_t<STORAGE, 1024, 2, 2, 2>(B, s);
	else if (r == 8) launch_tile_t<STORAGE, 1024, 2, 4, 2>(B, s);
	else launch_tile_t<STORAGE, 1024, 2, 4, 1>(B, s);
}

}  // namespace das
}  // namespace mista
