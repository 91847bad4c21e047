// Delay-and-sum over the analytic tensor: apodized complex accumulation with
// fractional-sample (linear) interpolation, PCF/SCF coherence statistics and
// the fused envelope.  Semantics of VectorialSTAProcessor.h:237-338 and
// processRowColumnSTA[PCF]Kernel (VectorialSTACUDAProcessor.cu:55-186):
//   pos = (offset + d_tx) + d_rx      (samples, FP32)
//   i = trunc(pos), k = pos - i;  pos >= 0 and i + 1 < L, else skipped
//   v = s[i] + k (s[i+1] - s[i]);  sum += v * w[rx][tx]
//   value = |sum| / (Ntx * Nrx), factor = PCF / SCF of the per-rx sums
// w[rx][tx] folds rx apodization, optional tx apodization and the per-channel
// FP16/BF16 storage scale.
//
// Kernels:
//  das_gather_kernel  one pixel per lane, global gathers (reference shape;
//                     the explicit gather variant).
//  das_record_sums_kernel / das_rx_sums_kernel + das_rx_stats_kernel  the
//                     fallback where no tile fits: per (pixel, rx) the sum over
//                     the transmits, from whole records passing through LDS or,
//                     for few pixels, by gathers; then a lane per pixel folds
//                     the per-rx sums in rx order.
//  das_tile_kernel + das_tile_stats_kernel  the tiled form: a workgroup forms
//                     the per-rx sums of a tile of pixels for a few receive
//                     elements; for every (rx, tx) pair the tile's signal
//                     window is copied HBM -> LDS with direct loads
//                     (global_load_lds_dwordx4, a ring of buffers), so each
//                     sample pair costs one LDS read.  Tile delays, window
//                     starts, lengths and record-end flags come from tables
//                     built once per geometry.  Then a lane per pixel folds
//                     the sums in rx order.
#include "das_common.h"

#include <algorithm>
#include <cmath>
#include <vector>

namespace mista {

namespace das {
extern template void launch_tile_storage<MISTA_STORAGE_F32>(const TileBatch&, uint32_t, uint32_t, uint32_t, uint32_t, hipStream_t);
extern template void launch_tile_storage<MISTA_STORAGE_F16>(const TileBatch&, uint32_t, uint32_t, uint32_t, uint32_t, hipStream_t);
extern template void launch_tile_storage<MISTA_STORAGE_BF16>(const TileBatch&, uint32_t, uint32_t, uint32_t, uint32_t, hipStream_t);
extern template void launch_tile_storage<kStorageReal>(const TileBatch&, uint32_t, uint32_t, uint32_t, uint32_t, hipStream_t);
}  // namespace das

using namespace das;

namespace {

// ---------------------------------------------------------------- gather

// One pixel per lane, reference loop structure, global gathers.  CF == NONE:
// tx outer, rx inner into one accumulator (VectorialSTAProcessor.h:312-325).
// CF != NONE: rx outer, tx inner, which yields the same per-rx sums
// (VectorialSTAProcessor.h:269-284) one rx at a time.
// RX_OUTER: rx outer without a coherence factor too, the tiled kernel's order.
template<int STORAGE, int CF, bool RX_OUTER>
__global__ void __launch_bounds__(256) das_gather_kernel(const DasArgs a)
{
	const uint64_t p = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
	if (p >= a.npix) return;
	const float* dcol = a.delay + p;
	const uint32_t L = a.L;
	// pos in [0, L-1) <=> i = trunc(pos) satisfies i + 1 < L; the float
	// compare also rejects NaN and values past 2^32
	const float lim = static_cast<float>(L - 1u);
	if constexpr (CF == MISTA_CF_NONE && !RX_OUTER) {
		float sr = 0.0f, si = 0.0f;
		for (uint32_t t = 0; t < a.ntx; ++t) {
			const float txo = a.offset + dcol[static_cast<uint64_t>(a.first_tx + t) * a.npix];
			for (uint32_t r = 0; r < a.nrx; ++r) {
				const float pos = txo + dcol[static_cast<uint64_t>(r) * a.npix];
				if (pos >= 0.0f && pos < lim) {
					const uint32_t i = static_cast<uint32_t>(pos);
					const float k = pos - static_cast<float>(i);
					const uint64_t ch = (static_cast<uint64_t>(t) * a.nrx + r) * L + i;
					const float2 v0 = load_sample<STORAGE>(a.tensor, ch);
					const float2 v1 = load_sample<STORAGE>(a.tensor, ch + 1);
					const float w = a.weight(r, t);
					sr = fmaf(fmaf(k, v1.x - v0.x, v0.x), w, sr);
					si = fmaf(fmaf(k, v1.y - v0.y, v0.y), w, si);
				}
			}
		}
		a.value[p] = PixelStats<MISTA_CF_NONE>::magnitude(a, sr, si);
		if (a.factor) a.factor[p] = 1.0f;
	} else {
		PixelStats<CF> st;
		for (uint32_t r = 0; r < a.nrx; ++r) {
			const float drx = dcol[static_cast<uint64_t>(r) * a.npix];
			float ar = 0.0f, ai = 0.0f;
			for (uint32_t t = 0; t < a.ntx; ++t) {
				const float pos = (a.offset + dcol[static_cast<uint64_t>(a.first_tx + t) * a.npix]) + drx;
				if (pos >= 0.0f && pos < lim) {
					const uint32_t i = static_cast<uint32_t>(pos);
					const float k = pos - static_cast<float>(i);
					const uint64_t ch = (static_cast<uint64_t>(t) * a.nrx + r) * L + i;
					const float2 v0 = load_sample<STORAGE>(a.tensor, ch);
					const float2 v1 = load_sample<STORAGE>(a.tensor, ch + 1);
					const float w = a.weight(r, t);
					ar = fmaf(fmaf(k, v1.x - v0.x, v0.x), w, ar);
					ai = fmaf(fmaf(k, v1.y - v0.y, v0.y), w, ai);
				}
			}
			st.add_rx(ar, ai, r == 0);
		}
		st.write(a, p);
	}
}

// The per-rx sums of the tiled kernel, a lane per (pixel, rx): lanes of a
// workgroup take consecutive pixels of one rx (grid y), so the delay-table
// and partial-sum accesses are coalesced and the weights uniform.  The sum
// over the transmits is the tiled kernel's fma chain in transmit order (an
// excluded position adds nothing, where the tiled kernel adds a zero entry);
// out to partial[rx][pixel].  With far more lanes than pixels this keeps
// the GPU busy on grids too coarse for any tile (a window past 64 KiB) or too
// small to fill it one pixel per lane.
template<int STORAGE>
__global__ void __launch_bounds__(256) das_rx_sums_kernel(const DasArgs a)
{
	const uint64_t p = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
	const uint32_t r = blockIdx.y;
	if (p >= a.npix) return;
	const float* dcol = a.delay + p;
	const float lim = static_cast<float>(a.L - 1u);
	const float drx = dcol[static_cast<uint64_t>(r) * a.npix];
	float ar = 0.0f, ai = 0.0f;
	for (uint32_t t = 0; t < a.ntx; ++t) {
		const float pos = (a.offset + dcol[static_cast<uint64_t>(a.first_tx + t) * a.npix]) + drx;
		if (pos >= 0.0f && pos < lim) {
			const uint32_t i = static_cast<uint32_t>(pos);
			const float k = pos - static_cast<float>(i);
			const uint64_t ch = (static_cast<uint64_t>(t) * a.nrx + r) * a.L + i;
			const float2 v0 = load_sample<STORAGE>(a.tensor, ch);
			const float2 v1 = load_sample<STORAGE>(a.tensor, ch + 1);
			const float w = a.weight(r, t);
			ar = fmaf(fmaf(k, v1.x - v0.x, v0.x), w, ar);
			ai = fmaf(fmaf(k, v1.y - v0.y, v0.y), w, ai);
		}
	}
	a.partial[static_cast<uint64_t>(r) * a.npix + p] = make_float2(ar, ai);
}

// The same sums with every record passing through LDS: a workgroup takes one
// receive element and up to 1024 P pixels (lane: pixels pb 1024 P + k 1024 +
// tid), and copies the receive element's records HBM -> LDS transmit after
// transmit, each once, in `pieces` of at most half the LDS, so that one piece
// is copied while the one before is used.  A position lies in exactly one piece
// (consecutive pieces overlap by four entries), so the sums are the same fma
// chains as above.  Bound by reading the tensor once per pixel block: the gather
// form moves a 128-byte line for the 8 or 16 bytes of a pair (192 elements, 96 x
// 96 points, 32 768 FP16 samples: 4.81 ms; this 0.94, 5.1 TB/s).
struct RecordArgs {
	uint32_t pieces, slots;   // pieces of a record, 1 KiB slots of a piece
	uint32_t step;            // entries from one piece to the next
	uint32_t npb;             // pixel blocks
};
constexpr uint32_t kRecordLanes = 1024;
constexpr uint32_t kRecordLds = 160u * 1024u;

template<int STORAGE, int P>
__global__ void __launch_bounds__(kRecordLanes) das_record_sums_kernel(const DasArgs a, const RecordArgs R)
{
	using E = typename Entry<STORAGE>::T;
	constexpr uint32_t ESZ = sizeof(E), NW = kRecordLanes / 64;
	extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
	const uint32_t tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64);
	// the pixel blocks of a receive element follow each other on one XCD and
	// share its records through the L2
	const uint32_t item = xcd_item(), r = item / R.npb, pb = item % R.npb;
	const uint32_t buf_bytes = R.slots * 1024u;
	const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<size_t>((__attribute__((address_space(3))) void*)smem));
	const uint32_t voff = tid % 64 * 16;
	const uint64_t chan_bytes = static_cast<uint64_t>(a.L) * ESZ;
	const uint64_t p0 = static_cast<uint64_t>(pb) * (kRecordLanes * P) + tid;

	float drx[P], dt[P], dnext[P], ar[P], ai[P];
	uint64_t px[P];
#pragma unroll
	for (int k = 0; k < P; ++k) {
		// lanes past the last pixel shadow it
		const uint64_t p = p0 + static_cast<uint64_t>(k) * kRecordLanes;
		px[k] = p < a.npix ? p : a.npix - 1;
		drx[k] = a.delay[static_cast<uint64_t>(r) * a.npix + px[k]];
		ar[k] = ai[k] = 0.0f;
	}
	auto load_delays = [&](uint32_t t) {
		const float* row = a.delay + static_cast<uint64_t>(a.first_tx + t) * a.npix;
#pragma unroll
		for (int k = 0; k < P; ++k) dnext[k] = row[px[k]];
	};
	load_delays(0);

	// Copy cursor: piece is_j of transmit is_t into buffer is_b.  Only the slots
	// with entries up to index L; the last slot may reach past them (into the
	// next channel, or the padding after the tensor).
	uint32_t is_t = 0, is_j = 0, is_b = 0;
	const unsigned char* chan = static_cast<const unsigned char*>(a.tensor) + r * chan_bytes;
	auto issue = [&]() {
		const uint32_t first = is_j * R.step;
		const uint32_t need = ((a.L + 1u - first) * ESZ + 1023u) / 1024u, n = need < R.slots ? need : R.slots;
		const uint32_t h = (n + NW - 1) / NW, s0 = wave * h;
		uint32_t left = s0 < n ? (h < n - s0 ? h : n - s0) : 0u;
		const unsigned char* src = chan + static_cast<uint64_t>(first) * ESZ + s0 * 1024u;
		uint32_t dst = lds0 + is_b * buf_bytes + s0 * 1024u;
		for (; left > 4; left -= 4, src += 4096, dst += 4096) lds_dma16_slots(src, voff, dst, 4);
		lds_dma16_slots(src, voff, dst, left);
		is_b ^= 1u;
		if (++is_j == R.pieces) {
			is_j = 0;
			++is_t;
			chan += chan_bytes * a.nrx;
		}
	};
	issue();
	uint32_t buf = 0;
	for (uint32_t t = 0; t < a.ntx; ++t) {
		const float w = a.weight(r, t);
		for (uint32_t j = 0; j < R.pieces; ++j) {
			// this piece and, with a transmit's first, its delays have arrived;
			// every wave is done with the other buffer
			MISTA_VMCNT(0);
			if (j == 0) {
#pragma unroll
				for (int k = 0; k < P; ++k) {
					asm volatile("" : "+v"(dnext[k]));
					dt[k] = a.offset + dnext[k];
				}
			}
			__syncthreads();
			if (is_t < a.ntx) issue();
			if (j == 0 && t + 1 < a.ntx) load_delays(t + 1);
			const uint32_t first = j * R.step, end = j + 1 == R.pieces ? a.L - 1u : first + R.step;
			const uint32_t lo = __float_as_uint(static_cast<float>(first)), span = __float_as_uint(static_cast<float>(end)) - lo;
			const uint32_t base = lds0 + buf * buf_bytes;
			constexpr int G = P < 4 ? P : 4;   // pixels whose LDS reads are in flight together
#pragma unroll
			for (int k0 = 0; k0 < P; k0 += G) {
				uint32_t addr[G];
				float kf[G];
				bool ok[G];
#pragma unroll
				for (int q = 0; q < G; ++q) {
					const float pos = dt[k0 + q] + drx[k0 + q];
					// first <= pos < end by the bit patterns, in order for
					// floats >= 0; negative values and NaN are above them
					ok[q] = __float_as_uint(pos) - lo < span;
					kf[q] = __builtin_amdgcn_fractf(pos);
					addr[q] = ok[q] ? (static_cast<uint32_t>(pos) - first) * ESZ + base : base;
				}
				typename LdsPair<ESZ>::T v[G];
				lds_read_pairs<ESZ, G>(addr, v);
#pragma unroll
				for (int q = 0; q < G; ++q) {
					const float2 s = Entry<STORAGE>::lerp2(v[q], kf[q]);
					const float nr = fmaf(s.x, w, ar[k0 + q]);
					ar[k0 + q] = ok[q] ? nr : ar[k0 + q];
					if constexpr (STORAGE != kStorageReal) {
						const float ni = fmaf(s.y, w, ai[k0 + q]);
						ai[k0 + q] = ok[q] ? ni : ai[k0 + q];
					}
				}
			}
			buf ^= 1u;
		}
	}
#pragma unroll
	for (int k = 0; k < P; ++k) {
		const uint64_t p = p0 + static_cast<uint64_t>(k) * kRecordLanes;
		if (p < a.npix) a.partial[static_cast<uint64_t>(r) * a.npix + p] = make_float2(ar[k], ai[k]);
	}
}

// A lane per pixel: the per-rx sums in rx order through the same statistics
// as both other kernels (so the images equal the tiled kernel's).
template<int CF>
__global__ void __launch_bounds__(64) das_rx_stats_kernel(const DasArgs a)
{
	const uint64_t p = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
	if (p >= a.npix) return;
	PixelStats<CF> st;
	const float2* src = a.partial + p;
	uint32_t r = 0;
	for (; r + 16 <= a.nrx; r += 16) {   // loads in flight: few lanes share the chip
		float2 v[16];
#pragma unroll
		for (uint32_t k = 0; k < 16; ++k) v[k] = src[(r + k) * a.npix];
#pragma unroll
		for (uint32_t k = 0; k < 16; ++k) st.add_rx(v[k].x, v[k].y, r + k == 0);
	}
	for (; r < a.nrx; ++r) {
		const float2 v = src[r * a.npix];
		st.add_rx(v.x, v.y, r == 0);
	}
	st.write(a, p);
}

// Record form: pixels a lane (p) and pixel blocks, pieces of a record.  Up to 256
// workgroups, a CU each, as long as the records' bytes (each block copies all of
// them) stay below 64 for each pixel, half a cache line of the gather form, and 12
// pixels a lane.  Not where one block passes that (few pixels), nor where a record
// takes more than 8 pieces, which every pixel passes.
bool record_plan(const FrameGeom& g, RecordArgs& R, uint32_t& p)
{
	constexpr uint32_t kMaxP = 12;
	const uint64_t bytes = (static_cast<uint64_t>(g.L) + 1u) * storage_bytes(g.storage);
	const uint64_t blocks = (g.npix + kRecordLanes - 1) / kRecordLanes, few = (blocks + kMaxP - 1) / kMaxP;
	const uint64_t most = g.npix * 64u / bytes;   // blocks whose records are that many bytes
	const uint64_t npb = std::max(few, std::min({blocks, static_cast<uint64_t>(256u / std::min(g.nrx, 256u)), most}));
	const uint32_t cap = kRecordLds / 2048u - 1u;   // slots of the largest piece
	const uint64_t pieces = (bytes + cap * 1024u - 33u) / (cap * 1024u - 32u);
	if (pieces > 8 || npb > most || npb * g.nrx >= (1ull << 31)) return false;
	R.npb = static_cast<uint32_t>(npb);
	R.pieces = static_cast<uint32_t>(pieces);
	R.slots = static_cast<uint32_t>((bytes + pieces - 1) / pieces + 32u + 1023u) / 1024u;
	R.step = R.slots * 1024u / static_cast<uint32_t>(storage_bytes(g.storage)) - 4u;
	p = static_cast<uint32_t>((blocks + npb - 1) / npb);
	return true;
}

template<int STORAGE>
void launch_record(const FrameGeom& g, const DasArgs& a, const RecordArgs& R, uint32_t p, hipStream_t s)
{
	const uint32_t lds = 2u * R.slots * 1024u;
	auto go = [&](auto kern) {
		HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
				static_cast<int>(lds)));
		hipLaunchKernelGGL(kern, dim3(g.nrx * R.npb), dim3(kRecordLanes), lds, s, a, R);
	};
	if (p <= 1) go(das_record_sums_kernel<STORAGE, 1>);
	else if (p <= 2) go(das_record_sums_kernel<STORAGE, 2>);
	else if (p <= 4) go(das_record_sums_kernel<STORAGE, 4>);
	else if (p <= 8) go(das_record_sums_kernel<STORAGE, 8>);
	else go(das_record_sums_kernel<STORAGE, 12>);
}

template<int STORAGE>
void launch_rx_parallel(const FrameGeom& g, const DasArgs& a, hipStream_t s)
{
	const uint32_t nb = static_cast<uint32_t>((g.npix + 255) / 256), ns = static_cast<uint32_t>((g.npix + 63) / 64);
	RecordArgs R;
	uint32_t p = 0;
	if (record_plan(g, R, p)) launch_record<STORAGE>(g, a, R, p, s);
	else hipLaunchKernelGGL(das_rx_sums_kernel<STORAGE>, dim3(nb, g.nrx), dim3(256), 0, s, a);
	HIP_CHECK(hipGetLastError());
	switch (g.cf_kind) {
	case MISTA_CF_NONE: hipLaunchKernelGGL(das_rx_stats_kernel<MISTA_CF_NONE>, dim3(ns), dim3(64), 0, s, a); break;
	case MISTA_CF_PCF: hipLaunchKernelGGL(das_rx_stats_kernel<MISTA_CF_PCF>, dim3(ns), dim3(64), 0, s, a); break;
	default: hipLaunchKernelGGL(das_rx_stats_kernel<MISTA_CF_SCF>, dim3(ns), dim3(64), 0, s, a); break;
	}
}

template<int STORAGE, bool RX_OUTER>
void launch_gather(const FrameGeom& g, const DasArgs& a, hipStream_t s)
{
	const dim3 grid(static_cast<uint32_t>((g.npix + 255) / 256));
	switch (g.cf_kind) {
	case MISTA_CF_NONE:
		hipLaunchKernelGGL((das_gather_kernel<STORAGE, MISTA_CF_NONE, RX_OUTER>), grid, dim3(256), 0, s, a);
		break;
	case MISTA_CF_PCF:
		hipLaunchKernelGGL((das_gather_kernel<STORAGE, MISTA_CF_PCF, true>), grid, dim3(256), 0, s, a);
		break;
	default:
		hipLaunchKernelGGL((das_gather_kernel<STORAGE, MISTA_CF_SCF, true>), grid, dim3(256), 0, s, a);
		break;
	}
	HIP_CHECK(hipGetLastError());
}

template<bool RX_OUTER>
void launch_gather_any(const FrameGeom& g, const DasArgs& a, hipStream_t s)
{
	switch (g.storage) {
	case MISTA_STORAGE_F32: launch_gather<MISTA_STORAGE_F32, RX_OUTER>(g, a, s); break;
	case MISTA_STORAGE_F16: launch_gather<MISTA_STORAGE_F16, RX_OUTER>(g, a, s); break;
	case kStorageReal: launch_gather<kStorageReal, RX_OUTER>(g, a, s); break;
	default: launch_gather<MISTA_STORAGE_BF16, RX_OUTER>(g, a, s); break;
	}
}

// A lane per tile point: its per-rx sums (the tiled kernel's, [tiles][nrx]
// [tile points]) in rx order through the same statistics as the other forms.
// Bound by reading the sums once (8 bytes per pixel and receive element).
template<int CF>
__global__ void __launch_bounds__(256) das_tile_stats_kernel(const DasArgs a, const TileGeom tg, uint32_t tile0,
		uint32_t npts)
{
	const uint32_t per = npts / 256;
	const uint32_t tl = blockIdx.x / per, q = (blockIdx.x % per) * 256 + threadIdx.x;
	uint32_t col, row;
	bool valid;
	tg.pixel(tile0 + tl, q, col, row, valid);
	if (!valid) return;
	const float2* src = a.partial + static_cast<uint64_t>(tl) * a.nrx * npts + q;
	PixelStats<CF> st;
	uint32_t r = 0;
	for (; r + 4 <= a.nrx; r += 4) {   // four loads in flight
		float2 v[4];
#pragma unroll
		for (uint32_t k = 0; k < 4; ++k) v[k] = src[static_cast<uint64_t>(r + k) * npts];
#pragma unroll
		for (uint32_t k = 0; k < 4; ++k) st.add_rx(v[k].x, v[k].y, r + k == 0);
	}
	for (; r < a.nrx; ++r) {
		const float2 v = src[static_cast<uint64_t>(r) * npts];
		st.add_rx(v.x, v.y, r == 0);
	}
	st.write(a, static_cast<uint64_t>(col) * tg.n2 + row);
}

// Delays of a run of tiles in lane order: [tiles][nrx + ntx][npts], the rx
// rows as in the delay table, the tx rows with the offset added (the first
// add of every position).  Points outside the grid hold the point they shadow.
__global__ void __launch_bounds__(256) tile_delays_kernel(const float* __restrict__ delay, uint64_t npix, TileGeom tg,
		uint32_t tile0, uint32_t npts, uint32_t nrx, uint32_t first_tx, uint32_t rows, float offset,
		float* __restrict__ td)
{
	const uint32_t per = npts / 256;
	const uint32_t tl = blockIdx.x / per, q = (blockIdx.x % per) * 256 + threadIdx.x;
	uint32_t col, row;
	bool valid;
	tg.pixel(tile0 + tl, q, col, row, valid);
	const float* src = delay + static_cast<uint64_t>(col) * tg.n2 + row;
	float* dst = td + static_cast<uint64_t>(tl) * rows * npts + q;
	for (uint32_t e = blockIdx.y; e < rows; e += gridDim.y) {
		float d;
		if (e < nrx) d = src[static_cast<uint64_t>(e) * npix];
		else d = offset + src[static_cast<uint64_t>(first_tx + e - nrx) * npix];
		dst[static_cast<uint64_t>(e) * npts] = d;
	}
}

// (min, max) of every row of the tile delays: a wave per (tile, row).
__global__ void __launch_bounds__(256) tile_bounds_kernel(const float* __restrict__ td, uint64_t nrows, uint32_t npts,
		float2* __restrict__ bounds)
{
	const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
	if (i >= nrows) return;
	const uint32_t lane = threadIdx.x & 63;
	const float* src = td + i * npts;
	float mn = 3.4e38f, mx = -3.4e38f;
	for (uint32_t k = lane; k < npts; k += 64) {
		const float d = src[k];
		mn = fminf(mn, d);
		mx = fmaxf(mx, d);
	}
	for (int o = 32; o > 0; o >>= 1) {
		mn = fminf(mn, __shfl_xor(mn, o, 64));
		mx = fmaxf(mx, __shfl_xor(mx, o, 64));
	}
	if (lane == 0) bounds[i] = make_float2(mn, mx);
}

// Window words of a tile ([rx groups][ntx][kRxGroup]) and the slots of
// its longest window; max_slots takes the longest of all tiles.  A workgroup
// per tile.
__global__ void __launch_bounds__(256) window_params_kernel(const float2* __restrict__ bounds, uint32_t ntx,
		uint32_t nrx, uint32_t nrx_pad, uint32_t L, uint32_t esz, uint32_t* __restrict__ words,
		uint32_t* __restrict__ slots, uint32_t* __restrict__ max_slots)
{
	__shared__ uint32_t red[4];
	const uint32_t tile = blockIdx.x;
	const float2* tb = bounds + static_cast<uint64_t>(tile) * (nrx + ntx);
	const uint32_t n = nrx_pad * ntx;
	uint32_t* out = words + static_cast<uint64_t>(tile) * n;
	uint32_t mslots = 1;
	for (uint32_t i = threadIdx.x; i < n; i += 256) {
		const uint32_t t = i / kRxGroup % ntx, r = i / (kRxGroup * ntx) * kRxGroup + i % kRxGroup;
		uint32_t word = kEdgeBit;   // padding or nothing to stage: excluded
		if (r < nrx) {
			const float2 bt = tb[nrx + t], br = tb[r];
			const float lo = bt.x + br.x;
			const float hi = bt.y + br.y;
			// lo past the record end or NaN: nothing staged, every lane of
			// the pair is excluded by the predicated path.  (lo is never
			// negative: delays are >= 0 and the peak offset is >= 0.)
			if (lo >= 0.0f && lo < static_cast<float>(L)) {
				const uint32_t ws = static_cast<uint32_t>(floorf(lo));
				const float fhi = floorf(hi);
				// entries [ws, floor(hi) + 1], never past index L (one past the record)
				uint32_t need = (fhi >= static_cast<float>(L)) ? L + 1u - ws : static_cast<uint32_t>(fhi) + 2u - ws;
				need = min(need, L + 1u - ws);
				const uint32_t k = (need * esz + 1023u) / 1024u;
				mslots = max(mslots, k);
				const bool edge = fhi + 1.0f >= static_cast<float>(L - 1u);
				word = ws * esz | (min(k, 127u) << kSlotShift) | (edge ? kEdgeBit : 0u);
			}
		}
		out[i] = word;
	}
	for (int o = 32; o > 0; o >>= 1)
		mslots = max(mslots, static_cast<uint32_t>(__shfl_xor(static_cast<int>(mslots), o, 64)));
	if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mslots;
	__syncthreads();
	if (threadIdx.x == 0) {
		for (int w = 1; w < 4; ++w) mslots = max(mslots, red[w]);
		slots[tile] = mslots;
		atomicMax(max_slots, mslots);
	}
}

}  // namespace

namespace {

__global__ void zero_u32_kernel(uint32_t* p) { *p = 0u; }

// Tile shape p0 (see launch_tiled) of a geometry.
struct TilePlan {
	TileGeom tg;
	uint32_t ntiles = 0, npts = 0, esz = 0;
	uint64_t key = 0;        // what the window tables depend on, besides grid and offset
	bool ok = false;
};

TilePlan tile_plan(const FrameGeom& g, int p0)
{
	TilePlan tp;
	const uint32_t ny = g.ny ? g.ny : 1u;
	uint32_t tw1 = 16, tw2 = 1, tzh = 16;
	if (ny > 1) { tw1 = 8; tw2 = 8; tzh = 4; }
	switch (p0) {
	case 2: tw1 = 8; tw2 = 1; tzh = 32; break;
	case 3: tw1 = 32; tw2 = 1; tzh = 8; break;
	case 4: tw1 = 8; tw2 = 8; tzh = 4; break;
	case 5: tw1 = 16; tw2 = 1; tzh = 32; break;
	case 6: tw1 = 32; tw2 = 1; tzh = 16; break;
	case 7: tw1 = 8; tw2 = 8; tzh = 8; break;
	case 8: tw1 = 32; tw2 = 1; tzh = 32; break;
	case 9: tw1 = 64; tw2 = 1; tzh = 32; break;
	case 10: tw1 = 16; tw2 = 8; tzh = 8; break;
	case 11: tw1 = 16; tw2 = 16; tzh = 8; break;
	default: break;
	}
	tp.npts = tw1 * tw2 * tzh;
	// More than 128 transmits: 256-point tiles, which copy the most bytes per
	// pixel and pair, are not offered.
	if (g.ntx > 128 && tp.npts < 512) return tp;
	if (g.L >= kMaxWindowL) return tp;
	tp.esz = static_cast<uint32_t>(storage_bytes(g.storage));
	const uint32_t nx = g.n1 / ny;
	tp.tg = TileGeom{g.n1, g.n2, ny, nx, tw1, tw2, tzh, (nx + tw1 - 1) / tw1, (ny + tw2 - 1) / tw2, (g.n2 + tzh - 1) / tzh};
	const uint64_t ntiles64 = static_cast<uint64_t>(tp.tg.tiles_x) * tp.tg.tiles_y * tp.tg.tiles_z;
	if (ntiles64 * (pad_nrx(g.nrx) / kRxGroup) >= (1ull << 31)) return tp;
	tp.ntiles = static_cast<uint32_t>(ntiles64);
	tp.key = 0x9E3779B97F4A7C15ull;
	for (uint64_t v : {static_cast<uint64_t>(p0), static_cast<uint64_t>(ny), static_cast<uint64_t>(tp.esz),
				static_cast<uint64_t>(g.L), static_cast<uint64_t>(g.first_tx), static_cast<uint64_t>(g.ntx)})
		tp.key = (tp.key ^ v) * 0x100000001B3ull;
	tp.ok = true;
	return tp;
}

size_t bounds_bytes(const FrameGeom& g, const TilePlan& tp, uint32_t ntiles)
{
	return static_cast<size_t>(ntiles) * (g.nrx + g.ntx) * sizeof(float2);
}
size_t words_bytes(const FrameGeom& g, const TilePlan& tp, uint32_t ntiles)
{
	return static_cast<size_t>(ntiles) * pad_nrx(g.nrx) * g.ntx * sizeof(uint32_t);
}
size_t delays_bytes(const FrameGeom& g, const TilePlan& tp, uint32_t ntiles)
{
	return static_cast<size_t>(ntiles) * (g.nrx + g.ntx) * tp.npts * sizeof(float);
}
// Per-rx sums of one tile.
size_t sums_bytes(const FrameGeom& g, const TilePlan& tp)
{
	return static_cast<size_t>(g.nrx) * tp.npts * sizeof(float2);
}

// Delays, their bounds, window words and longest windows of the tiles
// [tile0, tile0 + n) into the given buffers; max_slots keeps the longest.
void build_window_tables(const FrameGeom& g, const TilePlan& tp, uint32_t tile0, uint32_t n, const float* d_delay,
		float* td, float2* bounds, uint32_t* words, uint32_t* slots, uint32_t* max_slots, hipStream_t s)
{
	const uint32_t rows = g.nrx + g.ntx;
	const uint32_t nb = n * (tp.npts / 256);
	hipLaunchKernelGGL(tile_delays_kernel, dim3(nb, std::max(1u, std::min(rows, 16384u / std::max(1u, nb)))), dim3(256), 0, s,
			d_delay, g.npix, tp.tg, tile0, tp.npts, g.nrx, g.first_tx, rows, g.offset, td);
	HIP_CHECK(hipGetLastError());
	const uint64_t nrows = static_cast<uint64_t>(n) * rows;
	hipLaunchKernelGGL(tile_bounds_kernel, dim3(static_cast<uint32_t>((nrows + 3) / 4)), dim3(256), 0, s, td, nrows, tp.npts,
			bounds);
	HIP_CHECK(hipGetLastError());
	hipLaunchKernelGGL(window_params_kernel, dim3(n), dim3(256), 0, s, bounds, g.ntx, g.nrx, pad_nrx(g.nrx), g.L, tp.esz, words,
			slots, max_slots);
	HIP_CHECK(hipGetLastError());
}

// The same into the first places of a handle's tables.
void build_tables(const FrameGeom& g, const TilePlan& tp, uint32_t tile0, uint32_t n, const float* d_delay, DasScratch& scratch,
		hipStream_t s)
{
	build_window_tables(g, tp, tile0, n, d_delay, scratch.delays.as<float>(), scratch.bounds.as<float2>(),
			scratch.params.as<uint32_t>(), scratch.slots.as<uint32_t>(), scratch.partial.as<uint32_t>(), s);
}

uint32_t read_u32(const uint32_t* d, hipStream_t s)
{
	uint32_t v = 0;
	HIP_CHECK(hipMemcpyAsync(&v, d, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
	HIP_CHECK(hipStreamSynchronize(s));
	return v;
}

// How a tile's sums are formed (das_tile's template parameters).
struct Chunking {
	uint32_t r = 0;       // receive elements per workgroup: pairs per transmit step
	uint32_t nt = 0;      // lanes
	uint32_t rc = 0;      // receive elements per chunk
	uint32_t nbmax = 0;   // most chunk buffers
	uint32_t lds = 0;     // LDS bytes
	uint32_t nbuf = 0;    // chunk buffers of the tile with the longest window
	bool same(const Chunking& o) const { return r == o.r && nt == o.nt && rc == o.rc && nbmax == o.nbmax && lds == o.lds; }
	// p1 that gives this chunking again, with the budget that was asked for
	int p1(uint32_t npts, int asked) const
	{
		const uint32_t wide = npts != 2048u || nt == 512u ? 0u : rc == 2u ? 2u : 1u;
		return static_cast<int>(r | (nbuf << 8) | (wide << 24)) | (asked & 0xFF0000);
	}
};

// Chunking of the tiled kernel over windows of at most S slots.  p1: byte 0
// pairs per transmit step (4, 8, or 16 on 512-point tiles), byte 1 most chunk
// buffers, byte 2 LDS budget in KiB (default: the smallest in which two
// buffers of the longest window fit, of those that put 4, 3, 2 or 1
// workgroups on a CU; LDS is handed out in 1280-byte blocks, of which 52 KiB
// take a third and 53 KiB more), byte 3 for 2048-point tiles: 1 = 1024 lanes in
// any budget, 2 = the same with chunks of two receive elements.  Returns false
// when nothing fits.
bool choose_chunking(uint32_t npts, int p1, uint32_t S, Chunking& c)
{
	if (S > kMaxSlots) return false;
	// (8 on 256 points: they have 4 only, whose ring is the smaller one)
	const uint32_t asked_r = static_cast<uint32_t>(p1) & 0xFF, want_r = npts == 256u && asked_r == 8u ? 4u : asked_r;
	const uint32_t want_nb = (static_cast<uint32_t>(p1) >> 8) & 0xFF;
	const uint32_t want_kb = (static_cast<uint32_t>(p1) >> 16) & 0xFF;
	const uint32_t wide = npts == 2048u ? static_cast<uint32_t>(p1) >> 24 & 3u : 0u;
	c.nbmax = want_nb ? std::max(2u, std::min(want_nb, 4u)) : 4u;
	for (uint32_t kb : {40u, 52u, 80u, 160u}) {
		if (want_kb) {
			if (kb != 40u) break;
			kb = std::min(want_kb, 160u);
		}
		c.nt = npts <= 512 ? 256u : npts == 1024 ? 512u : kb <= 80u && !wide ? 512u : 1024u;
		// (2048 points: two workgroups a CU at most)
		if (!want_kb && npts == 2048u && kb < 80u) continue;
		c.lds = kb * 1024u;
		for (uint32_t r : {4u, 8u, 16u}) {
			if (want_r ? r != want_r : r == 16u) continue;
			if ((r == 16u && npts != 512u) || (r == 8u && (npts == 256u || (npts == 2048u && (c.nt == 512u || wide == 2u))))) continue;
			const uint32_t rc = npts == 2048u && (c.nt == 512u || wide == 2u) ? 2u : 4u;
			c.r = r;
			c.rc = rc;
			if (r == 16u) c.nt = 512u;
			c.nbuf = tile_buffers(c.nbmax, c.lds, S, rc, r / rc, npts);
			if (c.nbuf) return true;
		}
	}
	// long windows on 2048 points: chunks of two receive elements in the whole LDS
	if (npts == 2048u && p1 == 0) return choose_chunking(npts, 4 | (160 << 16) | (2 << 24), S, c);
	return false;
}

TileArgs tile_args(const FrameGeom& g, const DasArgs& a, uint32_t ntiles, const Chunking& c)
{
	TileArgs A;
	A.tensor = a.tensor;
	A.td = nullptr;
	A.words = nullptr;
	A.slots = nullptr;
	A.w = a.w;
	A.partial = a.partial;
	A.ntx = g.ntx;
	A.nrx = g.nrx;
	A.L = g.L;
	A.ntiles = ntiles;
	A.ngrp = (g.nrx + c.r - 1) / c.r;
	A.ngrp4 = pad_nrx(g.nrx) / kRxGroup;
	A.lds = c.lds;
	A.nbmax = c.nbmax;
	return A;
}

// Launches the tiled kernel of the batch's storage.
void launch_batch(int storage, const TileBatch& B, uint32_t npts, const Chunking& c, hipStream_t s)
{
	switch (storage) {
	case MISTA_STORAGE_F32: launch_tile_storage<MISTA_STORAGE_F32>(B, npts, c.r, c.rc, c.nt, s); break;
	case MISTA_STORAGE_F16: launch_tile_storage<MISTA_STORAGE_F16>(B, npts, c.r, c.rc, c.nt, s); break;
	case kStorageReal: launch_tile_storage<kStorageReal>(B, npts, c.r, c.rc, c.nt, s); break;
	default: launch_tile_storage<MISTA_STORAGE_BF16>(B, npts, c.r, c.rc, c.nt, s); break;
	}
	HIP_CHECK(hipGetLastError());
}

// The statistics of the tiles [tile0, tile0 + n), whose sums start at a.partial.
void launch_tile_stats(const FrameGeom& g, const TilePlan& tp, const DasArgs& a, uint32_t tile0, uint32_t n, hipStream_t s)
{
	const dim3 grid(n * (tp.npts / 256));
	switch (g.cf_kind) {
	case MISTA_CF_NONE:
		hipLaunchKernelGGL(das_tile_stats_kernel<MISTA_CF_NONE>, grid, dim3(256), 0, s, a, tp.tg, tile0, tp.npts);
		break;
	case MISTA_CF_PCF:
		hipLaunchKernelGGL(das_tile_stats_kernel<MISTA_CF_PCF>, grid, dim3(256), 0, s, a, tp.tg, tile0, tp.npts);
		break;
	default:
		hipLaunchKernelGGL(das_tile_stats_kernel<MISTA_CF_SCF>, grid, dim3(256), 0, s, a, tp.tg, tile0, tp.npts);
		break;
	}
	HIP_CHECK(hipGetLastError());
}

// Most bytes of per-rx sums held at a time: a frame whose sums need more runs
// its tiles in several launches.
constexpr size_t kSumsBytes = static_cast<size_t>(1) << 30;

uint32_t slab_tiles(const FrameGeom& g, const TilePlan& tp)
{
	return static_cast<uint32_t>(std::max<size_t>(1, std::min<size_t>(tp.ntiles, kSumsBytes / sums_bytes(g, tp))));
}

// The tiles [tile0, tile0 + n) of a frame: per-rx sums, then statistics.
void run_tiles(const FrameGeom& g, const TilePlan& tp, const TileArgs& first, const DasArgs& a, uint32_t tile0, uint32_t n,
		const Chunking& c, hipStream_t s)
{
	TileBatch B{};
	B.jobs[0] = first;
	B.njobs = 1;
	B.total = B.first[1] = n * first.ngrp;
	launch_batch(g.storage, B, tp.npts, c, s);
	launch_tile_stats(g, tp, a, tile0, n, s);
}

// The shape that is reported for p0 (0: the default).
int reported_shape(const TilePlan& tp, int p0) { return p0 == 0 ? (tp.tg.ny > 1 ? 4 : 1) : p0; }

// Bytes of the tables of n tiles.
size_t table_bytes(const FrameGeom& g, const TilePlan& tp, uint32_t n)
{
	return delays_bytes(g, tp, n) + bounds_bytes(g, tp, n) + words_bytes(g, tp, n) + n * sizeof(uint32_t);
}

// Tables and sums of a slab of a frame whose tables are not kept whole.
constexpr size_t kSlabBytes = static_cast<size_t>(1) << 30;

// How many tiles' tables and sums a frame holds at a time within a limit: whole,
// the tables of all tiles and the sums of a slab of them, else both of a slab.
struct TileRun {
	bool whole = false;
	uint32_t slab = 0;
	uint32_t tables(const TilePlan& tp) const { return whole ? tp.ntiles : slab; }
};

TileRun tile_run(const FrameGeom& g, const TilePlan& tp, size_t limit)
{
	TileRun r;
	r.slab = slab_tiles(g, tp);
	r.whole = table_bytes(g, tp, tp.ntiles) + r.slab * sums_bytes(g, tp) <= limit;
	if (!r.whole) {
		const size_t per = table_bytes(g, tp, 1) + sums_bytes(g, tp);
		r.slab = static_cast<uint32_t>(std::max<size_t>(1, std::min<size_t>(r.slab, std::min(limit, kSlabBytes) / per)));
	}
	return r;
}

// Tables of tile shape p0 (see tile_run), built when the grid, shape or offset
// changed, which synchronises s; a slab's are built again as it runs.  Where the
// device has no room for them, a smaller slab; false when the shape does not apply
// or not even a tile's fit.
bool ensure_tables(const FrameGeom& g, const TilePlan& tp, DasScratch& scratch, const float* d_delay, hipStream_t s, TileRun& run)
{
	if (!tp.ok) return false;
	if (scratch.cap_version != g.grid_version) {
		scratch.table_cap = scratch.table_limit;
		scratch.cap_version = g.grid_version;
	}
	uint32_t* d_max = static_cast<uint32_t*>(scratch.partial.reserve(256));
	for (;;) {
		run = tile_run(g, tp, scratch.table_cap);
		const uint32_t n = run.tables(tp);
		DeviceBuffer* const buf[5] = {&scratch.delays, &scratch.bounds, &scratch.params, &scratch.slots, &scratch.partials};
		const size_t bytes[5] = {delays_bytes(g, tp, n), bounds_bytes(g, tp, n), words_bytes(g, tp, n), n * sizeof(uint32_t),
				run.slab * sums_bytes(g, tp)};
		// a buffer that grows loses what it held, and so do all where another
		// shape's larger ones would pass the limit together with this one's
		bool grows = false, fits = true;
		size_t need = 0, held = 0;
		for (int k = 0; k < 5; ++k) {
			grows = grows || (k < 4 && bytes[k] > buf[k]->capacity());
			need += bytes[k];
			held += std::max(bytes[k], buf[k]->capacity());
		}
		const bool drop = held > std::max(need, scratch.table_cap);
		if (grows || drop) scratch.bounds_version = ~0ull;
		if (drop)
			for (DeviceBuffer* b : buf) b->release();
		for (int k = 0; k < 5; ++k) fits = fits && buf[k]->try_reserve(bytes[k]);
		if (fits) break;
		scratch.bounds_version = ~0ull;
		for (DeviceBuffer* b : buf) b->release();
		if (n == 1) return false;
		scratch.table_cap = std::min(run.whole ? kSlabBytes : need / 2, need - 1);
	}
	const bool same = scratch.bounds_version == g.grid_version && scratch.params_key == tp.key && scratch.params_offset == g.offset;
	if (!same || (run.whole && !scratch.whole)) {
		scratch.bounds_version = ~0ull;   // nothing half-built is kept
		hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, s, d_max);
		HIP_CHECK(hipGetLastError());
		const uint32_t n = run.tables(tp);
		for (uint32_t t0 = 0; t0 < tp.ntiles; t0 += n) build_tables(g, tp, t0, std::min(n, tp.ntiles - t0), d_delay, scratch, s);
		scratch.max_slots = read_u32(d_max, s);
		scratch.bounds_version = g.grid_version;
		scratch.params_key = tp.key;
		scratch.params_offset = g.offset;
	}
	scratch.whole = run.whole;
	return true;
}

// Tile shapes that the tuner tries, in order.  The larger tiles copy fewer bytes
// per pixel and pair (64x32 points: 0.67 window entries per point and pair against
// 1.63 at 16x32, 128-element frame; DAS 5.8 ms at 64x32, 8.3 at 32x32, 9.1 at
// 32x16).  The large ones go first, where they give every CU several workgroups.
std::vector<int> tuner_shapes(const FrameGeom& g)
{
	std::vector<int> shapes;
	for (int p0 : (g.ny > 1 ? std::vector<int>{11, 10} : std::vector<int>{9, 8})) {
		const TilePlan tp = tile_plan(g, p0);
		if (tp.ok && static_cast<uint64_t>(tp.ntiles) * (pad_nrx(g.nrx) / kRxGroup) >= 1024u) shapes.push_back(p0);
	}
	for (int p0 : (g.ny > 1 ? std::vector<int>{7, 4} : std::vector<int>{6, 5, 1, 3, 2})) shapes.push_back(p0);
	return shapes;
}

}  // namespace

// A sixteenth of the device's memory.  Tables kept whole save building them in every
// frame (1024 x 64 elements over 128 x 128 x 96 points, 7 GB of tables: DAS 46.6 ms
// whole, 71.0 a slab at a time); past the limit the copy of the delays would stand
// in the way of other handles' delay tables and tensors.
size_t das_table_limit(int device)
{
	size_t total = 0;
	HIP_CHECK(hipDeviceTotalMem(&total, device));
	return total / 16;
}

size_t das_table_bytes(const FrameGeom& g, size_t limit)
{
	size_t most[5] = {0, 0, 0, 0, 0}, one = 0;
	for (int p0 : tuner_shapes(g)) {
		const TilePlan tp = tile_plan(g, p0);
		if (!tp.ok) continue;
		const TileRun run = tile_run(g, tp, limit);
		const uint32_t n = run.tables(tp);
		const size_t bytes[5] = {delays_bytes(g, tp, n), bounds_bytes(g, tp, n), words_bytes(g, tp, n), n * sizeof(uint32_t),
				run.slab * sums_bytes(g, tp)};
		size_t sum = 0;
		for (int k = 0; k < 5; ++k) {
			most[k] = std::max(most[k], bytes[k]);
			sum += bytes[k];
		}
		one = std::max(one, sum);
	}
	return std::min(std::max(one, limit), most[0] + most[1] + most[2] + most[3] + most[4]);
}

// Builds (or reuses) the tables for tile shape p0 and runs the tiled kernel with
// the chunking p1 (see choose_chunking).  p0: 0/1 = 16x16 (planes) or 8x8x4
// (volumes), 2 = 8x32, 3 = 32x8, 4 = 8x8x4; 512 points: 5 = 16x32,
// 6 = 32x16, 7 = 8x8x8; 1024 points: 8 = 32x32, 10 = 16x8x8; 2048 points:
// 9 = 64x32, 11 = 16x16x8.  Returns false when the windows do not fit.
bool launch_tiled(const FrameGeom& g, int p0, int p1, DasScratch& scratch, const DasArgs& args, const float* d_delay,
		hipStream_t s)
{
	const TilePlan tp = tile_plan(g, p0);
	TileRun run;
	if (!ensure_tables(g, tp, scratch, d_delay, s, run)) return false;
	Chunking c;
	if (!choose_chunking(tp.npts, p1, scratch.max_slots, c)) return false;
	DasArgs a = args;
	a.partial = scratch.partials.as<float2>();
	for (uint32_t t0 = 0; t0 < tp.ntiles; t0 += run.slab) {
		const uint32_t n = std::min(run.slab, tp.ntiles - t0), first = run.whole ? t0 : 0u;
		if (!run.whole) build_tables(g, tp, t0, n, d_delay, scratch, s);
		TileArgs A = tile_args(g, a, n, c);
		A.td = scratch.delays.as<const float>() + delays_bytes(g, tp, first) / sizeof(float);
		A.words = scratch.params.as<const uint32_t>() + words_bytes(g, tp, first) / sizeof(uint32_t);
		A.slots = scratch.slots.as<const uint32_t>() + first;
		run_tiles(g, tp, A, a, t0, n, c, s);
	}
	scratch.last_p0 = reported_shape(tp, p0);
	scratch.last_p1 = c.p1(tp.npts, p1);
	return true;
}

// Kernel arguments of a frame.
DasArgs das_args(const FrameGeom& g, const void* d_tensor, const float* d_delay, const float* d_w, float* d_value,
		float* d_factor)
{
	DasArgs a;
	a.partial = nullptr;
	a.tensor = d_tensor;
	a.delay = d_delay;
	a.w = d_w;
	a.value = d_value;
	a.factor = d_factor;
	a.npix = g.npix;
	a.first_tx = g.first_tx;
	a.ntx = g.ntx;
	a.nrx = g.nrx;
	a.L = g.L;
	a.offset = g.offset;
	if (g.cf_kind == MISTA_CF_PCF) {
		// CoherenceFactor.h:243-246: sigma0 = pi/sqrt(3) (stored as float),
		// factor = gamma / sigma0
		const float sigma0 = static_cast<float>(3.14159265358979323846 / std::sqrt(3.0));
		a.cf_factor = g.cf_param / sigma0;
	} else {
		a.cf_factor = g.cf_param;
	}
	a.inv_num = 1.0f / static_cast<float>(static_cast<uint64_t>(g.ntx) * g.nrx);
	a.signed_value = (g.storage == kStorageReal) ? 1 : 0;
	return a;
}

// ---------------------------------------------------------------- no allocation

// Bytes of the window tables that decide whether the entry point takes a
// geometry (its documented limit): transmits padded to 32, 64, 128 or equal
// blocks of whole 8-pair chunks, and the sums between those blocks.
static size_t noalloc_table_bytes(const FrameGeom& g, const TilePlan& tp)
{
	const size_t pad = budget_pad_ntx(g.ntx);
	auto up = [](size_t b) { return (b + 255) / 256 * 256; };
	return up(pad > 128 ? static_cast<size_t>(g.nrx) * g.npix * sizeof(float2) : 0) +
			up(static_cast<size_t>(tp.ntiles) * g.num_elements * sizeof(float2)) +
			up(static_cast<size_t>(tp.ntiles) * g.nrx * pad * sizeof(uint32_t)) + 256;
}

void launch_das_noalloc(const FrameGeom& g, int tuned_p0, int tuned_p1, DasScratch& last, const void* d_tensor,
		const float* d_delay, const float* d_w, float* d_value, float* d_factor, hipStream_t s)
{
	unsigned char* base = noalloc_scratch();
	DasArgs a = das_args(g, d_tensor, d_delay, d_w, d_value, d_factor);
	// the tuned tile shape when it fits, else the default, else the larger tiles
	std::vector<std::pair<int, int>> shapes;
	if (tuned_p0 >= 0) shapes.emplace_back(tuned_p0, tuned_p1);
	const std::vector<int> defaults = g.ny > 1 ? std::vector<int>{4, 7} : std::vector<int>{1, 5, 6};
	for (int p0 : defaults) shapes.emplace_back(p0, 0);
	if (!g.finite_weights) shapes.clear();
	size_t need_min = ~size_t(0);
	for (int p0 : defaults) {
		FrameGeom gl = g;
		gl.L = std::min(g.L, kMaxWindowL - 1);   // (the shape alone, whatever the record)
		const TilePlan tp = tile_plan(gl, p0);
		if (tp.ok) need_min = std::min(need_min, noalloc_table_bytes(g, tp));
	}
	if (need_min != ~size_t(0) && need_min > kNoAllocTableBytes)
		MISTA_THROW(MISTA_E_INVALID_PARAM, "The DAS window tables of this geometry need " << need_min
				<< " bytes; the no-allocation entry point holds at most " << kNoAllocTableBytes << '.');
	// no tile of the frame fits the scratch, or the record the window words, or none may run
	bool too_large = g.L >= kMaxWindowL || !g.finite_weights;
	for (const auto& sh : shapes) {
		const TilePlan tp = tile_plan(g, sh.first);
		if (!tp.ok) continue;
		// the scratch: longest window, then the tables and sums of `slab` tiles
		size_t off[6] = {256, 0, 0, 0, 0, 0};
		auto layout = [&](uint32_t n) {
			const size_t bytes[5] = {delays_bytes(g, tp, n), bounds_bytes(g, tp, n), words_bytes(g, tp, n),
					static_cast<size_t>(n) * sizeof(uint32_t), n * sums_bytes(g, tp)};
			for (int k = 0; k < 5; ++k) off[k + 1] = off[k] + (bytes[k] + 255) / 256 * 256;
			return off[5] <= kNoAllocScratchBytes;
		};
		if (!layout(1)) {
			too_large = true;
			continue;
		}
		const size_t per = off[5] - 256;   // an upper bound per tile
		const uint32_t slab = static_cast<uint32_t>(std::min<size_t>(tp.ntiles, (kNoAllocScratchBytes - 256) / per));
		if (!layout(slab)) MISTA_THROW(MISTA_E_INVALID_STATE, "no-allocation DAS scratch layout");
		uint32_t* d_max = reinterpret_cast<uint32_t*>(base);
		float* td = reinterpret_cast<float*>(base + off[0]);
		uint32_t* words = reinterpret_cast<uint32_t*>(base + off[2]);
		uint32_t* slots = reinterpret_cast<uint32_t*>(base + off[3]);
		a.partial = reinterpret_cast<float2*>(base + off[4]);
		auto build = [&](uint32_t t0, uint32_t n) {
			build_window_tables(g, tp, t0, n, d_delay, td, reinterpret_cast<float2*>(base + off[1]), words, slots, d_max, s);
		};
		hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, s, d_max);
		HIP_CHECK(hipGetLastError());
		for (uint32_t t0 = 0; t0 < tp.ntiles; t0 += slab) build(t0, std::min(slab, tp.ntiles - t0));
		Chunking c;
		if (!choose_chunking(tp.npts, sh.second, read_u32(d_max, s), c)) continue;
		for (uint32_t t0 = 0; t0 < tp.ntiles; t0 += slab) {
			const uint32_t n = std::min(slab, tp.ntiles - t0);
			if (slab < tp.ntiles) build(t0, n);
			TileArgs A = tile_args(g, a, n, c);
			A.td = td;
			A.words = words;
			A.slots = slots;
			run_tiles(g, tp, A, a, t0, n, c, s);
		}
		last.last_p0 = reported_shape(tp, sh.first);
		last.last_p1 = c.p1(tp.npts, sh.second);
		return;
	}
	if (!too_large)
		MISTA_THROW(MISTA_E_INVALID_PARAM, "The signal windows of this geometry do not fit the tiled DAS kernel.");
	// a tile's tables alone pass the scratch: one pixel per lane, which needs none
	launch_gather_any<true>(g, a, s);
	last.last_p0 = -1;
	last.last_p1 = 0;
}

// ---------------------------------------------------------------- batches

uint32_t launch_das_batch(const std::vector<DasBatchItem>& items, hipStream_t s)
{
	struct Ready {
		size_t i;
		TilePlan tp;
		int p0, p1;
		uint64_t cls;
	};
	std::vector<Ready> ready;
	std::vector<size_t> alone;
	for (size_t i = 0; i < items.size(); ++i) {
		const DasBatchItem& it = items[i];
		const FrameGeom& g = *it.g;
		int p0 = -1, p1 = 0;
		if (!g.finite_weights) {
			// no tiles
		} else if (it.t->variant != 1 && (it.t->variant == 2 || it.t->p0 || it.t->p1)) {
			p0 = it.t->p0;
			p1 = it.t->p1;
		} else if (it.t->variant != 1 && it.scratch->tuned_p0 >= 0) {
			p0 = it.scratch->tuned_p0;
			p1 = it.scratch->tuned_p1;
		}
		TilePlan tp;
		TileRun run;
		if (p0 >= 0) tp = tile_plan(g, p0);
		if (p0 < 0 || !ensure_tables(g, tp, *it.scratch, it.delay, s, run) || it.scratch->max_slots > kMaxSlots ||
				!run.whole || run.slab < tp.ntiles) {
			alone.push_back(i);   // untuned geometry (it tunes alone), gather kernel, no tiled form, or a slab at a time
			continue;
		}
		const uint64_t cls = static_cast<uint64_t>(g.storage) | (static_cast<uint64_t>(tp.npts) << 32);
		ready.push_back({i, tp, p0, p1, cls});
	}
	uint32_t shared = 0;
	std::vector<bool> done(ready.size(), false);
	for (size_t a0 = 0; a0 < ready.size(); ++a0) {
		if (done[a0]) continue;
		// the next group: frames of a0's class, in order, at most kMaxBatch
		std::vector<size_t> grp;
		uint64_t total = 0;
		for (size_t b = a0; b < ready.size() && grp.size() < kMaxBatch; ++b) {
			const uint64_t n = static_cast<uint64_t>(ready[b].tp.ntiles) * (pad_nrx(items[ready[b].i].g->nrx) / kRxGroup);
			if (done[b] || ready[b].cls != ready[a0].cls || total + n >= (1ull << 31)) continue;
			grp.push_back(b);
			total += n;
		}
		uint32_t S = 0;
		bool same_p1 = true;
		for (size_t b : grp) {
			S = std::max(S, items[ready[b].i].scratch->max_slots);
			same_p1 = same_p1 && ready[b].p1 == ready[grp[0]].p1;
		}
		const FrameGeom& g0 = *items[ready[grp[0]].i].g;
		Chunking c;
		const uint32_t npts = ready[grp[0]].tp.npts;
		bool fits = choose_chunking(npts, same_p1 ? ready[grp[0]].p1 : 0, S, c);
		if (!fits) fits = choose_chunking(npts, 0, S, c);
		for (size_t b : grp) done[b] = true;
		if (!fits || grp.size() == 1) {
			for (size_t b : grp) alone.push_back(ready[b].i);
			continue;
		}
		TileBatch B{};
		B.njobs = static_cast<uint32_t>(grp.size());
		uint32_t first = 0;
		std::vector<DasArgs> args;
		for (uint32_t k = 0; k < B.njobs; ++k) {
			const Ready& r = ready[grp[k]];
			const DasBatchItem& it = items[r.i];
			DasArgs a = das_args(*it.g, it.tensor, it.delay, it.w, it.value, it.factor);
			a.partial = it.scratch->partials.as<float2>();
			TileArgs& A = B.jobs[k];
			A = tile_args(*it.g, a, r.tp.ntiles, c);
			A.td = it.scratch->delays.as<const float>();
			A.words = it.scratch->params.as<const uint32_t>();
			A.slots = it.scratch->slots.as<const uint32_t>();
			B.first[k] = first;
			first += r.tp.ntiles * A.ngrp;
			args.push_back(a);
			it.scratch->last_p0 = reported_shape(r.tp, r.p0);
			it.scratch->last_p1 = c.p1(npts, 0);
		}
		B.first[B.njobs] = first;
		B.total = first;
		launch_batch(g0.storage, B, npts, c, s);
		for (uint32_t k = 0; k < B.njobs; ++k) {
			const Ready& r = ready[grp[k]];
			launch_tile_stats(*items[r.i].g, r.tp, args[k], 0, r.tp.ntiles, s);
		}
		++shared;
	}
	for (size_t i : alone) {
		const DasBatchItem& it = items[i];
		launch_das(*it.g, *it.t, *it.scratch, it.tensor, it.delay, it.w, it.value, it.factor, s);
	}
	return shared;
}

// Tail padding of the analytic tensor (bytes): a staged window is copied as
// whole 1 KiB slots from its first entry, so the last channel's copies may
// read up to kMaxSlots KiB past its last sample.
size_t tensor_tail_padding() { return static_cast<size_t>(kMaxSlots) * 1024; }

void launch_das(const FrameGeom& g, const DasTuning& t, DasScratch& scratch, const void* d_tensor,
		const float* d_delay, const float* d_w, float* d_value, float* d_factor, hipStream_t s)
{
	const DasArgs a = das_args(g, d_tensor, d_delay, d_w, d_value, d_factor);

	const bool can_tile = t.variant != 1 && g.L < kMaxWindowL && g.finite_weights;
	if (can_tile) {
		if (t.variant == 2 || t.p0 || t.p1) {
			if (launch_tiled(g, t.p0, t.p1, scratch, a, d_delay, s)) return;
		} else {
			// Autotuner: on the first frame of a geometry, time every
			// candidate tile shape, LDS budget and chunk size (each writes
			// the same images) and keep the fastest for the frames that
			// follow.
			const uint64_t key = g.grid_version ^ (static_cast<uint64_t>(g.L) << 20) ^ (static_cast<uint64_t>(g.ntx) << 40) ^
					(static_cast<uint64_t>(g.nrx) << 50) ^ (static_cast<uint64_t>(g.storage) << 60) ^
					(static_cast<uint64_t>(g.cf_kind) << 62) ^ static_cast<uint64_t>(g.offset * 1024.0f);
			if (scratch.tuned_key != key) {
				// Smaller planes are tried only where no large shape fits,
				// 256-point tiles only where nothing larger than 512 points won.
				const std::vector<int> shapes = tuner_shapes(g);
				hipEvent_t e0 = nullptr, e1 = nullptr;
				HIP_CHECK(hipEventCreate(&e0));
				HIP_CHECK(hipEventCreate(&e1));
				float best = 0.0f;
				int bp0 = -1, bp1 = 0;
				// frames this long are not searched chunking by chunking: once a
				// run takes longer than this, each remaining tile shape gets
				// one timed run of its first fitting configuration
				constexpr float kTuneLimitMs = 150.0f;
				bool long_frame = false;
				int last_p0 = -1;   // shape whose tables are resident
				auto timed = [&](int p0, int p1, float& ms) {
					HIP_CHECK(hipEventRecord(e0, s));
					const bool run = launch_tiled(g, p0, p1, scratch, a, d_delay, s);
					HIP_CHECK(hipEventRecord(e1, s));
					HIP_CHECK(hipEventSynchronize(e1));
					HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
					return run;
				};
				for (int p0 : shapes) {
					const uint32_t npts = tile_plan(g, p0).npts;
					const uint32_t won = bp0 >= 0 ? tile_plan(g, bp0).npts : 0u;
					if (won > 512 && (npts == 256 || (npts == 512 && g.ny <= 1))) continue;
					TileRun held;
					if (!ensure_tables(g, tile_plan(g, p0), scratch, d_delay, s, held)) continue;
					// The smallest LDS budget that fits, which is all that a long
					// frame tries, then pairs per transmit step (4 or 8) in the
					// budgets worth a try.  2048 points: 512 lanes with two
					// workgroups a CU, 1024 lanes with two (4-byte entries: short
					// windows, 100-element BF16 frame 0.66 -> 0.55 ms; 8-byte ones
					// in chunks of two receive elements: 128-element frame 5.76 ->
					// 5.54 ms) or one; where none of them fits, the chunks of two
					// in the whole LDS (192 elements of 65 536 samples 4.14 ms
					// against 5.05 at 32x32).  1024 points: three workgroups a CU
					// where they fit (128-element F16 frame 3.96 -> 3.55 ms, RF
					// 1.03 -> 0.86), else two.
					const int wide = g.storage == MISTA_STORAGE_F32 ? 2 << 24 : 1 << 24;
					std::vector<int> cands = {0};
					if (npts == 2048) cands.insert(cands.end(), {4 | (80 << 16), 4 | (80 << 16) | wide, 8 | (160 << 16)});
					else if (npts == 1024) cands.push_back(4 | (80 << 16));
					else if (npts == 512) cands.push_back(8 | (52 << 16));
					std::vector<Chunking> tried;
					for (const int p1 : cands) {
						Chunking c;
						if (!choose_chunking(npts, p1, scratch.max_slots, c)) continue;
						if (std::any_of(tried.begin(), tried.end(), [&](const Chunking& q) { return q.same(c); })) continue;
						tried.push_back(c);
						// Best of three runs, as the first may find cold caches;
						// of two from 5 ms on, where runs agree within 2 % (the
						// first: 12).  A first run of over 1 ms (shorter ones hold
						// the load of the kernel) that is far enough behind the
						// best ends a chunking, and a shape, whose chunkings differ
						// by up to 1.42.  (256 elements, 512 x 512 points: first
						// frame 176 -> 108 ms.)
						float ms = 0.0f;
						bool run = false;
						for (int rep = 0; rep < (ms > 5.0f ? 2 : 3); ++rep) {
							float t = 0.0f;
							run = timed(p0, p1, t);
							if (!run) break;
							ms = rep == 0 ? t : std::min(ms, t);
							if (t > kTuneLimitMs || (bp0 >= 0 && t > 1.0f && t > 1.15f * best)) break;
						}
						if (!run) continue;
						last_p0 = p0;
						long_frame = long_frame || ms > kTuneLimitMs;
						const bool lost = bp0 >= 0 && ms > 1.0f && ms > 1.5f * best;
						if (bp0 < 0 || ms < best) {
							best = ms;
							bp0 = p0;
							bp1 = p1;
						}
						if (p1 == 0 && (long_frame || lost)) break;
					}
				}
				(void)hipEventDestroy(e0);
				(void)hipEventDestroy(e1);
				scratch.tuned_key = key;
				scratch.tuned_p0 = bp0;
				scratch.tuned_p1 = bp1;
				// every candidate wrote the same images; the winner runs once
				// more only if another shape's tables replaced its own
				if (bp0 >= 0 && (bp0 == last_p0 || launch_tiled(g, bp0, bp1, scratch, a, d_delay, s))) return;
			} else if (scratch.tuned_p0 >= 0 &&
					launch_tiled(g, scratch.tuned_p0, scratch.tuned_p1, scratch, a, d_delay, s)) {
				return;
			}
		}
	}
	scratch.last_p1 = 0;
	// no tile fits (or none was asked for): the rx-parallel form unless the
	// gather kernel was asked for or the per-rx sums would pass 4 GiB
	const size_t pb = static_cast<size_t>(g.nrx) * g.npix * sizeof(float2);   // partial[rx][pixel]
	if (t.variant != 1 && pb > 0 && pb <= (static_cast<size_t>(4) << 30)) {
		DasArgs b = a;
		b.partial = static_cast<float2*>(scratch.partials.reserve(pb));
		if (!b.partial || scratch.partials.capacity() < pb)
			MISTA_THROW(MISTA_E_NO_MEMORY, "no buffer for the per-rx sums (" << pb << " bytes)");
		scratch.last_p0 = -2;
		switch (g.storage) {
		case MISTA_STORAGE_F32: launch_rx_parallel<MISTA_STORAGE_F32>(g, b, s); break;
		case MISTA_STORAGE_F16: launch_rx_parallel<MISTA_STORAGE_F16>(g, b, s); break;
		case kStorageReal: launch_rx_parallel<kStorageReal>(g, b, s); break;
		default: launch_rx_parallel<MISTA_STORAGE_BF16>(g, b, s); break;
		}
		HIP_CHECK(hipGetLastError());
		return;
	}
	scratch.last_p0 = -1;
	launch_gather_any<false>(g, a, s);
}

}  // namespace mista

