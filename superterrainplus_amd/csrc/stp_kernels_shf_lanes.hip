// Single histogram filter with one lane per item: the standalone filter's passes for sample maps
// whose filter window holds at most LaneItems distinct items (any 16-bit ids).
//
// The rules are those of stp_stage_shf.hpp (bins in insertion order, the entering line added before
// the leaving one is removed). A group of L = 16, 32 or 64 lanes walks one line; lane q holds the
// window count of the q-th item of the map and its place among the bins. An item whose count leaves
// 0 takes the next place, and one whose count returns to 0 moves the later ones down, which is the
// reference's accumulator (STPSingleHistogramFilter.cpp:400-450) with the search over bins replaced by one
// compare in every lane and the shifts by one ballot. A step costs about 25 VALU instructions for
// 64 / L lines whatever the number of bins; both searches and shifts of the line-per-lane passes
// (singleHistogramFilter) grow with it.
//
// Lines are cut into segments of outputs that run in parallel. The window counts at a segment's
// start are summed afresh; the places there follow from each item's latest run start, a position
// that holds the item with none in the 2r + 1 positions before it: bins lie in the order of (run
// start, place in the column histogram there). Every segment summarises its positions per item (first,
// latest run start inside, last), and a later segment folds the summaries before it.
//
// What bounds it: latency. The 512^2 window of radius 32 with 15 items is 3.3 M wave steps over both
// passes, about 6 us of VALU issue; its bins are 31 MB, 6.5 us at the rate of a large copy. The rest is
// eight dependent launches and segments of at least 64 + 2r dependent steps. Measured there: 20.4 ms
// before (line by line, 8 and 9 waves) and 0.10 ms now (kernels: writing 25 us, vertical 18, counting
// 13, row summaries 9, scan 6, marking 5, ranking 3, clearing 2). Loads behind a bound check of their
// own are waited for one at a time: the loops fetch clamped blocks instead (counting 24 -> 13 us,
// marking 13 -> 5 us).
#include "stp_internal.hpp"

#include <algorithm>

using namespace SuperTerrainPlus;
using namespace SuperTerrainPlus::STPHeightfieldKernel;

namespace {

	typedef unsigned long long Mask;

	constexpr unsigned int LaneBlock = 256u, LaneWaves = LaneBlock / 64u;
	constexpr unsigned int ColumnBlock = 16u;         // columns of one workgroup of the vertical pass
	constexpr unsigned int BitmapWords = 65536u / 32u;
	constexpr unsigned int CountBits = 10u, CountMask = (1u << CountBits) - 1u; // a cell: count | place << 10
	constexpr unsigned int NoItem = 255u;             // no lane's item
	constexpr unsigned int NoPosition = 0xFFFFu;
	static_assert(LaneFilterRadius * 2u + 1u <= CountMask, "a column window's count fits a cell");
	static_assert(LaneItems <= 64u && LaneItems - 1u < (1u << (16u - CountBits)), "a place fits a cell");

	// Run summary of one item over the positions that enter during a segment (NoPosition: none).
	struct Summary {
		unsigned short First, Inner, Last, Pad;
	};

	struct LaneHeader {
		unsigned int Items, Overflow;
	};

	// Everything the kernels share, in the workspace.
	struct LaneArgs {
		const STPSample_t* Window; // first sample of the (map + 2r)^2 window
		unsigned int Pitch, Width, Height, Radius, Columns, Quads; // map, columns = Width + 2r, (columns + 3) / 4
		unsigned int Capacity, ColumnCapacity, Lanes;              // bins per pixel and per column, lanes the workspace holds
		unsigned int SegRows, SegColumns;                           // outputs per segment, vertical and horizontal
		unsigned int Segs;                                          // horizontal segments per row
		unsigned int* Bitmap;
		LaneHeader* Header;
		unsigned char* Id;         // item -> lane, present items only
		unsigned short* Item;      // lane -> item
		Summary *RowSummary, *ColumnSummary;
		unsigned short* Cell;      // [row][column / 4][lane][column % 4]
		unsigned int* Total;       // bins of (row, segment), then the first bin of each
		unsigned int* Offset;
		uint2* Bin;
		float Norm;
	};

	// __ballot takes an int, which costs a select and a compare on a condition
	__device__ inline Mask ballot(const bool v) {
		return __builtin_amdgcn_ballot_w64(v);
	}

	// Lanes per line: the smallest of 16, 32 and 64 that gives every item a lane.
	__device__ inline unsigned int groupLanes(const unsigned int items) {
		return items <= 16u ? 16u : (items <= 32u ? 32u : 64u);
	}

	// One lane's place in its group.
	struct Group {
		unsigned int L, Lane, First; // lanes per group, lane in the group, the group's first lane in the wave
		__device__ explicit Group(const unsigned int lanes) : L(lanes), Lane(threadIdx.x & (lanes - 1u)),
			First((threadIdx.x & 63u) & ~(lanes - 1u)) {}
		// the group's bits of a wave ballot
		__device__ inline Mask bits(const Mask ballot) const {
			return (ballot >> this->First) & (~0ull >> (64u - this->L));
		}
	};

	// The window state of one line: the lane's count and place, the group's number of bins.
	struct LineState {
		unsigned int Count, Place, Bins;
		// lanes whose item was absent and now enters (slot: their order in the entering column)
		__device__ inline void append(const Group& g, const bool fresh, const unsigned int slot) {
			const Mask b = ballot(fresh);
			if (b == 0ull) {
				return; // the whole wave
			}
			const unsigned int lane = g.First + g.Lane;
			unsigned int rank = 0u;
			for (Mask t = b; t != 0ull; t &= t - 1ull) {
				const unsigned int other = static_cast<unsigned int>(__builtin_ctzll(t));
				const unsigned int s = static_cast<unsigned int>(__builtin_amdgcn_readlane(static_cast<int>(slot), static_cast<int>(other)));
				rank += (other & ~(g.L - 1u)) == g.First && s < slot && other != lane ? 1u : 0u;
			}
			if (fresh) {
				this->Place = this->Bins + rank;
			}
			this->Bins += static_cast<unsigned int>(__popcll(g.bits(b)));
		}
		// lanes whose item left the window
		__device__ inline void erase(const Group& g, const bool gone) {
			const Mask b = ballot(gone);
			for (Mask t = b; t != 0ull; t &= t - 1ull) {
				const unsigned int other = static_cast<unsigned int>(__builtin_ctzll(t));
				const unsigned int p = static_cast<unsigned int>(__builtin_amdgcn_readlane(static_cast<int>(this->Place),
					static_cast<int>(other)));
				if ((other & ~(g.L - 1u)) == g.First) {
					this->Place -= this->Place > p ? 1u : 0u;
					this->Bins--;
				}
			}
		}
		// the places of the present items by ascending key (distinct within a group)
		__device__ inline void order(const Group& g, const unsigned int key) {
			const bool present = this->Count > 0u;
			const unsigned int k = present ? key : 0xFFFFFFFFu;
			unsigned int rank = 0u;
#pragma unroll 16
			for (unsigned int j = 0u; j < g.L; j++) {
				rank += static_cast<unsigned int>(__shfl(static_cast<int>(k), static_cast<int>(g.First + j), 64)) < k ? 1u : 0u;
			}
			this->Place = rank;
			this->Bins = static_cast<unsigned int>(__popcll(g.bits(ballot(present))));
		}
	};

	// Latest run start and last occurrence of an item over the positions seen so far.
	struct RunState {
		int Run = -1, Last = -0x40000000;
		__device__ inline void fold(const Summary s, const int window) {
			if (s.First != NoPosition) {
				if (s.Inner != NoPosition) {
					this->Run = s.Inner;
				} else if (static_cast<int>(s.First) - this->Last > window) {
					this->Run = s.First;
				}
				this->Last = s.Last;
			}
		}
		// `count` summaries from `s` on, `step` apart, fetched four at a time
		__device__ inline void fold(const Summary* s, const size_t step, const unsigned int count, const int window) {
			for (unsigned int t = 0u; t < count; t += 4u) {
				Summary v[4];
#pragma unroll
				for (unsigned int k = 0u; k < 4u; k++) {
					v[k] = s[min(t + k, count - 1u) * step];
				}
#pragma unroll
				for (unsigned int k = 0u; k < 4u; k++) {
					if (t + k < count) {
						this->fold(v[k], window);
					}
				}
			}
		}
	};
	// the summary being made
	struct RunSummary {
		// no occurrence yet: later than any position, so that no gap before the first one counts
		unsigned int First = NoPosition, Inner = NoPosition;
		int Last = NoPosition;
		__device__ inline void occur(const bool here, const unsigned int position, const unsigned int window) {
			const bool start = here && static_cast<int>(position) - this->Last > static_cast<int>(window);
			this->Inner = start ? position : this->Inner;
			this->First = min(this->First, here ? position : NoPosition);
			this->Last = here ? static_cast<int>(position) : this->Last;
		}
		__device__ inline Summary pack() const {
			return Summary {static_cast<unsigned short>(this->First), static_cast<unsigned short>(this->Inner),
				static_cast<unsigned short>(this->Last), 0u};
		}
	};

	__global__ void __launch_bounds__(LaneBlock) laneClearKERNEL(const LaneArgs a) {
		const unsigned int i = blockIdx.x * LaneBlock + threadIdx.x;
		if (i < BitmapWords) {
			a.Bitmap[i] = 0u;
		}
		if (i == 0u) {
			a.Header->Items = 0u;
			a.Header->Overflow = 0u;
		}
	}

	// The items of the window: one bit per 16-bit id, gathered per workgroup in LDS.
	constexpr unsigned int MarkRows = 8u; // fetched together
	__global__ void __launch_bounds__(LaneBlock) laneMarkKERNEL(const LaneArgs a) {
		__shared__ unsigned int seen[BitmapWords];
		for (unsigned int i = threadIdx.x; i < BitmapWords; i += LaneBlock) {
			seen[i] = 0u;
		}
		__syncthreads();
		const unsigned int column = blockIdx.x * LaneBlock + threadIdx.x, rows = a.Height + 2u * a.Radius,
			last = min((blockIdx.y + 1u) * MarkRows, rows);
		if (column < a.Columns) {
			unsigned int v[MarkRows];
#pragma unroll
			for (unsigned int k = 0u; k < MarkRows; k++) {
				v[k] = a.Window[static_cast<size_t>(min(blockIdx.y * MarkRows + k, last - 1u)) * a.Pitch + column];
			}
#pragma unroll
			for (unsigned int k = 0u; k < MarkRows; k++) {
				const unsigned int bit = 1u << (v[k] & 31u);
				if ((k == 0u || v[k] != v[k - 1u]) && (seen[v[k] >> 5u] & bit) == 0u) {
					atomicOr(seen + (v[k] >> 5u), bit);
				}
			}
		}
		__syncthreads();
		for (unsigned int i = threadIdx.x; i < BitmapWords; i += LaneBlock) {
			if (seen[i] != 0u) {
				atomicOr(a.Bitmap + i, seen[i]);
			}
		}
	}

	// Numbers the items in ascending order (one workgroup, eight words a thread).
	__global__ void __launch_bounds__(LaneBlock) laneRankKERNEL(const LaneArgs a) {
		constexpr unsigned int Words = BitmapWords / LaneBlock;
		__shared__ unsigned int sum[LaneBlock];
		unsigned int word[Words], n = 0u;
#pragma unroll
		for (unsigned int k = 0u; k < Words; k++) {
			word[k] = a.Bitmap[threadIdx.x * Words + k];
			n += static_cast<unsigned int>(__popc(word[k]));
		}
		sum[threadIdx.x] = n;
		__syncthreads();
		for (unsigned int d = 1u; d < LaneBlock; d <<= 1u) {
			const unsigned int v = threadIdx.x >= d ? sum[threadIdx.x - d] : 0u;
			__syncthreads();
			sum[threadIdx.x] += v;
			__syncthreads();
		}
		const unsigned int items = sum[LaneBlock - 1u];
		if (threadIdx.x == 0u) {
			a.Header->Items = items;
		}
		if (items > a.Lanes) {
			return;
		}
		unsigned int at = sum[threadIdx.x] - n;
#pragma unroll
		for (unsigned int k = 0u; k < Words; k++) {
			for (unsigned int w = word[k]; w != 0u; w &= w - 1u) {
				const unsigned int v = (threadIdx.x * Words + k) * 32u + static_cast<unsigned int>(__ffs(static_cast<int>(w))) - 1u;
				a.Id[v] = static_cast<unsigned char>(at);
				a.Item[at] = static_cast<unsigned short>(v);
				at++;
			}
		}
	}

	// Lane numbers of window rows [row0, row0 + rows) of ColumnBlock columns into LDS, column by column
	// (`stride` bytes each, four rows to a word; NoItem outside the window). row0 may be -4.
	__device__ inline void loadColumns(const LaneArgs& a, const unsigned int column0, const int row0, const unsigned int rows,
		unsigned int* const lds, const unsigned int stride) {
		const unsigned int words = rows / 4u, total = a.Height + 2u * a.Radius;
		for (unsigned int i = threadIdx.x; i < words * ColumnBlock; i += LaneBlock) {
			const unsigned int c = i % ColumnBlock, w = i / ColumnBlock, column = column0 + c;
			// clamped to the window, so that the four samples, then their lanes, are fetched together
			const STPSample_t* const from = a.Window + min(column, a.Columns - 1u);
			unsigned int id[4], packed = 0u;
#pragma unroll
			for (unsigned int k = 0u; k < 4u; k++) {
				const int row = min(max(row0 + static_cast<int>(w * 4u + k), 0), static_cast<int>(total) - 1);
				id[k] = from[static_cast<size_t>(row) * a.Pitch];
			}
#pragma unroll
			for (unsigned int k = 0u; k < 4u; k++) {
				id[k] = a.Id[id[k]];
			}
#pragma unroll
			for (unsigned int k = 0u; k < 4u; k++) {
				const int row = row0 + static_cast<int>(w * 4u + k);
				const bool inside = row >= 0 && row < static_cast<int>(total) && column < a.Columns;
				packed |= (inside ? id[k] : NoItem) << (8u * k);
			}
			lds[c * (stride / 4u) + w] = packed;
		}
		__syncthreads();
	}

	// bytes of one LDS column of `rows` rows: an odd number of words, so that the columns of a wave's
	// groups lie in different banks
	__host__ __device__ inline unsigned int columnStride(const unsigned int rows) {
		return (rows / 4u | 1u) * 4u;
	}
	// rows that loadColumns holds for a vertical segment: four before the first output's window, the
	// window's 2r, and one per output (a multiple of 4)
	__host__ __device__ inline unsigned int segmentRows(const unsigned int outputs, const unsigned int radius) {
		return 4u + 2u * radius + (outputs + 3u) / 4u * 4u;
	}

	// Vertical run summaries: segment s covers the rows that enter during its outputs, [y0 + 2r, y1 + 2r),
	// the first one also the 2r before them. No segment needs the last one's.
	__global__ void __launch_bounds__(LaneBlock) laneRowSummaryKERNEL(const LaneArgs a) {
		extern __shared__ unsigned int lds[];
		const unsigned int items = a.Header->Items;
		if (items > a.Lanes) {
			return;
		}
		const Group g(groupLanes(items));
		const unsigned int seg = blockIdx.y, column0 = blockIdx.x * ColumnBlock, window = 2u * a.Radius + 1u;
		const unsigned int first = seg == 0u ? 0u : seg * a.SegRows + 2u * a.Radius,
			last = (seg + 1u) * a.SegRows + 2u * a.Radius;
		const unsigned int rows = (last - first + 3u) / 4u * 4u, stride = columnStride(rows);
		loadColumns(a, column0, static_cast<int>(first), rows, lds, stride);
		const unsigned int perWave = 64u / g.L, wave = threadIdx.x / 64u;
		for (unsigned int b = 0u; b < ColumnBlock; b += perWave * LaneWaves) {
			const unsigned int c = b + wave * perWave + g.First / g.L;
			if (c >= ColumnBlock) {
				continue;
			}
			const unsigned int* const col = lds + c * (stride / 4u);
			RunSummary sum;
			for (unsigned int w = 0u; w < rows / 4u; w++) {
				const unsigned int packed = col[w];
#pragma unroll
				for (unsigned int k = 0u; k < 4u; k++) {
					sum.occur(((packed >> (8u * k)) & 0xFFu) == g.Lane && first + w * 4u + k < last, first + w * 4u + k, window);
				}
			}
			if (column0 + c < a.Columns) {
				a.RowSummary[(static_cast<size_t>(seg) * a.Columns + column0 + c) * g.L + g.Lane] = sum.pack();
			}
		}
	}

	// Vertical pass: the column histograms of ColumnBlock columns over one segment of rows, as cells.
	__global__ void __launch_bounds__(LaneBlock) laneVerticalKERNEL(const LaneArgs a) {
		extern __shared__ unsigned int lds[];
		const unsigned int items = a.Header->Items;
		if (items > a.Lanes) {
			return;
		}
		const Group g(groupLanes(items));
		const unsigned int seg = blockIdx.y, column0 = blockIdx.x * ColumnBlock, twice = 2u * a.Radius;
		const unsigned int y0 = seg * a.SegRows, y1 = min(y0 + a.SegRows, a.Height);
		const unsigned int rows = segmentRows(y1 - y0, a.Radius), stride = columnStride(rows);
		// LDS row i is window row y0 - 4 + i
		loadColumns(a, column0, static_cast<int>(y0) - 4, rows, lds, stride);
		const unsigned int perWave = 64u / g.L, wave = threadIdx.x / 64u;
		unsigned int most = 0u;
		// c is the same on every lane of a group, and `b` on every lane of the workgroup
		for (unsigned int b = 0u; b < ColumnBlock; b += perWave * LaneWaves) {
			const unsigned int c = b + wave * perWave + g.First / g.L, column = column0 + c;
			if (b + wave * perWave >= ColumnBlock) {
				continue; // the whole wave
			}
			const unsigned int* const col = lds + c * (stride / 4u);
			const bool stored = column < a.Columns;
			// the window before the first output: rows [y0 - 1, y0 + 2r), without row -1
			LineState line {0u, 0u, 0u};
			RunState run;
			unsigned int first = 0xFFFFu;
			line.Count = (col[0] >> 24u) == g.Lane ? 1u : 0u;
			for (unsigned int w = 0u; w < twice / 4u; w++) {
				const unsigned int packed = col[1u + w];
#pragma unroll
				for (unsigned int k = 0u; k < 4u; k++) {
					const bool here = ((packed >> (8u * k)) & 0xFFu) == g.Lane;
					line.Count += here ? 1u : 0u;
					first = here ? min(first, w * 4u + k) : first;
				}
			}
			if (seg == 0u) {
				// nothing before: every item's first occurrence is its run start
				run.Run = static_cast<int>(first);
			} else {
				run.fold(a.RowSummary + static_cast<size_t>(min(column, a.Columns - 1u)) * g.L + g.Lane,
					static_cast<size_t>(a.Columns) * g.L, seg, static_cast<int>(twice + 1u));
			}
			line.order(g, static_cast<unsigned int>(run.Run));
			most = max(most, line.Bins);
			unsigned int before = col[0];
			unsigned short* cell = a.Cell + ((static_cast<size_t>(y0) * a.Quads + column / 4u) * g.L + g.Lane) * 4u + column % 4u;
			const size_t pitch = static_cast<size_t>(a.Quads) * g.L * 4u;
			const auto step = [&](const unsigned int in4, const unsigned int out4, const unsigned int k) {
				const bool in = ((in4 >> (8u * k)) & 0xFFu) == g.Lane, out = ((out4 >> (8u * k)) & 0xFFu) == g.Lane;
				const bool fresh = in && line.Count == 0u;
				line.Count += in ? 1u : 0u;
				line.append(g, fresh, 0u);
				// as the line-by-line pass: an item that enters a full column before another leaves it
				most = max(most, line.Bins);
				line.Count -= out ? 1u : 0u;
				line.erase(g, out && line.Count == 0u);
				if (stored) {
					*cell = static_cast<unsigned short>(line.Count > 0u ? line.Count | (line.Place << CountBits) : 0u);
				}
				cell += pitch;
			};
			for (unsigned int y = y0; y < y1; y += 4u) {
				const unsigned int enter = col[1u + (y - y0 + twice) / 4u], next = col[1u + (y - y0) / 4u],
					leave = (next << 8u) | (before >> 24u);
				before = next;
				if (y + 4u <= y1) {
#pragma unroll
					for (unsigned int k = 0u; k < 4u; k++) {
						step(enter, leave, k);
					}
				} else {
					for (unsigned int k = 0u; y + k < y1; k++) {
						step(enter, leave, k);
					}
				}
			}
		}
		if (most > a.ColumnCapacity) {
			atomicOr(&a.Header->Overflow, 1u);
		}
	}

	// One lane's cells of a row: quads of four columns. The loops fetch Ahead quads before the first is
	// used; a bound on every quad would let the compiler move each load behind it.
	constexpr unsigned int Ahead = 4u;
	struct RowCells {
		const uint2* Line;
		unsigned int Stride;
		__device__ RowCells(const LaneArgs& a, const Group& g, const unsigned int row) :
			Line(reinterpret_cast<const uint2*>(a.Cell) + static_cast<size_t>(row) * a.Quads * g.L + g.Lane), Stride(g.L) {}
		__device__ inline uint2 quad(const unsigned int q) const { return this->Line[static_cast<size_t>(q) * this->Stride]; }
		__device__ static inline unsigned int part(const uint2 v, const unsigned int k) {
			return ((k & 2u ? v.y : v.x) >> (16u * (k & 1u))) & 0xFFFFu;
		}
		// f(cell, position) for the columns of quads [q, last)
		template <class F>
		__device__ inline void each(unsigned int q, const unsigned int last, F&& f) const {
			for (; q + Ahead <= last; q += Ahead) {
				uint2 v[Ahead];
#pragma unroll
				for (unsigned int j = 0u; j < Ahead; j++) {
					v[j] = this->quad(q + j);
				}
#pragma unroll
				for (unsigned int i = 0u; i < Ahead * 4u; i++) {
					f(part(v[i / 4u], i % 4u), q * 4u + i);
				}
			}
			for (; q < last; q++) {
				const uint2 v = this->quad(q);
#pragma unroll
				for (unsigned int k = 0u; k < 4u; k++) {
					f(part(v, k), q * 4u + k);
				}
			}
		}
		// f(x, entering cell, leaving cell) for the outputs [x0, x1), x0 a multiple of 4: column x + 2r
		// enters and x - 1 leaves (`left` for the first)
		template <class F>
		__device__ inline void walk(const unsigned int x0, const unsigned int x1, const unsigned int radius, const unsigned int left,
			F&& f) const {
			const unsigned int shift = radius / 2u, lastQuad = (x1 - 1u) / 4u; // 2r columns
			unsigned int q = x0 / 4u, out = left;
			uint2 e[Ahead], l[Ahead];
			// quads past the last are the last again
			const auto fetch = [&](uint2 (&en)[Ahead], uint2 (&ln)[Ahead], const unsigned int first) {
#pragma unroll
				for (unsigned int j = 0u; j < Ahead; j++) {
					en[j] = this->quad(min(first + j, lastQuad) + shift);
					ln[j] = this->quad(min(first + j, lastQuad));
				}
			};
			fetch(e, l, q);
			for (; (q + Ahead) * 4u <= x1; q += Ahead) {
				uint2 en[Ahead], ln[Ahead];
				fetch(en, ln, q + Ahead);
#pragma unroll
				for (unsigned int i = 0u; i < Ahead * 4u; i++) {
					f(q * 4u + i, part(e[i / 4u], i % 4u), i == 0u ? out : part(l[(i - 1u) / 4u], (i - 1u) % 4u));
				}
				out = part(l[Ahead - 1u], 3u);
#pragma unroll
				for (unsigned int j = 0u; j < Ahead; j++) {
					e[j] = en[j];
					l[j] = ln[j];
				}
			}
			for (; q <= lastQuad; q++) {
				const uint2 ve = this->quad(q + shift), vl = this->quad(q);
#pragma unroll
				for (unsigned int k = 0u; k < 4u; k++) {
					if (q * 4u + k < x1) {
						f(q * 4u + k, part(ve, k), k == 0u ? out : part(vl, k - 1u));
					}
				}
				out = part(vl, 3u);
			}
		}
	};

	// Row and segment of a group: consecutive rows of one segment share a wave.
	struct RowTask {
		unsigned int Row, X0, X1, Seg;
		bool Valid;
		__device__ RowTask(const LaneArgs& a, const Group& g) {
			const unsigned int groups = LaneBlock / g.L;
			this->Seg = blockIdx.y;
			this->X0 = this->Seg * a.SegColumns;
			this->X1 = min(this->X0 + a.SegColumns, a.Width);
			const unsigned int row = blockIdx.x * groups + threadIdx.x / g.L;
			this->Valid = row < a.Height;
			this->Row = min(row, a.Height - 1u);
		}
	};

	// Horizontal counting pass: bins of every (row, segment), the capacity test, and the run summaries
	// of the columns that enter during the segment (the first one also has the 2r before them).
	__global__ void __launch_bounds__(LaneBlock) laneCountKERNEL(const LaneArgs a) {
		const unsigned int items = a.Header->Items;
		if (items > a.Lanes) {
			return;
		}
		const Group g(groupLanes(items));
		if (blockIdx.x * (LaneBlock / g.L) >= a.Height) {
			return; // the grid is sized for 64 lanes per line
		}
		const RowTask t(a, g);
		const unsigned int window = 2u * a.Radius + 1u;
		const RowCells cells(a, g, t.Row);
		const unsigned int quad0 = t.X0 / 4u, quads = a.Radius / 2u;
		// the window before the first output: columns [x0 - 1, x0 + 2r), without column -1
		const unsigned int left = t.Seg == 0u ? 0u : RowCells::part(cells.quad(quad0 - 1u), 3u);
		unsigned int count = left & CountMask, total = 0u;
		RunSummary sum;
		if (t.Seg == 0u) {
			cells.each(quad0, quad0 + quads, [&](const unsigned int cell, const unsigned int position) {
				count += cell & CountMask;
				sum.occur((cell & CountMask) > 0u, position, window);
			});
		} else {
			cells.each(quad0, quad0 + quads, [&](const unsigned int cell, unsigned int) { count += cell & CountMask; });
		}
		unsigned int most = static_cast<unsigned int>(__popcll(g.bits(ballot(count > 0u))));
		cells.walk(t.X0, t.X1, a.Radius, left, [&](const unsigned int x, const unsigned int in, const unsigned int out) {
			const unsigned int n = in & CountMask;
			const bool fresh = n > 0u && count == 0u;
			count += n;
			sum.occur(n > 0u, x + 2u * a.Radius, window);
			// as the line-by-line pass: the entering column is added before the leaving one goes
			if (ballot(fresh) != 0ull) {
				most = max(most, static_cast<unsigned int>(__popcll(g.bits(ballot(count > 0u)))));
			}
			count -= out & CountMask;
			total += count > 0u ? 1u : 0u;
		});
		for (unsigned int d = 1u; d < g.L; d <<= 1u) {
			total += static_cast<unsigned int>(__shfl_xor(static_cast<int>(total), static_cast<int>(d), 64));
		}
		if (t.Valid) {
			if (g.Lane == 0u) {
				a.Total[static_cast<size_t>(t.Row) * a.Segs + t.Seg] = total;
			}
			a.ColumnSummary[(static_cast<size_t>(t.Seg) * a.Height + t.Row) * g.L + g.Lane] = sum.pack();
		}
		if (most > a.Capacity) {
			atomicOr(&a.Header->Overflow, 1u);
		}
	}

	// First bin of every (row, segment), in place; the bin total and the flags for the host.
	constexpr unsigned int ScanThreads = 1024u;
	__global__ void __launch_bounds__(ScanThreads) laneScanKERNEL(const LaneArgs a, STPLaneFilterReport* const report) {
		__shared__ unsigned int sum[ScanThreads / 64u];
		const unsigned int n = a.Height * a.Segs, items = a.Header->Items, lane = threadIdx.x & 63u, wave = threadIdx.x / 64u;
		unsigned int carry = 0u;
		if (items <= a.Lanes) {
			for (unsigned int base = 0u; base < n; base += ScanThreads) {
				const unsigned int i = base + threadIdx.x, v = i < n ? a.Total[i] : 0u;
				unsigned int inc = v;
#pragma unroll
				for (unsigned int d = 1u; d < 64u; d <<= 1u) {
					const unsigned int o = __shfl_up(inc, d, 64);
					inc += lane >= d ? o : 0u;
				}
				if (lane == 63u) {
					sum[wave] = inc;
				}
				__syncthreads();
				unsigned int add = carry;
				for (unsigned int w = 0u; w < ScanThreads / 64u; w++) {
					add += w < wave ? sum[w] : 0u;
					carry += sum[w];
				}
				if (i < n) {
					a.Total[i] = add + inc - v;
				}
				__syncthreads();
			}
		}
		if (threadIdx.x == 0u) {
			a.Offset[static_cast<size_t>(a.Width) * a.Height] = carry;
			report->Held = items <= a.Lanes ? 1u : 0u;
			report->Overflow = a.Header->Overflow;
			report->Bins = carry;
		}
	}

	// Horizontal writing pass: every pixel's bins in order, and its first bin.
	__global__ void __launch_bounds__(LaneBlock) laneWriteKERNEL(const LaneArgs a) {
		const unsigned int items = a.Header->Items;
		// more bins than the capacity would leave the output array
		if (items > a.Lanes || a.Header->Overflow != 0u) {
			return;
		}
		const Group g(groupLanes(items));
		if (blockIdx.x * (LaneBlock / g.L) >= a.Height) {
			return;
		}
		const RowTask t(a, g);
		const unsigned int window = 2u * a.Radius + 1u;
		const RowCells cells(a, g, t.Row);
		const unsigned int quad0 = t.X0 / 4u, quads = a.Radius / 2u;
		const unsigned int left = t.Seg == 0u ? 0u : RowCells::part(cells.quad(quad0 - 1u), 3u);
		LineState line {left & CountMask, 0u, 0u};
		int start = static_cast<int>(NoPosition);
		if (t.Seg == 0u) {
			// nothing before: every item's first occurrence is its run start
			cells.each(quad0, quad0 + quads, [&](const unsigned int cell, const unsigned int position) {
				line.Count += cell & CountMask;
				start = min(start, (cell & CountMask) > 0u ? static_cast<int>(position) : static_cast<int>(NoPosition));
			});
		} else {
			cells.each(quad0, quad0 + quads, [&](const unsigned int cell, unsigned int) { line.Count += cell & CountMask; });
			RunState run;
			run.fold(a.ColumnSummary + static_cast<size_t>(t.Row) * g.L + g.Lane, static_cast<size_t>(a.Height) * g.L, t.Seg,
				static_cast<int>(window));
			start = run.Run;
		}
		// bins lie by (run start, place in the column histogram there)
		unsigned int key = 0u;
		if (line.Count > 0u) {
			const unsigned int c = static_cast<unsigned int>(start);
			key = (c << 6u) | (RowCells::part(cells.quad(c / 4u), c % 4u) >> CountBits);
		}
		line.order(g, key);
		unsigned int at = a.Total[static_cast<size_t>(t.Row) * a.Segs + t.Seg], kept = 0u;
		const unsigned int item = g.Lane < items ? a.Item[g.Lane] : 0u;
		unsigned int* const offset = a.Offset + static_cast<size_t>(t.Row) * a.Width;
		cells.walk(t.X0, t.X1, a.Radius, left, [&](const unsigned int x, const unsigned int in, const unsigned int out) {
			const unsigned int n = in & CountMask;
			const bool fresh = n > 0u && line.Count == 0u;
			line.Count += n;
			line.append(g, fresh, in >> CountBits);
			line.Count -= out & CountMask;
			line.erase(g, (out & CountMask) > 0u && line.Count == 0u);
			if (line.Count > 0u && t.Valid) {
				a.Bin[at + line.Place] = make_uint2(item, __float_as_uint(static_cast<float>(line.Count) * a.Norm));
			}
			// lane j keeps the offset of the j-th of L pixels, stored together
			const unsigned int j = (x - t.X0) & (g.L - 1u);
			kept = j == g.Lane ? at : kept;
			if ((j == g.L - 1u || x + 1u == t.X1) && g.Lane <= j && t.Valid) {
				offset[x - j + g.Lane] = kept;
			}
			at += line.Bins;
		});
	}

	inline size_t align256(const size_t v) {
		return (v + 255u) & ~static_cast<size_t>(255u);
	}

	// Outputs per segment: 64, the most segments that pay for the 2r positions each sums afresh,
	// doubled while the lines alone keep the chip busy and while the window is much longer.
	unsigned int segmentLength(const unsigned int lines, const unsigned int outputs, const unsigned int radius) {
		unsigned int s = 64u;
		while (s < 512u && (s < radius || static_cast<unsigned long long>(lines) * ((outputs + s - 1u) / s) >= 65536ull)) {
			s *= 2u;
		}
		return s;
	}

	// Lanes the workspace holds per line: 64 while the cells take at most a gigabyte (8 M pixels), on
	// larger maps twice the bin capacity (the items of a whole map are often more than those of one window),
	// from 16 to 64. A map of more items is found out on the device and goes line by line after all: 32^2 with
	// 24 items takes 51 us here, 145 line by line, and took 181 where the workspace held 16 lanes.
	constexpr size_t LaneCellBytes = 1ull << 30u;
	unsigned int workspaceLanes(const uint2 map, const unsigned int quads, const unsigned int bin_capacity) {
		const size_t cells = static_cast<size_t>(map.y) * quads * 4u * sizeof(unsigned short);
		return cells * LaneItems <= LaneCellBytes ? LaneItems
			: (bin_capacity <= 8u ? 16u : (bin_capacity <= 16u ? 32u : LaneItems));
	}

	// Places in the workspace; fills every field but the sample map's.
	size_t carve(char* const base, const uint2 map, const unsigned int radius, const unsigned int cap, LaneArgs& a) {
		size_t at = 0u;
		const auto take = [&](const size_t bytes) {
			char* const here = base + at;
			at += align256(bytes);
			return here;
		};
		a.Width = map.x;
		a.Height = map.y;
		a.Radius = radius;
		a.Columns = map.x + 2u * radius;
		a.Quads = (a.Columns + 3u) / 4u;
		a.Capacity = cap;
		a.ColumnCapacity = cap < 2u * radius + 1u ? cap : 2u * radius + 1u;
		a.Lanes = workspaceLanes(map, a.Quads, cap);
		a.SegRows = segmentLength(a.Columns, map.y, radius);
		a.SegColumns = segmentLength(map.y, map.x, radius);
		a.Segs = (map.x + a.SegColumns - 1u) / a.SegColumns;
		const unsigned int rowSegs = (map.y + a.SegRows - 1u) / a.SegRows;
		const size_t pixels = static_cast<size_t>(map.x) * map.y;
		a.Bitmap = reinterpret_cast<unsigned int*>(take(BitmapWords * sizeof(unsigned int)));
		a.Header = reinterpret_cast<LaneHeader*>(take(sizeof(LaneHeader)));
		a.Id = reinterpret_cast<unsigned char*>(take(65536u));
		a.Item = reinterpret_cast<unsigned short*>(take(LaneItems * sizeof(unsigned short)));
		static_assert(BitmapWords * sizeof(unsigned int) + 65536u + 512u == LaneItemBytes && sizeof(LaneHeader) <= 256u
			&& LaneItems * sizeof(unsigned short) <= 256u, "the numbered items come first");
		a.RowSummary = reinterpret_cast<Summary*>(take(static_cast<size_t>(rowSegs) * a.Columns * a.Lanes * sizeof(Summary)));
		a.ColumnSummary = reinterpret_cast<Summary*>(take(static_cast<size_t>(a.Segs) * map.y * a.Lanes * sizeof(Summary)));
		a.Cell = reinterpret_cast<unsigned short*>(take(static_cast<size_t>(map.y) * a.Quads * 4u * a.Lanes * sizeof(unsigned short)));
		a.Total = reinterpret_cast<unsigned int*>(take(static_cast<size_t>(map.y) * a.Segs * sizeof(unsigned int)));
		a.Offset = reinterpret_cast<unsigned int*>(take((pixels + 1u) * sizeof(unsigned int)));
		a.Bin = reinterpret_cast<uint2*>(take(pixels * cap * sizeof(uint2)));
		const unsigned int w = 2u * radius + 1u;
		a.Norm = 1.0f / static_cast<float>(w * w);
		return at;
	}

} // namespace

size_t STPHeightfieldKernel::laneFilterBytes(const uint2 map_size, const unsigned int radius, const unsigned int bin_capacity) {
	LaneArgs a {};
	return carve(nullptr, map_size, radius, bin_capacity, a);
}

bool STPHeightfieldKernel::laneFilterApplies(const uint2 map_size, const unsigned int radius, const unsigned int bin_capacity) {
	// Positions (and window counts) of a line in 16 bits; grids of at most 65535 segments. A workspace beyond
	// 64 GiB is only taken where the line-by-line passes take as much (bin capacities of 1 to 3 take less).
	return radius <= LaneFilterRadius && map_size.x + 2ull * radius < NoPosition && map_size.y + 2ull * radius < NoPosition
		&& laneFilterBytes(map_size, radius, bin_capacity)
			<= std::max<size_t>(64ull << 30u, filterWorkspaceBytes(map_size, radius, bin_capacity));
}

namespace {
	LaneArgs laneArguments(const STPSample_t* const sample, const unsigned int pitch, const uint2 start, const uint2 map_size,
		const unsigned int radius, const unsigned int bin_capacity, void* const workspace) {
		STP_ASSERT_DOMAIN(radius > 0u && (radius & 1u) == 0u, "radius should be an positive even number");
		STP_ASSERT_DOMAIN(radius <= start.x && radius <= start.y,
			"radius is too large and will overflow nearest neighbour boundary");
		if (bin_capacity == 0u || bin_capacity > MaxBinCapacity) {
			STP_THROW(STPInvalidArgument, "histogram bin capacity must be in [1, 64]");
		}
		if (!sample || map_size.x == 0u || map_size.y == 0u || !workspace || !laneFilterApplies(map_size, radius, bin_capacity)) {
			STP_THROW(STPInvalidArgument, "invalid sample map");
		}
		LaneArgs a {};
		carve(static_cast<char*>(workspace), map_size, radius, bin_capacity, a);
		a.Window = sample + static_cast<size_t>(start.y - radius) * pitch + (start.x - radius);
		a.Pitch = pitch;
		return a;
	}

	__global__ void laneReportKERNEL(const LaneArgs a, STPLaneFilterReport* const report) {
		report->Held = a.Header->Items <= a.Lanes ? 1u : 0u;
	}
} // namespace

void STPHeightfieldKernel::laneFilterItems(const STPSample_t* const sample, const unsigned int pitch, const uint2 start,
	const uint2 map_size, const unsigned int radius, const unsigned int bin_capacity, void* const workspace,
	const hipStream_t stream) {
	const LaneArgs a = laneArguments(sample, pitch, start, map_size, radius, bin_capacity, workspace);
	laneClearKERNEL<<<(BitmapWords + LaneBlock - 1u) / LaneBlock, LaneBlock, 0, stream>>>(a);
	laneMarkKERNEL<<<dim3((a.Columns + LaneBlock - 1u) / LaneBlock, (a.Height + 2u * radius + MarkRows - 1u) / MarkRows), LaneBlock, 0,
		stream>>>(a);
	laneRankKERNEL<<<1, LaneBlock, 0, stream>>>(a);
	STP_CHECK_HIP(hipGetLastError());
}

void STPHeightfieldKernel::laneFilterReport(const uint2 map_size, const unsigned int radius, const unsigned int bin_capacity,
	const void* const workspace, STPLaneFilterReport* const report, const hipStream_t stream) {
	LaneArgs a {};
	carve(const_cast<char*>(static_cast<const char*>(workspace)), map_size, radius, bin_capacity, a);
	laneReportKERNEL<<<1, 1, 0, stream>>>(a, report);
	STP_CHECK_HIP(hipGetLastError());
}

STPAlgorithm::STPSingleHistogram STPHeightfieldKernel::laneFilter(const STPSample_t* const sample, const unsigned int pitch,
	const uint2 start, const uint2 map_size, const unsigned int radius, const unsigned int bin_capacity, void* const workspace,
	STPLaneFilterReport* const report, const hipStream_t stream) {
	if (!report) {
		STP_THROW(STPInvalidArgument, "null report");
	}
	laneFilterItems(sample, pitch, start, map_size, radius, bin_capacity, workspace, stream);
	const LaneArgs a = laneArguments(sample, pitch, start, map_size, radius, bin_capacity, workspace);
	const unsigned int rowSegs = (a.Height + a.SegRows - 1u) / a.SegRows, columnBlocks = (a.Columns + ColumnBlock - 1u) / ColumnBlock;
	if (rowSegs > 1u) {
		// segment 0 also holds the 2r rows before its first output
		const unsigned int bytes = columnStride((a.SegRows + 2u * radius + 3u) / 4u * 4u) * ColumnBlock;
		laneRowSummaryKERNEL<<<dim3(columnBlocks, rowSegs - 1u), LaneBlock, bytes, stream>>>(a);
	}
	laneVerticalKERNEL<<<dim3(columnBlocks, rowSegs), LaneBlock,
		columnStride(segmentRows(a.SegRows, radius)) * ColumnBlock, stream>>>(a);
	const dim3 rows((a.Height + LaneWaves - 1u) / LaneWaves, a.Segs);
	laneCountKERNEL<<<rows, LaneBlock, 0, stream>>>(a);
	laneScanKERNEL<<<1, ScanThreads, 0, stream>>>(a, report);
	laneWriteKERNEL<<<rows, LaneBlock, 0, stream>>>(a);
	STP_CHECK_HIP(hipGetLastError());
	return STPAlgorithm::STPSingleHistogram {reinterpret_cast<const STPAlgorithm::STPSingleHistogram::STPBin*>(a.Bin), a.Offset};
}
