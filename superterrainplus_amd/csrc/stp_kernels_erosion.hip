// Free-slip particle hydraulic erosion and FP32 -> UINT16 formatting (per-chunk launches).
//
// Behaviour follows SuperTerrain+/SuperTerrain+/Private/GPGPU/STPHeightfieldKernel.cu:80-122
// and SuperTerrain+/SuperTerrain+/Private/GPGPU/STPRainDrop.cu:18-164 (drop logic in
// stp_stage_erosion.hpp).
//
// MI355X design:
//  * Parallel mode: one lane per drop. Heights are read with relaxed agent-scope atomic loads,
//    which bypass the per-CU vector L1, so a drop sees other CUs' updates as soon as L2 has
//    them (the reference's plain loads can hit a stale L1 line). Updates are hardware FP32
//    atomic adds executed at L2 (no CAS loop). The brush (index, weight) is staged in LDS and
//    read with a wave-uniform address, i.e. an LDS broadcast; the heights under the brush are
//    fetched in one group before the atomics are issued.
//  * Serialized mode: one wavefront walks the drops in index order; all lanes carry the same
//    drop state, the brush taps are spread over the lanes, and the sediment sum is taken in tap
//    order with lane reads, so the result is bit-exact against the FP32 oracle.
//  Roofline: L2 atomics + dependent-latency chains; per drop-step the algorithmic traffic is
//  32 B of height reads, plus 25 x (4 B read + 8 B atomic) for an erode step at r = 3, or
//  4 x 8 B atomics for a deposit step.
#include "stp_stage_erosion.hpp"

using namespace SuperTerrainPlus;
using namespace SuperTerrainPlus::STPStage;

namespace {

	constexpr unsigned int ParallelBlock = 256u;

	__global__ void __launch_bounds__(ParallelBlock) erosionParallelKERNEL(float* const map, const ErosionArgs a,
		const int* const brush_index, const float* const brush_weight, float* const ledger, uint2* const drop_info,
		const unsigned int* const gate) {
		extern __shared__ int2 brush[]; // (index, weight bits)
		if (gate && (gate[0] | gate[1]) == 0u) {
			// another path eroded the map: the whole grid leaves at once
			return;
		}
		for (unsigned int k = threadIdx.x; k < a.BrushSize; k += blockDim.x) {
			brush[k] = make_int2(brush_index[k], __float_as_int(brush_weight[k]));
		}
		__syncthreads();
		const unsigned int drop = blockIdx.x * blockDim.x + threadIdx.x;
		if (drop < a.Rain.RainDropCount) {
			erodeDropAnyBrush(GlobalSurface {map, a.Total.x}, a, brush, drop, drop, ledger, drop_info);
		}
	}

	constexpr unsigned int SerialLanes = 64u;

	__global__ void __launch_bounds__(SerialLanes) erosionSerialKERNEL(float* const map, const ErosionArgs a,
		const int* const brush_index, const float* const brush_weight, float* const ledger, uint2* const drop_info,
		const unsigned int* const gate) {
		if (gate && *gate == 0u) {
			return; // other work eroded the map
		}
		const unsigned int lane = threadIdx.x;
		const unsigned int W = a.Total.x;
		for (unsigned int drop = 0u; drop < a.Rain.RainDropCount; drop++) {
			DropState d = spawn(a, drop);
			float lost = 0.0f;
			unsigned int steps = 0u, erodeSteps = 0u, depositSteps = 0u, killed = 0u;
			if (!spawnInside(a, d)) {
				d.volume = DeadVolume;
				killed = 1u;
			}
			for (unsigned int life = 0u; alive(a, d, life); life++) {
				steps++;
				const unsigned int cellX = static_cast<unsigned int>(d.px), cellY = static_cast<unsigned int>(d.py);
				const unsigned int mapIndex = cellY * W + cellX;
				const float ox = d.px - static_cast<float>(static_cast<int>(d.px)),
					oy = d.py - static_cast<float>(static_cast<int>(d.py));
				float3 hg;
				if (!moveDrop<false>(a, map, d, hg) || !cellInside(a, cellX, cellY)) {
					lost = d.sediment;
					d.volume = 0.0f;
					d.sediment = 0.0f;
					killed = 1u;
					break;
				}
				const float deltaHeight = heightGradient<false>(map, W, d.px, d.py).x - hg.x;
				const float cap = fmaxf(-deltaHeight * d.speed * d.volume * a.Rain.SedimentCapacityFactor,
					a.Rain.minSedimentCapacity);
				if (d.sediment > cap || deltaHeight > 0.0f) {
					const float amount = (deltaHeight > 0.0f) ? fminf(deltaHeight, d.sediment)
															  : (d.sediment - cap) * a.Rain.DepositSpeed;
					d.sediment -= amount;
					// four distinct cells, one lane each
					if (lane < 4u) {
						const unsigned int cell = mapIndex + (lane & 1u) + ((lane >> 1) ? W : 0u);
						const float fx = (lane & 1u) ? ox : (1.0f - ox), fy = (lane >> 1) ? oy : (1.0f - oy);
						map[cell] = map[cell] + amount * fx * fy;
					}
					depositSteps++;
				} else {
					const float amount = fminf((cap - d.sediment) * a.Rain.ErodeSpeed, -deltaHeight);
					for (unsigned int base = 0u; base < a.BrushSize; base += SerialLanes) {
						const unsigned int k = base + lane;
						float ds = 0.0f;
						if (k < a.BrushSize) {
							const unsigned int ei = mapIndex + static_cast<unsigned int>(brush_index[k]);
							const float wa = amount * brush_weight[k];
							const float h = map[ei];
							ds = (h < wa) ? h : wa;
							map[ei] = h - ds;
						}
						const unsigned int group = min(SerialLanes, a.BrushSize - base);
						for (unsigned int j = 0u; j < group; j++) {
							d.sediment += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ds), j));
						}
					}
					erodeSteps++;
				}
				// make this step's writes visible to every lane before the next read
				__syncthreads();
				advance(a, d, deltaHeight);
			}
			if (lane == 0u) {
				if (ledger) {
					ledger[drop] = lost + d.sediment;
				}
				if (drop_info) {
					drop_info[drop] = packDropInfo(steps, erodeSteps, depositSteps, killed);
				}
			}
		}
	}

	// ---- ordered erosion: the serialized drops, many at a time
	//
	// The serialized mode's result is that of the drops run one after another in index order. A drop
	// touches only cells near its path, so a later drop may run while earlier ones are still on their way
	// as long as none of them can reach what it touches: unit steps move a drop at most one cell, and an
	// earlier drop with n steps left stays within n cells of where it is. Every wave takes the next drop
	// (in index order), runs it OrderedSteps steps at a time on a copy of its surroundings in LDS, writes
	// back the cells it changed and publishes its cell and the steps it has left; before each such chunk it
	// waits until every earlier unfinished drop is too far away to touch the chunk's cells. What is read
	// is then exactly what the earlier drops left, and what is written nobody earlier will read: the
	// same sums in the same order, bit for bit.
	//
	// Every wait ends: drops are taken in index order by waves that are already running, a drop waits
	// for lower indices only, and the lowest unfinished one waits for nobody. A wave that still
	// polls after `poll_limit` rounds raises the stop word, on which every wave leaves; the
	// serialized kernel then erodes the saved map.
	//
	// What bounds it: the chain of drops in each other's way, each link a poll, a window load, the
	// chunk's steps and the write-back. Longer chunks have fewer of these but wait for more distance.
	// Measured on a 512^2 map with 8192 drops of 30 steps: one wave alone (1 us a step, four dependent
	// trips to memory) 251 ms; here 6.8 ms with chunks of 4 steps, 7.0 with 3 or 6, 8.1 with 8, 8.8 with
	// 10. A loop over the brush's sums instead of straight-line code took 8.8 ms with chunks of 6.
	constexpr unsigned int OrderedWaves = 128u; // a chain is never wider: 128 to 1024 waves model the same
	constexpr unsigned int OrderedSteps = 4u;   // steps of one chunk
	constexpr unsigned int OrderedList = 2u * OrderedWaves;
	constexpr unsigned int OrderedLifetime = 256u, OrderedRadius = 16u;
	// taps of the radius-16 brush (dx^2 + dy^2 < 256)
	constexpr unsigned int OrderedTaps = 800u;

	struct OrderedHeader {
		unsigned int Ticket, Stop;
	};
	typedef unsigned long long DropWord; // steps left << 32 | cell y << 16 | cell x; 0 steps left: finished

	__device__ inline DropWord dropWord(const unsigned int left, const unsigned int x, const unsigned int y) {
		return (static_cast<DropWord>(left) << 32u) | (y << 16u) | x;
	}
	// Chebyshev distance of a drop's cell from (x, y)
	__device__ inline int cellDistance(const DropWord w, const int x, const int y) {
		return max(abs(static_cast<int>(w & 0xFFFFu) - x), abs(static_cast<int>((w >> 16u) & 0xFFFFu) - y));
	}
	template <class T>
	__device__ inline T agentLoad(const T* const p) {
		return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	}
	template <class T>
	__device__ inline void agentStore(T* const p, const T v) {
		__hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	}

	// whether the drop takes a step at all
	__device__ inline bool orderedStarts(const ErosionArgs& a, const DropState& d) {
		return spawnInside(a, d) && alive(a, d, 0u);
	}

	__global__ void __launch_bounds__(256) orderedSpawnKERNEL(const ErosionArgs a, DropWord* const word, OrderedHeader* const header) {
		const unsigned int drop = blockIdx.x * 256u + threadIdx.x;
		if (drop == 0u) {
			header->Ticket = 0u;
			header->Stop = 0u;
		}
		if (drop < a.Rain.RainDropCount) {
			const DropState d = spawn(a, drop);
			word[drop] = orderedStarts(a, d) ? dropWord(a.Rain.MaxLifetime, static_cast<unsigned int>(d.px), static_cast<unsigned int>(d.py))
											: 0ull;
		}
	}

	// Cells a drop touches beyond the steps it takes: its brush r - 1 around the cells it leaves, and the
	// 2 x 2 cell it arrives at, whose corner may lie one further than the steps (their fractions add up).
	__host__ __device__ inline unsigned int orderedReach(const unsigned int radius) {
		return radius > 3u ? radius - 1u : 2u;
	}
	// Window of a chunk: its steps start within OrderedSteps of the centre, and one step may cross two
	// cell borders when a direction rounds above 1.
	__host__ __device__ inline unsigned int orderedWindow(const unsigned int radius) {
		return 2u * (OrderedSteps + (radius > 4u ? radius - 1u : 3u)) + 1u;
	}
	constexpr unsigned int OrderedFetch = 8u; // window cells a lane fetches at once

	// d + v of lanes 0 .. Taps - 1, in lane order
	template <unsigned int Taps>
	__device__ inline float addLanes(float d, const float v) {
#pragma unroll
		for (unsigned int j = 0u; j < Taps; j++) {
			d += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), j));
		}
		return d;
	}

	// Taps: the brush size (9, 25 or 45: its sums are straight-line code), or 0 for any
	template <unsigned int Taps>
	__global__ void __launch_bounds__(64) orderedErosionKERNEL(float* const map, const ErosionArgs a, const int* const brush_index,
		const float* const brush_weight, DropWord* const word, OrderedHeader* const header, const unsigned int poll_limit) {
		extern __shared__ float window[]; // side x side, the same as fetched, the taps' offsets and weights
		__shared__ unsigned int before[OrderedList];
		const unsigned int lane = threadIdx.x, r = a.Rain.ErosionBrushRadius, reach = orderedReach(r);
		const int side = static_cast<int>(orderedWindow(r)), half = side / 2, cells = side * side;
		float* const fetched = window + cells;
		int* const tap = reinterpret_cast<int*>(fetched + cells);
		float* const weight = reinterpret_cast<float*>(tap + a.BrushSize);
		const int W = static_cast<int>(a.Total.x), H = static_cast<int>(a.Total.y);
		for (unsigned int k = lane; k < a.BrushSize; k += 64u) {
			// the map's linear offset dy * W + dx, |dx| < r < W / 2
			const int shifted = brush_index[k] + static_cast<int>(r) * W + W / 2, dy = shifted / W - static_cast<int>(r),
				dx = shifted % W - W / 2;
			tap[k] = dy * side + dx;
			weight[k] = brush_weight[k];
		}
		__syncthreads();
		unsigned int low = 0u; // every drop below it has finished
		for (;;) {
			unsigned int drop = 0u;
			if (lane == 0u) {
				drop = __hip_atomic_fetch_add(&header->Ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			}
			drop = static_cast<unsigned int>(__builtin_amdgcn_readfirstlane(static_cast<int>(drop)));
			if (drop >= a.Rain.RainDropCount) {
				return;
			}
			DropState d = spawn(a, drop);
			if (!orderedStarts(a, d)) {
				continue; // published as finished from the start
			}
			// The earlier drops that could ever be in this one's way. Each unfinished one is held by
			// another wave, and a finished one may be seen late: more than the list holds are read again.
			const int spawnX = static_cast<int>(d.px), spawnY = static_cast<int>(d.py);
			const int margin = 2 * static_cast<int>(reach) + 1;
			unsigned int waiting = 0u, firstOpen = drop;
			do {
				waiting = 0u;
				firstOpen = drop;
				for (unsigned int base = low; base < drop; base += 64u) {
					const unsigned int i = base + lane;
					const DropWord w = i < drop ? agentLoad(word + i) : 0ull;
					const int left = static_cast<int>(w >> 32u);
					const int distance = cellDistance(w, spawnX, spawnY);
					const unsigned long long open = __builtin_amdgcn_ballot_w64(left > 0);
					if (open != 0ull && firstOpen == drop) {
						firstOpen = base + static_cast<unsigned int>(__builtin_ctzll(open));
					}
					const bool near = left > 0 && distance <= left + static_cast<int>(a.Rain.MaxLifetime) + margin;
					const unsigned long long b = __builtin_amdgcn_ballot_w64(near);
					const unsigned int at = waiting + static_cast<unsigned int>(__popcll(b & ((1ull << lane) - 1ull)));
					if (near && at < OrderedList) {
						before[at] = i;
					}
					waiting += static_cast<unsigned int>(__popcll(b));
				}
			} while (waiting > OrderedList);
			low = firstOpen;
			__syncthreads();

			bool dead = false;
			for (unsigned int life = 0u; !dead && alive(a, d, life);) {
				const int centreX = static_cast<int>(d.px), centreY = static_cast<int>(d.py);
				const unsigned int steps = min(OrderedSteps, a.Rain.MaxLifetime - life);
				// wait until no earlier drop can still touch the chunk's cells
				for (unsigned int poll = 0u;; poll++) {
					unsigned int kept = 0u;
					bool blocked = false;
					for (unsigned int base = 0u; base < waiting; base += 64u) {
						const unsigned int i = base + lane < waiting ? before[base + lane] : 0u;
						const DropWord w = base + lane < waiting ? agentLoad(word + i) : 0ull;
						const int left = static_cast<int>(w >> 32u);
						blocked = blocked || (left > 0 && cellDistance(w, centreX, centreY) <= left + static_cast<int>(steps) + margin);
						const unsigned long long b = __builtin_amdgcn_ballot_w64(left > 0);
						__syncthreads(); // every lane has read its entry
						if (left > 0) {
							before[kept + static_cast<unsigned int>(__popcll(b & ((1ull << lane) - 1ull)))] = i;
						}
						kept += static_cast<unsigned int>(__popcll(b));
						__syncthreads();
					}
					waiting = kept;
					if (__builtin_amdgcn_ballot_w64(blocked) == 0ull) {
						break;
					}
					if (agentLoad(&header->Stop) != 0u || poll >= poll_limit) {
						agentStore(&header->Stop, 1u);
						return;
					}
					__builtin_amdgcn_s_sleep(1);
				}
				__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");

				// the window, clamped to the map (cells outside are never used); lane cells step by 64 cells
				// of the row-major window
				const int startY = static_cast<int>(lane) / side, startX = static_cast<int>(lane) - startY * side;
				for (int c = static_cast<int>(lane), x = startX, y = startY; c - static_cast<int>(lane) < cells;) {
					float v[OrderedFetch];
#pragma unroll
					for (unsigned int k = 0u; k < OrderedFetch; k++) {
						const int mx = min(max(centreX - half + x, 0), W - 1), my = min(max(centreY - half + y, 0), H - 1);
						v[k] = agentLoad(map + static_cast<size_t>(my) * W + mx);
						x += 64 % side;
						y += 64 / side + (x >= side ? 1 : 0);
						x -= x >= side ? side : 0;
					}
#pragma unroll
					for (unsigned int k = 0u; k < OrderedFetch; k++) {
						if (c < cells) {
							window[c] = v[k];
							fetched[c] = v[k];
						}
						c += 64;
					}
				}
				__syncthreads();
				const int originX = centreX - half, originY = centreY - half;
				const auto gradient = [&](const int x, const int y, const float px, const float py) {
					const float* const p = window + (y - originY) * side + (x - originX);
					return cornerGradient(p[0], p[1], p[side], p[side + 1], px - static_cast<float>(x), py - static_cast<float>(y));
				};
				for (unsigned int s = 0u; s < steps && alive(a, d, life); s++) {
					const int cellX = static_cast<int>(d.px), cellY = static_cast<int>(d.py);
					if (max(abs(cellX - centreX), abs(cellY - centreY)) > static_cast<int>(OrderedSteps)) {
						break; // a new window
					}
					life++;
					const float ox = d.px - static_cast<float>(cellX), oy = d.py - static_cast<float>(cellY);
					const float3 hg = gradient(cellX, cellY, d.px, d.py);
					if (!moveDropAlong(a, d, hg) || !cellInside(a, static_cast<unsigned int>(cellX), static_cast<unsigned int>(cellY))) {
						dead = true;
						break;
					}
					const float deltaHeight = gradient(static_cast<int>(d.px), static_cast<int>(d.py), d.px, d.py).x - hg.x;
					const float cap = fmaxf(-deltaHeight * d.speed * d.volume * a.Rain.SedimentCapacityFactor,
						a.Rain.minSedimentCapacity);
					float* const here = window + (cellY - originY) * side + (cellX - originX);
					if (d.sediment > cap || deltaHeight > 0.0f) {
						const float amount = (deltaHeight > 0.0f) ? fminf(deltaHeight, d.sediment)
																  : (d.sediment - cap) * a.Rain.DepositSpeed;
						d.sediment -= amount;
						if (lane < 4u) {
							float* const p = here + (lane & 1u) + ((lane >> 1) ? side : 0);
							const float fx = (lane & 1u) ? ox : (1.0f - ox), fy = (lane >> 1) ? oy : (1.0f - oy);
							*p = *p + amount * fx * fy;
						}
					} else {
						const float amount = fminf((cap - d.sediment) * a.Rain.ErodeSpeed, -deltaHeight);
						const auto take = [&](const unsigned int k) {
							float* const p = here + tap[k];
							const float wa = amount * weight[k];
							const float h = *p;
							const float ds = (h < wa) ? h : wa;
							*p = h - ds;
							return ds;
						};
						if constexpr (Taps > 0u) {
							d.sediment = addLanes<Taps>(d.sediment, lane < Taps ? take(lane) : 0.0f);
						} else {
							for (unsigned int base = 0u; base < a.BrushSize; base += 64u) {
								const float ds = base + lane < a.BrushSize ? take(base + lane) : 0.0f;
								const unsigned int group = min(64u, a.BrushSize - base);
								for (unsigned int j = 0u; j < group; j++) {
									d.sediment += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ds), j));
								}
							}
						}
					}
					// this step's writes before the next step's reads
					__syncthreads();
					advance(a, d, deltaHeight);
				}
				// changed cells back to the map, then the progress
				__syncthreads();
				for (int c = static_cast<int>(lane), x = startX, y = startY; c < cells; c += 64) {
					const float v = window[c];
					if (__float_as_uint(v) != __float_as_uint(fetched[c])) {
						agentStore(map + static_cast<size_t>(originY + y) * W + (originX + x), v);
					}
					x += 64 % side;
					y += 64 / side + (x >= side ? 1 : 0);
					x -= x >= side ? side : 0;
				}
				__builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
				__syncthreads();
				if (lane == 0u) {
					const bool more = !dead && alive(a, d, life);
					agentStore(word + drop, more ? dropWord(a.Rain.MaxLifetime - life, static_cast<unsigned int>(d.px),
						static_cast<unsigned int>(d.py)) : 0ull);
				}
			}
		}
	}

	__global__ void __launch_bounds__(256) orderedRestoreKERNEL(const OrderedHeader* const header, const float* const saved,
		float* const map, const unsigned long long count) {
		if (header->Stop == 0u) {
			return;
		}
		const unsigned long long i = static_cast<unsigned long long>(blockIdx.x) * 256u + threadIdx.x;
		if (i < count) {
			map[i] = saved[i];
		}
	}

	__global__ void __launch_bounds__(256) formatKERNEL(const float* const input, STPHeightFixed_t* const output,
		const unsigned long long count) {
		const unsigned long long i4 = (static_cast<unsigned long long>(blockIdx.x) * blockDim.x + threadIdx.x) * 4ull;
		if (i4 + 4ull <= count) {
			const float4 h = *reinterpret_cast<const float4*>(input + i4);
			ushort4 o;
			o.x = toFixed(h.x);
			o.y = toFixed(h.y);
			o.z = toFixed(h.z);
			o.w = toFixed(h.w);
			*reinterpret_cast<ushort4*>(output + i4) = o;
		} else {
			for (unsigned long long i = i4; i < count; i++) {
				output[i] = toFixed(input[i]);
			}
		}
	}

	// gate words: [0] a height out of range, [1] a status word copied from other work
	__global__ void gateClearKERNEL(unsigned int* const gate) {
		gate[0] = 0u;
		gate[1] = 0u;
	}

	constexpr unsigned int GateBlock = 256u, GateItems = 16u;

	__global__ void __launch_bounds__(GateBlock) heightGateKERNEL(const float* const map, const unsigned long long count,
		const float low, const float high, unsigned int* const gate) {
		const unsigned long long first = static_cast<unsigned long long>(blockIdx.x) * GateBlock * GateItems + threadIdx.x;
		bool out = false;
#pragma unroll
		for (unsigned int k = 0u; k < GateItems; k++) {
			const unsigned long long i = first + static_cast<unsigned long long>(k) * GateBlock;
			if (i < count) {
				const float h = map[i];
				// NaN fails both comparisons
				out = out || !(h >= low && h <= high);
			}
		}
		if (__any(out) && (threadIdx.x & 63u) == 0u) {
			atomicOr(gate, 1u);
		}
	}

	__global__ void gateStatusKERNEL(const unsigned int* const status, unsigned int* const gate) { gate[1] = *status; }

	__global__ void __launch_bounds__(256) selectUngatedKERNEL(const unsigned int* const gate, const float* const source,
		float* const map, const unsigned long long count) {
		if ((gate[0] | gate[1]) != 0u) {
			return;
		}
		const unsigned long long i = static_cast<unsigned long long>(blockIdx.x) * blockDim.x + threadIdx.x;
		if (i < count) {
			map[i] = source[i];
		}
	}

} // namespace

void STPHeightfieldKernel::heightGate(const float* const map, const unsigned long long count, const float low,
	const float high, unsigned int* const gate, const hipStream_t stream) {
	if (!map || !gate) {
		STP_THROW(STPInvalidArgument, "height gate needs a map and a gate");
	}
	gateClearKERNEL<<<1, 1, 0, stream>>>(gate);
	const unsigned long long per = static_cast<unsigned long long>(GateBlock) * GateItems;
	if (count != 0ull) {
		heightGateKERNEL<<<static_cast<unsigned int>((count + per - 1ull) / per), GateBlock, 0, stream>>>(map, count, low, high,
			gate);
	}
	STP_CHECK_HIP(hipGetLastError());
}

void STPHeightfieldKernel::copyGateStatus(const unsigned int* const status, unsigned int* const gate, const hipStream_t stream) {
	if (!status || !gate) {
		STP_THROW(STPInvalidArgument, "gate status needs a status word and a gate");
	}
	gateStatusKERNEL<<<1, 1, 0, stream>>>(status, gate);
	STP_CHECK_HIP(hipGetLastError());
}

void STPHeightfieldKernel::selectUngated(const unsigned int* const gate, const float* const source, float* const map,
	const unsigned long long count, const hipStream_t stream) {
	if (!gate || !source || !map) {
		STP_THROW(STPInvalidArgument, "select needs a gate, a source and a map");
	}
	if (count != 0ull) {
		selectUngatedKERNEL<<<static_cast<unsigned int>((count + 255ull) / 256ull), 256, 0, stream>>>(gate, source, map, count);
	}
	STP_CHECK_HIP(hipGetLastError());
}

namespace {
	// Arguments of an erosion of the whole merged map, after the checks every mode shares.
	ErosionArgs erosionArguments(const float* const height, const STPNearestNeighbourInformation& nn, const STPRainDropParameter& rd,
		const int* const brush_index, const float* const brush_weight, const unsigned int brush_size, const unsigned int stream_id) {
		if (!height || !brush_index || !brush_weight || brush_size == 0u) {
			STP_THROW(STPInvalidArgument, "erosion needs a heightmap and a non-empty brush");
		}
		if (nn.TotalMapSize.x != nn.MapSize.x * nn.ChunkNearestNeighbour.x
			|| nn.TotalMapSize.y != nn.MapSize.y * nn.ChunkNearestNeighbour.y || nn.MapSize.x < 2u || nn.MapSize.y < 2u) {
			STP_THROW(STPInvalidArgument, "inconsistent nearest-neighbour information");
		}
		const unsigned int r = rd.ErosionBrushRadius;
		if (r == 0u || 2u * r + 2u > nn.TotalMapSize.x || 2u * r + 2u > nn.TotalMapSize.y) {
			STP_THROW(STPInvalidArgument, "brush radius does not fit the merged map");
		}
		ErosionArgs a;
		a.Rain = rd;
		a.MapSize = nn.MapSize;
		a.SpawnOrigin = make_uint2((nn.ChunkNearestNeighbour.x / 2u) * nn.MapSize.x, (nn.ChunkNearestNeighbour.y / 2u) * nn.MapSize.y);
		a.Total = nn.TotalMapSize;
		a.BrushSize = brush_size;
		a.StreamId = stream_id;
		return a;
	}
} // namespace

void STPHeightfieldKernel::hydraulicErosion(float* const height, const STPNearestNeighbourInformation& nn,
	const STPRainDropParameter& rd, const int* const brush_index, const float* const brush_weight,
	const unsigned int brush_size, const unsigned int stream_id, const STPErosionMode mode, float* const ledger,
	uint2* const drop_info, const hipStream_t stream, const unsigned int* const gate) {
	const ErosionArgs a = erosionArguments(height, nn, rd, brush_index, brush_weight, brush_size, stream_id);
	if (rd.RainDropCount == 0u) {
		return;
	}
	if (mode == STPErosionMode::Parallel) {
		const unsigned int grid = (rd.RainDropCount + ParallelBlock - 1u) / ParallelBlock;
		erosionParallelKERNEL<<<grid, ParallelBlock, brush_size * sizeof(int2), stream>>>(height, a, brush_index,
			brush_weight, ledger, drop_info, gate);
	} else {
		if (gate) {
			STP_THROW(STPInvalidArgument, "a gated erosion is parallel");
		}
		erosionSerialKERNEL<<<1, SerialLanes, 0, stream>>>(height, a, brush_index, brush_weight, ledger, drop_info, nullptr);
	}
	STP_CHECK_HIP(hipGetLastError());
}

namespace {
	// places in the workspace: header, a word per drop, the saved map
	constexpr size_t OrderedWordAt = 256u;
	inline size_t orderedSavedAt(const unsigned int drops) {
		return (OrderedWordAt + drops * sizeof(DropWord) + 255u) & ~static_cast<size_t>(255u);
	}
} // namespace

bool STPHeightfieldKernel::orderedErosionApplies(const STPNearestNeighbourInformation& nn, const STPRainDropParameter& rd) noexcept {
	// without a lifetime every drop could reach everywhere; a drop's cell is published in 16 bits
	return rd.RainDropCount > 1u && rd.MaxLifetime > 0u && rd.MaxLifetime <= OrderedLifetime && rd.ErosionBrushRadius <= OrderedRadius
		&& nn.TotalMapSize.x <= 65535u && nn.TotalMapSize.y <= 65535u;
}

size_t STPHeightfieldKernel::orderedErosionBytes(const STPNearestNeighbourInformation& nn, const STPRainDropParameter& rd) {
	return orderedSavedAt(rd.RainDropCount) + static_cast<size_t>(nn.TotalMapSize.x) * nn.TotalMapSize.y * sizeof(float);
}

bool STPHeightfieldKernel::orderedErosionGaveUp(const void* const workspace, const hipStream_t stream) {
	OrderedHeader header;
	STP_CHECK_HIP(hipMemcpyAsync(&header, workspace, sizeof(header), hipMemcpyDeviceToHost, stream));
	STP_CHECK_HIP(hipStreamSynchronize(stream));
	return header.Stop != 0u;
}

void STPHeightfieldKernel::orderedErosion(float* const height, const STPNearestNeighbourInformation& nn,
	const STPRainDropParameter& rd, const int* const brush_index, const float* const brush_weight, const unsigned int brush_size,
	const unsigned int stream_id, void* const workspace, const hipStream_t stream, const unsigned int poll_limit) {
	const ErosionArgs a = erosionArguments(height, nn, rd, brush_index, brush_weight, brush_size, stream_id);
	if (!workspace || !orderedErosionApplies(nn, rd) || brush_size > OrderedTaps) {
		STP_THROW(STPInvalidArgument, "the ordered erosion does not take this map, brush or lifetime");
	}
	char* const base = static_cast<char*>(workspace);
	auto* const header = reinterpret_cast<OrderedHeader*>(base);
	auto* const word = reinterpret_cast<DropWord*>(base + OrderedWordAt);
	auto* const saved = reinterpret_cast<float*>(base + orderedSavedAt(rd.RainDropCount));
	const unsigned long long count = static_cast<unsigned long long>(nn.TotalMapSize.x) * nn.TotalMapSize.y;
	STP_CHECK_HIP(hipMemcpyAsync(saved, height, count * sizeof(float), hipMemcpyDeviceToDevice, stream));
	orderedSpawnKERNEL<<<(rd.RainDropCount + 255u) / 256u, 256, 0, stream>>>(a, word, header);
	const unsigned int side = orderedWindow(rd.ErosionBrushRadius),
		lds = 2u * (side * side + brush_size) * static_cast<unsigned int>(sizeof(float));
	const auto run = [&](auto kernel) {
		kernel<<<rd.RainDropCount < OrderedWaves ? rd.RainDropCount : OrderedWaves, 64, lds, stream>>>(height, a, brush_index,
			brush_weight, word, header, poll_limit);
	};
	switch (brush_size) {
	case 9u: run(orderedErosionKERNEL<9u>); break;
	case 25u: run(orderedErosionKERNEL<25u>); break;
	case 45u: run(orderedErosionKERNEL<45u>); break;
	default: run(orderedErosionKERNEL<0u>); break;
	}
	orderedRestoreKERNEL<<<static_cast<unsigned int>((count + 255ull) / 256ull), 256, 0, stream>>>(header, saved, height, count);
	erosionSerialKERNEL<<<1, SerialLanes, 0, stream>>>(height, a, brush_index, brush_weight, nullptr, nullptr, &header->Stop);
	STP_CHECK_HIP(hipGetLastError());
}

void STPHeightfieldKernel::formatHeightmap(const float* const input, STPHeightFixed_t* const output,
	const unsigned long long count, const hipStream_t stream) {
	if (count == 0ull) {
		return;
	}
	if (!input || !output) {
		STP_THROW(STPInvalidArgument, "format needs input and output");
	}
	if ((reinterpret_cast<uintptr_t>(input) & 15u) != 0u || (reinterpret_cast<uintptr_t>(output) & 7u) != 0u) {
		STP_THROW(STPInvalidArgument, "format needs 16-byte aligned input and 8-byte aligned output");
	}
	const unsigned long long threads = (count + 3ull) / 4ull;
	formatKERNEL<<<static_cast<unsigned int>((threads + 255ull) / 256ull), 256u, 0, stream>>>(input, output, count);
	STP_CHECK_HIP(hipGetLastError());
}
