// Per-feature-map statistics of a tensor on the device: count, mean, sum of squared deviations
// (double precision), minimum and maximum - the running state of nnForge's stat_data_bunch_writer
// (nnforge/stat_data_bunch_writer.cpp:45-79), which the reference fills on the host, one value at
// a time, from outputs copied back entry by entry.
//
// The reference's update is sequential (Welford). Here every workgroup reduces a run of entries of
// one feature map to (n, mean, m2) and the runs are merged in a fixed order, also in double precision;
// the result does not depend on scheduling.
// Inside a workgroup the sums are taken of (x - pivot), the pivot being the run's first value, so
// that a mean far from zero does not cancel the deviation. mean and m2 agree with the sequential
// update to a few units of double rounding; after the reference's conversion to fp32 that is
// at most one unit in the last place. Minimum and maximum use the reference's comparisons
// (NaN never enters); which of +0.0 / -0.0 is reported when both occur is not defined here.
#include "nnf_common.h"

#include <algorithm>
#include <cstdlib>
#include <mutex>
#include <type_traits>

namespace nnf
{
	namespace
	{
		constexpr int stat_block_size = 256;
		constexpr int stat_unroll = 4;                    // loads a lane has in flight
		// Workgroups of this kernel an MI355X holds at once: 256 compute units x 8 workgroups of 256
		// lanes (up to 64 vector registers: 8 wavefronts per SIMD).
		// The grid is cut so that it fills whole rounds of that many.
		constexpr uint32_t stat_resident_blocks = 2048;
		// what starting and finishing a workgroup costs, in floats of streaming (wavefront and LDS
		// reductions, the partial state)
		constexpr uint64_t stat_block_overhead_floats = 8192;

		// Partial states of nnf_hip_feature_map_stat_accumulate_static: a fixed array in the library's device
		// image instead of a caller's workspace. Every device the library runs on holds its own copy at its own
		// address for the life of the process. In host code the name `scratch` is only a handle for
		// hipGetSymbolAddress, never an address a kernel may be given.
		constexpr size_t stat_static_states = NNF_HIP_STAT_STATIC_SCRATCH_BYTES / sizeof(nnf_hip_running_stat);
		static __device__ __align__(256) unsigned char scratch[NNF_HIP_STAT_STATIC_SCRATCH_BYTES];

		constexpr int stat_max_devices = 64;
		std::mutex scratch_mutex;
		void* scratch_address[stat_max_devices] = {}; // per device, looked up once with that device current

		// address of the current device's copy of `scratch`
		int static_scratch_of_current_device(void** address)
		{
			int device = -1;
			hipError_t e = hipGetDevice(&device);
			if (e != hipSuccess)
				return hip_status(e);
			if ((device < 0) || (device >= stat_max_devices))
				return NNF_HIP_EUNSUPPORTED;
			std::lock_guard<std::mutex> lock(scratch_mutex);
			if (scratch_address[device] == nullptr)
			{
				void* found = nullptr;
				e = hipGetSymbolAddress(&found, HIP_SYMBOL(scratch));
				if (e != hipSuccess)
					return hip_status(e);
				if (found == nullptr)
					return NNF_HIP_EINVAL;
				scratch_address[device] = found;
			}
			*address = scratch_address[device];
			return NNF_HIP_OK;
		}

		struct stat_plan
		{
			uint32_t entries_per_run;
			uint32_t runs;
			uint32_t segments;          // pieces a plane is cut into (> 1 only with one entry per run)
			uint32_t units_per_segment; // in loads
		};

		// Loads (float4s) a plane takes. Planes that are no multiple of four floats start anywhere inside a float4, so this is
		// the most such a plane can touch.
		uint32_t units_of_plane(uint32_t plane)
		{
			return ((plane % 4) == 0) ? plane / 4 : plane / 4 + ((plane % 4 == 1) ? 1 : 2);
		}

		// The grid is (runs of entries) x (feature maps), every workgroup streaming entries_per_run
		// planes. All workgroups take equally long, so the launch lasts
		// ceil(workgroups / resident) rounds of one workgroup's time: the run length that minimises
		// rounds x (run length + overhead) is chosen. Measured on 128 entries of 256 feature maps of
		// 56x56: 6 runs of 22 entries (1536 workgroups, one round) 67.5 us, 13 runs of 10 (3328, two
		// nearly full rounds) 69-71 us, 8 runs of 16 (2048, one round and a seventh of another) 83 us.
		//
		// capacity: partial states the workspace holds; plans that need more are passed over. The longest
		// run the index arithmetic allows gives the fewest partial states, and that number never grows when
		// entries are taken away, so a workspace sized for some entry count holds a plan for every smaller
		// count as well (not necessarily with the same number of runs: 16 entries may be cut into 16 runs
		// where 29 entries were cut into 15). runs == 0 in the result: no plan fits the capacity.
		stat_plan plan_runs(uint32_t entry_count, uint32_t feature_map_count, uint32_t plane, uint64_t capacity)
		{
			// the kernel divides flat indices by the plane size with a multiplication, exact while
			// index * divisor < 2^32; a run of one entry needs no division
			const uint64_t units = units_of_plane(plane);
			stat_plan best = { 1, 0, 1, static_cast<uint32_t>(units) };
			uint64_t best_cost = ~0ull;
			for(uint32_t entries_per_run = 1; entries_per_run <= entry_count; ++entries_per_run)
			{
				if ((entries_per_run > 1) && (static_cast<uint64_t>(entries_per_run) * units * units >= (1ull << 32)))
					break;
				const uint32_t runs = (entry_count + entries_per_run - 1) / entries_per_run;
				const uint64_t blocks = static_cast<uint64_t>(runs) * feature_map_count;
				if (blocks > capacity)
					continue;
				const uint64_t rounds = (blocks + stat_resident_blocks - 1) / stat_resident_blocks;
				const uint64_t cost = rounds * (static_cast<uint64_t>(entries_per_run) * plane + stat_block_overhead_floats);
				if (cost < best_cost)
				{
					best_cost = cost;
					best.entries_per_run = entries_per_run;
					best.runs = runs;
				}
			}
			// Few planes, each long (statistics of input images, say): a plane is cut into segments so that
			// the grid still covers the machine; a segment keeps at least two rounds of loads per lane.
			if (best.runs == 0)
				return best;
			const uint64_t blocks = static_cast<uint64_t>(best.runs) * feature_map_count;
			const uint64_t min_segment_units = static_cast<uint64_t>(stat_block_size) * stat_unroll * 2;
			if ((best.entries_per_run == 1) && (blocks * 2 <= stat_resident_blocks) && (units >= 2 * min_segment_units))
			{
				const uint64_t wanted = std::min<uint64_t>(std::min<uint64_t>(stat_resident_blocks, capacity) / blocks, units / min_segment_units);
				best.units_per_segment = static_cast<uint32_t>((units + wanted - 1) / wanted);
				best.segments = static_cast<uint32_t>((units + best.units_per_segment - 1) / best.units_per_segment);
			}
			return best;
		}

		// The sums a lane keeps. Values are counted relative to the pivot; minimum and maximum go two values at a time through the
		// hardware's three-operand forms, which pass over quiet NaNs - std::min(current, val) / std::max(current, val) never take a
		// NaN val, and current is never NaN - so values are made quiet first.
		struct lane_sums
		{
			double s1 = 0.0, s2 = 0.0;
			float mn = 3.402823466e+38f, mx = -3.402823466e+38f;

			__device__ __forceinline__ void add(floatx4 v, double pivot)
			{
				#pragma unroll
				for(int c = 0; c < 4; ++c)
				{
					const double d = static_cast<double>(v[c]) - pivot;
					s1 += d;
					s2 = fma(d, d, s2);
				}
				#pragma unroll
				for(int c = 0; c < 4; c += 2)
				{
					const float a = __builtin_canonicalizef(v[c]), b = __builtin_canonicalizef(v[c + 1]);
					asm("v_min3_f32 %0, %1, %2, %3" : "=v"(mn) : "v"(mn), "v"(a), "v"(b));
					asm("v_max3_f32 %0, %1, %2, %3" : "=v"(mx) : "v"(mx), "v"(a), "v"(b));
				}
			}
		};

		// over the 16 lanes of a row, the result in all of them; minimum and maximum as the reference compares
		__device__ __forceinline__ double row_sum(double v)
		{
			v += dpp_move<0xB1>(v);
			v += dpp_move<0x4E>(v);
			v += dpp_move<0x141>(v);
			return v + dpp_move<0x140>(v);
		}

		template<int CTRL>
		__device__ __forceinline__ void row_min_max_step(float& mn, float& mx)
		{
			const float other_mn = dpp_move<CTRL>(mn), other_mx = dpp_move<CTRL>(mx);
			mn = (other_mn < mn) ? other_mn : mn;
			mx = (mx < other_mx) ? other_mx : mx;
		}

		__device__ __forceinline__ void row_min_max(float& mn, float& mx)
		{
			row_min_max_step<0xB1>(mn, mx);
			row_min_max_step<0x4E>(mn, mx);
			row_min_max_step<0x141>(mn, mx);
			row_min_max_step<0x140>(mn, mx);
		}

		// grid: (runs x segments, feature maps). Every load is an aligned float4 of the tensor. ALIGNED: planes are multiples of
		// four floats; otherwise a plane starts and ends inside a float4, and what belongs to its neighbours is replaced by
		// the pivot - a value of this feature map, whose deviation is zero. Figures are of the whole call, init and merge launches
		// included: 128 x 192 planes of 35 x 35 29.2 us with a float per load, 25.3 us this way; 20 x 100 of 127 x 127 32.3 -> 26.9 us.
		template<bool ALIGNED>
		__global__ void __launch_bounds__(stat_block_size) stat_runs_kernel(
			nnf_hip_running_stat* partial, const float* in, uint32_t entry_count, uint32_t feature_map_count, uint32_t plane,
			uint32_t entries_per_run, uint32_t units_per_plane, uint32_t unit_magic, uint32_t segments, uint32_t units_per_segment)
		{
			static_assert(stat_block_size == 256, "16 rows of 16 lanes");
			__shared__ double lds_s1[16], lds_s2[16];
			__shared__ float lds_mn[16], lds_mx[16];

			const uint32_t run = blockIdx.x / segments, segment = blockIdx.x - run * segments, fm = blockIdx.y;
			const uint32_t e0 = run * entries_per_run;
			const uint32_t entries_here = min(entries_per_run, entry_count - e0);
			// segments > 1: one entry per run, this workgroup takes a piece of its plane
			const uint32_t unit_begin = segment * units_per_segment;
			const uint32_t units = (segments > 1) ? min(units_per_segment, units_per_plane - unit_begin) : entries_here * units_per_plane;
			const uint32_t entry_stride = feature_map_count * plane;
			const uint32_t total = entry_count * entry_stride; // the tensor has fewer than 2^32 floats
			const uint32_t whole_vectors = total / 4;
			const uint32_t first_plane = (e0 * feature_map_count + fm) * plane; // where the run's first plane starts
			// floats of the plane in front of this segment's, and the segment's
			const uint32_t begin = ALIGNED ? unit_begin * 4 : max(unit_begin * 4, first_plane & 3u) - (first_plane & 3u);
			const uint32_t end = (segments > 1) ? min(plane, (unit_begin + units) * 4 - (ALIGNED ? 0u : first_plane & 3u)) : plane;
			const float pivot_value = in[first_plane + min(begin, plane - 1)];
			const double pivot = static_cast<double>(pivot_value);

			lane_sums sums;
			// COUNT float4s per lane; LAST: the run ends in this round. No lane-dependent branch around a load (with one, every
			// load of a round waited for the one before it): lanes past the end load the run's last float4 and leave it out.
			const auto round = [&](auto count_tag, auto last_tag, uint32_t first)
			{
				constexpr int COUNT = decltype(count_tag)::value;
				constexpr bool LAST = decltype(last_tag)::value;
				floatx4 v[COUNT];
				uint32_t position[ALIGNED ? 1 : COUNT]; // of the float4's first value inside its plane, "negative" in front of it
				#pragma unroll
				for(int k = 0; k < COUNT; ++k)
				{
					const uint32_t mine = first + k * stat_block_size + threadIdx.x;
					const uint32_t t = LAST ? min(mine, units - 1) : mine;
					const uint32_t e = (entries_here == 1) ? 0u : ((units_per_plane == 1) ? t : __umulhi(t, unit_magic));
					const uint32_t in_plane = t - e * units_per_plane + unit_begin;
					const uint32_t start = first_plane + e * entry_stride;
					uint32_t vector = start / 4 + in_plane;
					if (!ALIGNED)
					{
						// the tensor's last float4 may be partial: its values are added below
						position[ALIGNED ? 0 : k] = ((!LAST || (mine < units)) && (vector < whole_vectors)) ? in_plane * 4 - (start & 3u) : plane;
						vector = min(vector, whole_vectors - 1);
					}
					v[k] = load_stream(reinterpret_cast<const floatx4*>(in) + vector);
				}
				#pragma unroll
				for(int k = 0; k < COUNT; ++k)
				{
					if (ALIGNED)
					{
						if (!LAST || (first + k * stat_block_size + threadIdx.x < units))
							sums.add(v[k], pivot);
					}
					else
					{
						const uint32_t at = position[ALIGNED ? 0 : k];
						if (!((at < plane) && (at + 3 < plane)))
						{
							#pragma unroll
							for(int c = 0; c < 4; ++c)
								v[k][c] = (at + c < plane) ? v[k][c] : pivot_value;
						}
						sums.add(v[k], pivot);
					}
				}
			};
			if (ALIGNED || (whole_vectors != 0))
			{
				uint32_t first = 0;
				for(; first + stat_block_size * stat_unroll < units; first += stat_block_size * stat_unroll)
					round(std::integral_constant<int, stat_unroll>(), std::false_type(), first);
				static_assert(stat_unroll == 4, "the last round's cases");
				// as many loads as the rest needs: lanes without a value of their own spend the additions all the same, and the
				// additions in double are a third of a small launch (64 x 512 planes of 7 x 7 10.2 us with rounds of four only, 8.7 us)
				switch ((units - first + stat_block_size - 1) / stat_block_size)
				{
				case 1: round(std::integral_constant<int, 1>(), std::true_type(), first); break;
				case 2: round(std::integral_constant<int, 2>(), std::true_type(), first); break;
				case 3: round(std::integral_constant<int, 3>(), std::true_type(), first); break;
				default: round(std::integral_constant<int, 4>(), std::true_type(), first); break;
				}
			}
			// Up to three values behind the tensor's last whole float4: a lane each, in the workgroup whose run (and segment) they
			// belong to - the last plane's, unless planes are shorter than that.
			if (!ALIGNED && ((total & 3u) != 0) && ((plane < 4) || ((fm + 1 == feature_map_count) && (e0 + entries_here == entry_count))))
			{
				const uint32_t g = whole_vectors * 4 + threadIdx.x;
				const uint32_t g_plane = g / plane, g_entry = g_plane / feature_map_count;
				const bool mine = (g < total) && (g_plane - g_entry * feature_map_count == fm) && (g_entry - e0 < entries_here)
					&& ((segments == 1) || (whole_vectors - first_plane / 4 - unit_begin < units));
				if (mine)
				{
					floatx4 v = {in[g], pivot_value, pivot_value, pivot_value};
					sums.add(v, pivot);
				}
			}
			double s1 = sums.s1, s2 = sums.s2;
			float mn = sums.mn, mx = sums.mx;

			// rows of 16 lanes, then the workgroup
			s1 = row_sum(s1);
			s2 = row_sum(s2);
			row_min_max(mn, mx);
			const uint32_t row = threadIdx.x / 16;
			if ((threadIdx.x % 16) == 0)
			{
				lds_s1[row] = s1; lds_s2[row] = s2; lds_mn[row] = mn; lds_mx[row] = mx;
			}
			__syncthreads();
			if (threadIdx.x < 16)
			{
				s1 = row_sum(lds_s1[threadIdx.x]);
				s2 = row_sum(lds_s2[threadIdx.x]);
				mn = lds_mn[threadIdx.x];
				mx = lds_mx[threadIdx.x];
				row_min_max(mn, mx);
			}
			if (threadIdx.x == 0)
			{
				// the last segment of a plane may lie behind its end: no values
				const double n = (segments > 1) ? static_cast<double>(end - min(begin, end)) : static_cast<double>(entries_here) * static_cast<double>(plane);
				nnf_hip_running_stat r;
				r.n = n;
				r.mean = (n == 0.0) ? pivot : pivot + s1 / n;
				const double m2 = (n == 0.0) ? 0.0 : s2 - s1 * s1 / n;
				r.m2 = (m2 < 0.0) ? 0.0 : m2; // rounding may leave a tiny negative value where the deviation is zero
				r.min_val = mn;
				r.max_val = mx;
				partial[static_cast<size_t>(blockIdx.x) * feature_map_count + fm] = r;
			}
		}

		// A row of 16 lanes per feature map folds the runs into the running state. With m the mean of run 0:
		// mean = m + sum n_k (mean_k - m) / n, then m2 = sum m2_k + n_k (mean_k - mean)^2, the state being one more run; a lane takes
		// runs lane, lane + 16, ..., and the row's sums are combined the same way every time. (One lane per feature map merging run
		// after run, two divisions each: 4.5 us for 10 runs of 192 feature maps, this 2.8 us; 87 x 63 planes of 32 x 32, 33 runs,
		// the whole call 14.2 -> 9.9 us.) The launch is over in the time of its loads and of the instructions it has to fetch.
		constexpr uint32_t stat_merge_lanes = 16;
		__global__ void __launch_bounds__(stat_block_size) stat_merge_kernel(
			nnf_hip_running_stat* state, const nnf_hip_running_stat* partial, uint32_t feature_map_count, uint32_t runs, double values)
		{
			const uint32_t lane = threadIdx.x % stat_merge_lanes;
			const uint32_t fm = (blockIdx.x * stat_block_size + threadIdx.x) / stat_merge_lanes;
			if (fm >= feature_map_count)
				return;
			const nnf_hip_running_stat before = state[fm];
			const nnf_hip_running_stat own = partial[static_cast<size_t>(min(lane, runs - 1)) * feature_map_count + fm]; // most plans have a run a lane at most
			const double m = partial[fm].mean;
			const double own_n = (lane < runs) ? own.n : 0.0;
			double shifted = own_n * (own.mean - m);
			float mn = own.min_val, mx = own.max_val;
			for(uint32_t k = lane + stat_merge_lanes; k < runs; k += stat_merge_lanes)
			{
				const nnf_hip_running_stat r = partial[static_cast<size_t>(k) * feature_map_count + fm];
				shifted += r.n * (r.mean - m);
				mn = (r.min_val < mn) ? r.min_val : mn;
				mx = (mx < r.max_val) ? r.max_val : mx;
			}
			shifted = row_sum(shifted);
			row_min_max(mn, mx);
			const double n = before.n + values;
			const double before_mean = (before.n == 0.0) ? m : before.mean;
			const double mean = m + (shifted + before.n * (before_mean - m)) / n;
			double m2 = (lane < runs) ? own.m2 + own_n * ((own.mean - mean) * (own.mean - mean)) : 0.0;
			for(uint32_t k = lane + stat_merge_lanes; k < runs; k += stat_merge_lanes)
			{
				const nnf_hip_running_stat r = partial[static_cast<size_t>(k) * feature_map_count + fm];
				m2 += r.m2 + r.n * ((r.mean - mean) * (r.mean - mean));
			}
			m2 = row_sum(m2);
			if (lane == 0)
			{
				nnf_hip_running_stat s;
				s.n = n;
				s.mean = mean;
				s.m2 = m2 + (before.m2 + before.n * ((before_mean - mean) * (before_mean - mean)));
				s.min_val = (mn < before.min_val) ? mn : before.min_val;
				s.max_val = (before.max_val < mx) ? mx : before.max_val;
				state[fm] = s;
			}
		}

		__global__ void __launch_bounds__(stat_block_size) stat_init_kernel(nnf_hip_running_stat* state, uint32_t feature_map_count)
		{
			const uint32_t fm = blockIdx.x * stat_block_size + threadIdx.x;
			if (fm >= feature_map_count)
				return;
			// nnforge/stat_data_bunch_writer.h:48-55
			nnf_hip_running_stat s;
			s.n = 0.0;
			s.mean = 0.0;
			s.m2 = 0.0;
			s.min_val = 3.402823466e+38f;
			s.max_val = -3.402823466e+38f;
			state[fm] = s;
		}
	}

	int feature_map_stat_init(hipStream_t stream, nnf_hip_running_stat* device_stats, uint32_t feature_map_count)
	{
		if ((device_stats == nullptr) || (feature_map_count == 0))
			return NNF_HIP_EINVAL;
		if (!is_aligned16(device_stats))
			return NNF_HIP_EALIGN;
		NNF_LAUNCH(stat_init_kernel, dim3((feature_map_count + stat_block_size - 1) / stat_block_size), dim3(stat_block_size), 0, stream,
			device_stats, feature_map_count);
		const int status = launch_status();
		// Set-up of the statistics path on this device: the address of its static scratch array is looked up here,
		// so that nnf_hip_feature_map_stat_accumulate_static finds it ready (a failure is reported there).
		void* unused = nullptr;
		static_scratch_of_current_device(&unused);
		return status;
	}

	int feature_map_stat_workspace_bytes(uint32_t entry_count, uint32_t feature_map_count, uint32_t neuron_count_per_feature_map, size_t* bytes)
	{
		if ((bytes == nullptr) || (feature_map_count == 0) || (neuron_count_per_feature_map == 0))
			return NNF_HIP_EINVAL;
		const stat_plan p = plan_runs(std::max(1u, entry_count), feature_map_count, neuron_count_per_feature_map, ~0ull);
		*bytes = static_cast<size_t>(p.runs) * p.segments * feature_map_count * sizeof(nnf_hip_running_stat);
		return NNF_HIP_OK;
	}

	int feature_map_stat_partial_count(uint32_t entry_count, uint32_t feature_map_count, uint32_t neuron_count_per_feature_map,
		size_t workspace_bytes, uint32_t* partial_states)
	{
		if ((partial_states == nullptr) || (feature_map_count == 0) || (neuron_count_per_feature_map == 0))
			return NNF_HIP_EINVAL;
		*partial_states = 0;
		if (entry_count == 0)
			return NNF_HIP_OK;
		const stat_plan p = plan_runs(entry_count, feature_map_count, neuron_count_per_feature_map, workspace_bytes / sizeof(nnf_hip_running_stat));
		if (p.runs == 0)
			return NNF_HIP_EINVAL;
		*partial_states = p.runs * p.segments * feature_map_count;
		return NNF_HIP_OK;
	}

	namespace
	{
		// argument checks shared by the two accumulate entry points; NNF_HIP_OK with *nothing_to_do set for zero entries
		int check_accumulate_arguments(const nnf_hip_running_stat* device_stats, const float* input,
			uint32_t entry_count, uint32_t feature_map_count, uint32_t neuron_count_per_feature_map, bool* nothing_to_do)
		{
			*nothing_to_do = false;
			if ((device_stats == nullptr) || (feature_map_count == 0) || (neuron_count_per_feature_map == 0))
				return NNF_HIP_EINVAL;
			if (entry_count == 0)
			{
				*nothing_to_do = true; // nothing to fold in
				return NNF_HIP_OK;
			}
			if (input == nullptr)
				return NNF_HIP_EINVAL;
			if (!is_aligned16(device_stats) || !is_aligned16(input))
				return NNF_HIP_EALIGN;
			const uint64_t total = static_cast<uint64_t>(entry_count) * feature_map_count * neuron_count_per_feature_map;
			if ((total > NNF_HIP_MAX_ELEMENT_COUNT) || (feature_map_count > 65535u))
				return NNF_HIP_ETOOBIG;
			return NNF_HIP_OK;
		}

		// the two launches: runs of entries into `partial` (every state of the plan is written, none is read
		// before), then their merge into device_stats
		int launch_accumulate(hipStream_t stream, nnf_hip_running_stat* device_stats, nnf_hip_running_stat* partial, const stat_plan& p,
			const float* input, uint32_t entry_count, uint32_t feature_map_count, uint32_t neuron_count_per_feature_map)
		{
			const dim3 grid(p.runs * p.segments, feature_map_count);
			const uint32_t units = units_of_plane(neuron_count_per_feature_map);
			const uint32_t magic = (units >= 2) ? static_cast<uint32_t>(((1ull << 32) + units - 1) / units) : 0u;
			if ((neuron_count_per_feature_map % 4) == 0)
				NNF_LAUNCH(stat_runs_kernel<true>, grid, dim3(stat_block_size), 0, stream, partial, input, entry_count, feature_map_count,
					neuron_count_per_feature_map, p.entries_per_run, units, magic, p.segments, p.units_per_segment);
			else
				NNF_LAUNCH(stat_runs_kernel<false>, grid, dim3(stat_block_size), 0, stream, partial, input, entry_count, feature_map_count,
					neuron_count_per_feature_map, p.entries_per_run, units, magic, p.segments, p.units_per_segment);
			int status = launch_status();
			if (status != NNF_HIP_OK)
				return status;
			constexpr uint32_t maps_per_block = stat_block_size / stat_merge_lanes;
			NNF_LAUNCH(stat_merge_kernel, dim3((feature_map_count + maps_per_block - 1) / maps_per_block), dim3(stat_block_size), 0, stream,
				device_stats, partial, feature_map_count, p.runs * p.segments, static_cast<double>(entry_count) * neuron_count_per_feature_map);
			return launch_status();
		}
	}

	int feature_map_stat_accumulate(hipStream_t stream, nnf_hip_running_stat* device_stats, void* workspace, size_t workspace_bytes,
		const float* input, uint32_t entry_count, uint32_t feature_map_count, uint32_t neuron_count_per_feature_map)
	{
		bool nothing_to_do = false;
		const int rc = check_accumulate_arguments(device_stats, input, entry_count, feature_map_count, neuron_count_per_feature_map, &nothing_to_do);
		if ((rc != NNF_HIP_OK) || nothing_to_do)
			return rc;
		if (!is_aligned16(workspace))
			return NNF_HIP_EALIGN;
		if (workspace == nullptr)
			return NNF_HIP_EINVAL;
		// the plan is made inside what the workspace holds: a workspace sized for a packet of entries also
		// serves every shorter packet
		const stat_plan p = plan_runs(entry_count, feature_map_count, neuron_count_per_feature_map, workspace_bytes / sizeof(nnf_hip_running_stat));
		if (p.runs == 0)
			return NNF_HIP_EINVAL;
		return launch_accumulate(stream, device_stats, static_cast<nnf_hip_running_stat*>(workspace), p, input, entry_count, feature_map_count,
			neuron_count_per_feature_map);
	}

	int feature_map_stat_accumulate_static(hipStream_t stream, nnf_hip_running_stat* device_stats,
		const float* input, uint32_t entry_count, uint32_t feature_map_count, uint32_t neuron_count_per_feature_map)
	{
		bool nothing_to_do = false;
		const int rc = check_accumulate_arguments(device_stats, input, entry_count, feature_map_count, neuron_count_per_feature_map, &nothing_to_do);
		if ((rc != NNF_HIP_OK) || nothing_to_do)
			return rc;
		// one partial state per feature map is the least any launch shape needs
		if (feature_map_count > stat_static_states)
			return NNF_HIP_ESCRATCH;
		const stat_plan p = plan_runs(entry_count, feature_map_count, neuron_count_per_feature_map, stat_static_states);
		if (p.runs == 0)
			return NNF_HIP_ESCRATCH; // planes so long that the entries cannot share runs, and too many of them
		void* partial = nullptr;
		const int found = static_scratch_of_current_device(&partial);
		if (found != NNF_HIP_OK)
			return found;
		// nothing in the array has to start at zero: the first launch writes every state the second one reads
		return launch_accumulate(stream, device_stats, static_cast<nnf_hip_running_stat*>(partial), p, input, entry_count, feature_map_count,
			neuron_count_per_feature_map);
	}
}
