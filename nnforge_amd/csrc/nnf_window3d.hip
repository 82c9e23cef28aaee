// Maximum, minimum or sum over 3-D windows (subsampling of volumes), staged through LDS. The plain testers' loop over
// the window (nnforge/plain/max_subsampling_layer_tester_plain.cpp:175-290,
// nnforge/plain/average_subsampling_layer_tester_plain.cpp:34-148) is folded in its order where the order shows
// (nnf_window.h), so the results are the reference's bit for bit.
//
// A volume is one feature map of one entry. A workgroup produces a block of outputs: `slices` output slices of `rows` output
// rows of one volume, or all of several small volumes. The input that takes is one run of memory when the rows are whole
// slices (or whole volumes), and otherwise one run per input slice; it is copied to LDS with aligned float4 loads, eight in
// flight per lane, and every lane scans its windows there. What bounds the kernel is memory: each input value is fetched once,
// plus what neighbouring blocks share (windows wider than their stride). One lane per output reading its window from
// memory (window_nd_kernel, which keeps what does not fit here) runs at the rate its uncoalesced 4-byte loads leave: 2 x 2 x 2
// every 2 on 16 x 64 volumes of 28^3 (101 MB) 34.8 us there, 17.4 us here (5.8 TB/s); 8 x 34 of 53^3 56.4 -> 30.5 us;
// 3 x 3 x 3 every 2 on 4 x 40 of 64^3 121.9 -> 35.2 us, on 60 x 256 of 14^3 119.2 -> 39.8 us; 1 x 77 of 40^3 (22 MB) 9.0 -> 6.0 us.
#include "nnf_common.h"
#include "nnf_window.h"

#include <algorithm>

namespace nnf
{
	namespace
	{
		struct window3d_args
		{
			float* out;
			const float* in;
			uint32_t total_in;                       // floats in the input tensor
			uint32_t plane_count;                    // entries * feature maps
			uint32_t in_w, in_h, in_d, out_w, out_h, out_d;
			uint32_t win_w, win_h, win_d, stride_x, stride_y, stride_z;
			uint32_t planes;                         // volumes per workgroup (1 when a volume is split)
			uint32_t slices, rows;                   // output slices and rows per workgroup
			uint32_t slice_bands, row_bands;         // ceil(out_d / slices), ceil(out_h / rows)
			uint32_t run_vectors;                    // row_bands > 1: float4s in LDS per input slice
			uint32_t run_vectors_magic;
			uint32_t units_w, units_w_magic;         // a lane's units of work per output row (outputs, or pairs of them)
			uint32_t rows_magic, last_rows_magic;    // rows of a band, of the last band
			uint32_t slices_magic;
			uint32_t together;                       // blocks of a volume that share input: to one XCD (0: none do)
			float mult;                              // window_op_sum: the sum is multiplied by it
		};

		constexpr int stage3d_vectors_per_lane = 8;

		// WIN: 2 or 3 = windows of that size in every dimension, 0: the sizes are in the arguments.
		// TRUNC: windows may reach beyond the input (round up): a position beyond reads the last one inside again, which
		// was folded before and changes nothing.
		// PAIR (WIN 2 or 3, every 2 columns, rows of whole float4s, an even number of outputs per row: the host checks): a
		// lane takes two neighbouring outputs; the four columns both windows start in are one aligned 16-byte LDS read.
		template<int OP, int WIN, bool TRUNC, bool PAIR>
		__global__ void __launch_bounds__(max_block_size) window3d_kernel(const window3d_args a)
		{
			static_assert(!PAIR || (WIN > 0), "pairs of outputs: window size known");
			static_assert(!(TRUNC && (OP == window_op_sum)), "a truncated window re-reads values");
			extern __shared__ __align__(16) float lds_in[];

			const uint32_t bands = a.slice_bands * a.row_bands;
			const uint32_t block = xcd_grouped(blockIdx.x, a.together, gridDim.x);
			const uint32_t group = block / bands;
			const uint32_t slice_band = (block - group * bands) / a.row_bands;
			const uint32_t row_band = block - group * bands - slice_band * a.row_bands;
			const uint32_t first_plane = group * a.planes;
			const uint32_t planes_here = min(a.planes, a.plane_count - first_plane);
			const uint32_t first_slice = slice_band * a.slices, slices_here = min(a.slices, a.out_d - first_slice);
			const uint32_t first_row = row_band * a.rows, rows_here = min(a.rows, a.out_h - first_row);
			const uint32_t win_w = (WIN > 0) ? WIN : a.win_w;
			const uint32_t win_h = (WIN > 0) ? WIN : a.win_h;
			const uint32_t win_d = (WIN > 0) ? WIN : a.win_d;
			const uint32_t in_slice = a.in_w * a.in_h;
			const uint32_t in_plane = in_slice * a.in_d;

			// input slices [in_z0, in_z1) and, with several row bands, rows [in_y0, in_y1) of each
			const uint32_t in_z0 = first_slice * a.stride_z;
			const uint32_t in_z1 = (planes_here > 1) ? a.in_d : min(a.in_d, (first_slice + slices_here - 1) * a.stride_z + win_d);
			const uint32_t in_y0 = first_row * a.stride_y;
			const uint32_t in_y1 = min(a.in_h, (first_row + rows_here - 1) * a.stride_y + win_h);
			const bool one_run = a.row_bands == 1;
			const uint32_t g0 = first_plane * in_plane + in_z0 * in_slice + in_y0 * a.in_w; // first float staged
			const uint32_t run_floats = one_run ? (planes_here - 1) * in_plane + (in_z1 - in_z0) * in_slice : (in_y1 - in_y0) * a.in_w;
			const uint32_t shift = g0 & 3u;
			const uint32_t vectors = one_run ? (shift + run_floats + 3) / 4 : (in_z1 - in_z0) * a.run_vectors;
			const uint32_t whole_tensor_vectors = a.total_in / 4;

			for(uint32_t base = 0; base < vectors; base += stage3d_vectors_per_lane * max_block_size)
			{
				floatx4 t[stage3d_vectors_per_lane];
				#pragma unroll
				for(int k = 0; k < stage3d_vectors_per_lane; ++k)
				{
					// no branch around a load: what lies past the end of the range, of a run or of the tensor reads the last
					// float4 of the tensor or something nobody looks at
					const uint32_t i = min(base + k * max_block_size + threadIdx.x, vectors - 1);
					uint32_t v;
					if (one_run)
						v = g0 / 4 + i;
					else
					{
						const uint32_t run = fast_divide(i, a.run_vectors, a.run_vectors_magic);
						v = (g0 + run * in_slice) / 4 + (i - run * a.run_vectors);
					}
					t[k] = load_stream(reinterpret_cast<const floatx4*>(a.in) + min(v, whole_tensor_vectors - 1));
				}
				#pragma unroll
				for(int k = 0; k < stage3d_vectors_per_lane; ++k)
				{
					const uint32_t i = base + k * max_block_size + threadIdx.x;
					if (i < vectors)
						*reinterpret_cast<floatx4*>(lds_in + i * 4) = (OP == window_op_sum) ? t[k] : quiet(t[k]);
				}
			}
			// the tensor's last values, where they do not fill a float4 and belong to this block's last run
			const uint32_t last_run_start = one_run ? g0 : g0 + (in_z1 - in_z0 - 1) * in_slice;
			if (last_run_start + run_floats > whole_tensor_vectors * 4)
			{
				__syncthreads();
				const uint32_t g = whole_tensor_vectors * 4 + threadIdx.x;
				if (g < last_run_start + run_floats)
				{
					const uint32_t at = (one_run ? 0u : (in_z1 - in_z0 - 1) * a.run_vectors * 4) + (last_run_start & 3u) + (g - last_run_start);
					lds_in[at] = (OP == window_op_sum) ? a.in[g] : quiet(a.in[g]);
				}
			}
			__syncthreads();

			const uint32_t rows_magic = (row_band + 1 == a.row_bands) ? a.last_rows_magic : a.rows_magic;
			const uint32_t units = planes_here * slices_here * rows_here * a.units_w;
			for(uint32_t u = threadIdx.x; u < units; u += max_block_size)
			{
				const uint32_t all_rows = fast_divide(u, a.units_w, a.units_w_magic);
				const uint32_t ux = u - all_rows * a.units_w;
				const uint32_t all_slices = fast_divide(all_rows, rows_here, rows_magic);
				const uint32_t uy = all_rows - all_slices * rows_here;
				const uint32_t p = (planes_here > 1) ? fast_divide(all_slices, a.slices, a.slices_magic) : 0u;
				const uint32_t uz = all_slices - p * slices_here; // several volumes: slices_here == a.slices == out_d
				const uint32_t x0 = ux * (PAIR ? 2 * a.stride_x : a.stride_x);
				const uint32_t y0 = uy * a.stride_y, z0 = uz * a.stride_z; // inside the block
				const uint32_t last_x = TRUNC ? min(win_w, a.in_w - x0) - 1 : win_w - 1;
				const uint32_t last_y = TRUNC ? min(win_h, a.in_h - in_y0 - y0) - 1 : win_h - 1;
				const uint32_t last_z = TRUNC ? min(win_d, a.in_d - in_z0 - z0) - 1 : win_d - 1;
				// where slice z of the window starts in LDS
				const auto slice_at = [&](uint32_t z) -> const float*
				{
					const uint32_t inside = y0 * a.in_w + x0;
					if (one_run)
						return lds_in + shift + p * in_plane + (z0 + z) * in_slice + inside;
					return lds_in + (z0 + z) * (a.run_vectors * 4) + ((g0 + (z0 + z) * in_slice) & 3u) + inside;
				};
				float* const dst = a.out + ((static_cast<size_t>(first_plane + p) * a.out_d + first_slice + uz) * a.out_h + first_row + uy) * a.out_w + (PAIR ? 2 * ux : ux);
				if (WIN > 0)
				{
					constexpr int W = (WIN > 0) ? WIN : 1;
					float first[W * W * W], second[PAIR ? W * W * W : 1];
					#pragma unroll
					for(int z = 0; z < W; ++z)
					{
						const float* const slice = slice_at(TRUNC ? min(static_cast<uint32_t>(z), last_z) : z);
						#pragma unroll
						for(int y = 0; y < W; ++y)
						{
							const float* const row = slice + (TRUNC ? min(static_cast<uint32_t>(y), last_y) : y) * a.in_w;
							const int at = (z * W + y) * W;
							if (PAIR)
							{
								// columns x0 .. x0 + 3 lie inside the row; the second window's third column, x0 + 4, may not
								const floatx4 v = *reinterpret_cast<const floatx4*>(row);
								first[at] = v.x;
								first[at + 1] = v.y;
								second[PAIR ? at : 0] = v.z;
								second[PAIR ? at + 1 : 0] = v.w;
								if (W == 3)
								{
									first[at + W - 1] = v.z;
									second[PAIR ? at + W - 1 : 0] = (!TRUNC || (x0 + 4 < a.in_w)) ? row[4] : v.w;
								}
							}
							else
							{
								#pragma unroll
								for(int x = 0; x < W; ++x)
									first[at + x] = row[TRUNC ? min(static_cast<uint32_t>(x), last_x) : x];
							}
						}
					}
					if constexpr (PAIR)
					{
						float2 both;
						fold_values_twice<OP>(both.x, both.y, first, second);
						if (OP == window_op_sum)
						{
							both.x *= a.mult;
							both.y *= a.mult;
						}
						*reinterpret_cast<float2*>(dst) = both;
					}
					else
					{
						const float folded = fold_values<OP>(first);
						*dst = (OP == window_op_sum) ? folded * a.mult : folded;
					}
				}
				else
				{
					const auto scan = [&](auto fold_one)
					{
						for(uint32_t z = 0; z <= last_z; ++z)
						{
							const float* row = slice_at(z);
							for(uint32_t y = 0; y <= last_y; ++y, row += a.in_w)
								for(uint32_t x = 0; x <= last_x; ++x)
									fold_one(row[x]);
						}
					};
					float current = window_fold_start<OP>();
					if (OP == window_op_sum)
					{
						scan([&](float v) { current += v; });
						current *= a.mult;
					}
					else
					{
						constexpr bool is_min = (OP == window_op_min);
						scan([&](float v) { current = hw_fold<is_min>(current, v); });
						if (current == 0.0f)
						{
							// which zero: the first one in scan order, as the reference's fold keeps it
							current = window_fold_start<OP>();
							scan([&](float v) { current = fold<is_min>(current, v); });
						}
					}
					*dst = current;
				}
			}
		}

		template<int OP, bool TRUNC>
		void launch_window3d(hipStream_t stream, const window3d_args& a, uint32_t grid, size_t lds_bytes, bool pair)
		{
			const bool w2 = (a.win_w == 2) && (a.win_h == 2) && (a.win_d == 2), w3 = (a.win_w == 3) && (a.win_h == 3) && (a.win_d == 3);
			const dim3 g(grid), b(max_block_size);
			if (w2 && pair) NNF_LAUNCH((window3d_kernel<OP, 2, TRUNC, true>), g, b, lds_bytes, stream, a);
			else if (w2) NNF_LAUNCH((window3d_kernel<OP, 2, TRUNC, false>), g, b, lds_bytes, stream, a);
			else if (w3 && pair) NNF_LAUNCH((window3d_kernel<OP, 3, TRUNC, true>), g, b, lds_bytes, stream, a);
			else if (w3) NNF_LAUNCH((window3d_kernel<OP, 3, TRUNC, false>), g, b, lds_bytes, stream, a);
			else NNF_LAUNCH((window3d_kernel<OP, 0, TRUNC, false>), g, b, lds_bytes, stream, a);
		}

		// LDS floats a workgroup stages: five workgroups per compute unit (4K, 6K, 13K instead: 18.5, 21.1 and 20.3 us for 16 x 64
		// volumes of 28^3, 31.7, 30.5, 36.3 us for 4 x 40 of 64^3); fewer where the tensor would not give every compute unit four
		// workgroups otherwise (1 x 77 of 40^3: 6.0 us; ten per compute unit 7.7 us)
		constexpr uint32_t volume_staging_floats = 8u * 1024u - 8u;
		constexpr uint32_t volume_staging_floats_min = 2u * 1024u;
		constexpr uint32_t volume_workgroups_wanted = 1024u;
		constexpr uint32_t volume_staging_floats_max = 15u * 1024u;
	}

	// Plans and launches the 3-D window kernel. op: 0 maximum, 1 minimum, 2 maximum with windows cut off at the input's edge
	// (round up), 3 minimum likewise, 4 sum times mult. False (nothing launched) when not even one window's rows fit LDS.
	bool window3d_launch(hipStream_t stream, int op, float mult, float* output, const float* input, uint32_t input_total, uint32_t plane_count,
		const uint32_t (&in_size)[3], const uint32_t (&out_size)[3], const uint32_t (&window)[3], const uint32_t (&stride)[3])
	{
		if (input_total < 4)
			return false;
		window3d_args a = {};
		a.out = output;
		a.in = input;
		a.total_in = input_total;
		a.plane_count = plane_count;
		a.in_w = in_size[0]; a.in_h = in_size[1]; a.in_d = in_size[2];
		a.out_w = out_size[0]; a.out_h = out_size[1]; a.out_d = out_size[2];
		a.win_w = window[0]; a.win_h = window[1]; a.win_d = window[2];
		a.stride_x = stride[0]; a.stride_y = stride[1]; a.stride_z = stride[2];
		a.mult = mult;
		const uint64_t slice = static_cast<uint64_t>(a.in_w) * a.in_h, volume = slice * a.in_d;
		const uint64_t out_slice = static_cast<uint64_t>(a.out_w) * a.out_h, out_volume = out_slice * a.out_d;
		const auto input_span = [](uint64_t outputs, uint32_t stride, uint32_t window, uint32_t size) { return std::min<uint64_t>(size, (outputs - 1) * stride + window); };
		a.planes = 1;
		a.rows = a.out_h;
		a.slices = a.out_d;
		const uint32_t wanted_floats = std::max(volume_staging_floats_min, std::min(volume_staging_floats, input_total / volume_workgroups_wanted));
		if (volume <= wanted_floats)
		{
			// whole volumes: enough of them for a few outputs per lane, few enough to keep the grid wide
			a.planes = static_cast<uint32_t>(std::max<uint64_t>(1, std::min<uint64_t>(wanted_floats / volume, (4u * max_block_size + out_volume - 1) / out_volume)));
		}
		else
		{
			// The block (slices x rows of outputs) whose input fits and is least per output: what neighbouring blocks both fetch
			// is least. Among equals (windows as wide as their stride: all of them) the largest block.
			double best = 0.0;
			uint64_t best_floats = 0;
			for(uint32_t floats : { wanted_floats, volume_staging_floats, volume_staging_floats_max })
			{
				for(uint32_t s = 1; s <= a.out_d; ++s)
				{
					const uint64_t depth = input_span(s, a.stride_z, a.win_d, a.in_d);
					if (depth * a.win_h * a.in_w > floats)
						break;
					uint32_t r = a.out_h;
					if (depth * slice > floats)
					{
						const uint64_t per_slice = floats / depth, rows_in = (per_slice - std::min<uint64_t>(per_slice, 8)) / a.in_w; // a run is padded to whole float4s
						if (rows_in < a.win_h)
							break;
						r = static_cast<uint32_t>(std::min<uint64_t>(a.out_h, (rows_in - a.win_h) / a.stride_y + 1));
						const uint32_t bands = (a.out_h + r - 1) / r;
						r = (a.out_h + bands - 1) / bands;
					}
					const uint64_t block_floats = depth * ((r == a.out_h) ? a.in_h : input_span(r, a.stride_y, a.win_h, a.in_h)) * a.in_w;
					const double per_output = static_cast<double>(block_floats) / (static_cast<double>(s) * r);
					if ((best == 0.0) || (per_output < 0.995 * best) || ((per_output < 1.005 * best) && (block_floats > best_floats)))
					{
						best = per_output;
						best_floats = block_floats;
						a.slices = s;
						a.rows = r;
					}
				}
				if (best != 0.0)
					break;
			}
			if (best == 0.0)
				return false;
			const uint32_t bands = (a.out_d + a.slices - 1) / a.slices;
			a.slices = (a.out_d + bands - 1) / bands;
		}
		a.slice_bands = (a.out_d + a.slices - 1) / a.slices;
		a.row_bands = (a.out_h + a.rows - 1) / a.rows;
		// Blocks that share input values, or cache lines at the ends of their runs, meet in one XCD's L2: 4 x 40 volumes of 64^3 in
		// 3 x 3 x 3 every 2 41.6 -> 35.2 us, in 2 x 2 x 2 35.8 -> 31.3 us. Blocks of whole slices without overlap share nothing
		// (16 x 64 volumes of 28^3: 17.8 us grouped, 17.4 us in plain order).
		a.together = ((a.row_bands > 1) || (a.win_d > a.stride_z)) ? a.slice_bands * a.row_bands : 0u;
		const uint64_t depth = (a.planes > 1) ? a.in_d : input_span(a.slices, a.stride_z, a.win_d, a.in_d);
		uint64_t lds_floats;
		if (a.row_bands == 1)
			lds_floats = (a.planes - 1) * volume + depth * slice + 8;
		else
		{
			a.run_vectors = static_cast<uint32_t>((input_span(a.rows, a.stride_y, a.win_h, a.in_h) * a.in_w + 3 + 3) / 4); // wherever the run starts inside a float4
			lds_floats = depth * a.run_vectors * 4 + 8;
		}
		const bool pair = (a.stride_x == 2) && ((a.in_w % 4) == 0) && ((a.out_w % 2) == 0) && (a.win_w == a.win_h) && (a.win_w == a.win_d) && ((a.win_w == 2) || (a.win_w == 3));
		a.units_w = pair ? a.out_w / 2 : a.out_w;
		// the divisions by multiplication are exact below 2^16
		if ((lds_floats > volume_staging_floats_max + 1024) || (static_cast<uint64_t>(a.planes) * a.slices * a.rows * a.units_w >= (1u << 16)))
			return false;
		a.units_w_magic = magic_of(a.units_w);
		a.rows_magic = magic_of(a.rows);
		a.last_rows_magic = magic_of(a.out_h - (a.row_bands - 1) * a.rows);
		a.slices_magic = magic_of(a.slices);
		a.run_vectors_magic = magic_of(a.run_vectors);
		const uint64_t grid = static_cast<uint64_t>((a.plane_count + a.planes - 1) / a.planes) * a.slice_bands * a.row_bands;
		if (grid > 0x7FFFFFFFull)
			return false;
		const size_t lds_bytes = static_cast<size_t>(lds_floats) * sizeof(float);
		switch (op)
		{
		case 0: launch_window3d<window_op_max, false>(stream, a, static_cast<uint32_t>(grid), lds_bytes, pair); break;
		case 1: launch_window3d<window_op_min, false>(stream, a, static_cast<uint32_t>(grid), lds_bytes, pair); break;
		case 2: launch_window3d<window_op_max, true>(stream, a, static_cast<uint32_t>(grid), lds_bytes, pair); break;
		case 3: launch_window3d<window_op_min, true>(stream, a, static_cast<uint32_t>(grid), lds_bytes, pair); break;
		default: launch_window3d<window_op_sum, false>(stream, a, static_cast<uint32_t>(grid), lds_bytes, pair); break;
		}
		return true;
	}
}
