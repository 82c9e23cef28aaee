// The fold of a window's values - maximum, minimum or sum - shared by the window kernels (nnf_max.hip: 1-D and 2-D windows,
// windows over feature maps and entries; nnf_window3d.hip: volumes).
#pragma once

#include "nnf_common.h"

namespace nnf
{
	namespace
	{
		constexpr int max_block_size = 256; // lanes per workgroup of the window kernels

		// std::max<float>(current, new_val) / std::min<float>(current, new_val)
		template<bool IS_MIN>
		__device__ __forceinline__ float fold(float current, float new_val)
		{
			if (IS_MIN)
				return (new_val < current) ? new_val : current;
			return (current < new_val) ? new_val : current;
		}

		// What the window kernels do with the values of a window, scanned x fastest:
		// maximum, minimum (both from the -/+1.0e37F start value), or their left-to-right sum times a
		// multiplier (average subsampling, nnforge/plain/average_subsampling_layer_tester_plain.cpp:125-145).
		constexpr int window_op_max = 0;
		constexpr int window_op_min = 1;
		constexpr int window_op_sum = 2;

		template<int OP>
		__device__ __forceinline__ float window_fold(float current, float new_val)
		{
			if (OP == window_op_sum)
				return current + new_val;
			return fold<OP == window_op_min>(current, new_val);
		}

		template<int OP>
		__device__ __forceinline__ float window_fold_start()
		{
			if (OP == window_op_sum)
				return 0.0f;
			return (OP == window_op_min) ? 1.0e37f : -1.0e37f;
		}

		// ---- the hardware's maximum / minimum, with the reference's result ------------------------
		// std::max<float>(current, new) from a finite start value never holds a NaN (current < NaN is false), so a
		// window's result is the largest of the start value and the window's numbers - whatever the order of
		// the fold - with one exception: when that largest value is a zero, the fold keeps the first zero it met,
		// -0.0 or +0.0, while v_max_f32 ranks +0.0 above -0.0. The kernels therefore fold with v_max3_f32 /
		// v_min3_f32 (two values per instruction instead of a compare and a select per value) and a lane whose
		// result is a zero folds its window again the reference's way. v_max_f32 passes over a quiet NaN operand but
		// answers a signalling one with a NaN, which the next fold would then pass over together with everything
		// folded so far: the values are made quiet (canonical) once, on their way into LDS.
		__device__ __forceinline__ float quiet(float v)
		{
			return __builtin_canonicalizef(v);
		}

		__device__ __forceinline__ floatx4 quiet(floatx4 v)
		{
			floatx4 q;
			q.x = quiet(v.x); q.y = quiet(v.y); q.z = quiet(v.z); q.w = quiet(v.w);
			return q;
		}

		template<bool IS_MIN>
		__device__ __forceinline__ float hw_fold(float a, float b)
		{
			float d;
			if (IS_MIN)
				asm("v_min_f32 %0, %1, %2" : "=v"(d) : "v"(a), "v"(b));
			else
				asm("v_max_f32 %0, %1, %2" : "=v"(d) : "v"(a), "v"(b));
			return d;
		}

		template<bool IS_MIN>
		__device__ __forceinline__ float hw_fold3(float a, float b, float c)
		{
			float d;
			if (IS_MIN)
				asm("v_min3_f32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
			else
				asm("v_max3_f32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
			return d;
		}

		// The largest (smallest) of the start value and COUNT quiet values: the window's result, unless it is a zero.
		template<int OP, int COUNT>
		__device__ __forceinline__ float fold_values_hw(const float (&v)[COUNT])
		{
			constexpr bool is_min = (OP == window_op_min);
			float current = window_fold_start<OP>();
			#pragma unroll
			for(int i = 0; i + 1 < COUNT; i += 2)
				current = hw_fold3<is_min>(current, v[i], v[i + 1]);
			if (COUNT % 2 != 0)
				current = hw_fold<is_min>(current, v[COUNT - 1]);
			return current;
		}

		// The reference's fold of COUNT values in the order given.
		template<int OP, int COUNT>
		__device__ __forceinline__ float fold_values_in_order(const float (&v)[COUNT])
		{
			float current = window_fold_start<OP>();
			#pragma unroll
			for(int i = 0; i < COUNT; ++i)
				current = window_fold<OP>(current, v[i]);
			return current;
		}

		// One window: the values in scan order (quiet ones, for maximum and minimum).
		template<int OP, int COUNT>
		__device__ __forceinline__ float fold_values(const float (&v)[COUNT])
		{
			if (OP == window_op_sum)
				return fold_values_in_order<OP>(v);
			float current = fold_values_hw<OP>(v);
			if (current == 0.0f)
				current = fold_values_in_order<OP>(v); // which zero: the first one in scan order
			return current;
		}

		// Two windows behind one test, so that the lanes without a zero jump over one block of code instead of
		// stepping through two short ones.
		template<int OP, int COUNT>
		__device__ __forceinline__ void fold_values_twice(float& first_result, float& second_result, const float (&first)[COUNT], const float (&second)[COUNT])
		{
			if (OP == window_op_sum)
			{
				first_result = fold_values_in_order<OP>(first);
				second_result = fold_values_in_order<OP>(second);
				return;
			}
			first_result = fold_values_hw<OP>(first);
			second_result = fold_values_hw<OP>(second);
			if ((first_result == 0.0f) || (second_result == 0.0f))
			{
				first_result = fold_values_in_order<OP>(first);
				second_result = fold_values_in_order<OP>(second);
			}
		}
	}
}
