/*
 * Softmax and fused softmax + cross-entropy for rows of up to 131,072 fp8 or
 * 16-bit or 65,536 fp32 columns at any alignment: the "_rows" and "_wide_rows"
 * kernels of softmax_xent.hip's ops (same arithmetic), chosen by
 * smx_kernel_for.
 *
 * The main kernels give every row a whole CU and prefetch the next one, which
 * pays for rows of about 100,000 columns: each row costs them 7 us (16-bit) of
 * 16 unrolled chunks and two workgroup reductions whatever its length, and
 * rows that are not 16-byte aligned went element by element, three times
 * through memory. What bounds these kernels is HBM from about 4000 columns
 * on. Measured on MI355X, main -> these, bf16 softmax / fused loss:
 *   16384 x 1000   478 ->  15 us      561 ->  24 us
 *   16384 x 8192   480 ->  87 us      564 ->  93 us  (537 MB: 6.2 / 5.8 TB/s)
 *    4096 x 32000  151 ->  92 us      187 ->  96 us  (524 MB: 5.7 / 5.5 TB/s)
 *    4096 x 50257  765 -> 156 us      687 -> 162 us  (823 MB: 5.3 / 5.1 TB/s)
 *    1024 x 128257 557 -> 116 us      588 -> 127 us
 * and softmax of fp8 logits into bf16:
 *    4096 x 1000    43 -> 6.3 us,  4096 x 32000 102 -> 71 us (393 MB: 5.5 TB/s),
 *    1024 x 50257  171 -> 32 us,   1024 x 100001 373 -> 80 us
 */

/* A chunk: 16 bytes, or for fp8 logits, whose outputs are 16-bit, 8 bytes, so
 * that a lane's output chunk is 16 bytes too. */
template <typename T>
struct SmxChunk {
	static constexpr int N = VecOf<T>::N;
	typedef R16 raw;
	__device__ static __forceinline__ raw load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) { return buf_load16_nt(r, voff, soff); }
	/* for data that other workgroups of the launch read too */
	__device__ static __forceinline__ raw load_again(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) { return buf_load16(r, voff, soff); }
	__device__ static __forceinline__ void unpack(const raw & r, float * f) { unpack16<T>(r, f); }
};
template <typename T>
struct SmxChunkFp8 {
	static constexpr int N = 8;
	typedef R8 raw;
	template <int AUX>
	__device__ static __forceinline__ raw load_aux(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
		const u32x2_v v = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, AUX);
		raw o;
		o.w[0] = v.x;
		o.w[1] = v.y;
		return o;
	}
	__device__ static __forceinline__ raw load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) { return load_aux<BUF_AUX_NT>(r, voff, soff); }
	__device__ static __forceinline__ raw load_again(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) { return load_aux<0>(r, voff, soff); }
	__device__ static __forceinline__ void unpack(const raw & r, float * f) { unpack8_fp8<T>(r, f); }
	__device__ static __forceinline__ void opaque(raw & r) { reg_barrier8(r); }
};
template <> struct SmxChunk<fp8e4m3_t> : SmxChunkFp8<fp8e4m3_t> {};
template <> struct SmxChunk<fp8e5m2_t> : SmxChunkFp8<fp8e5m2_t> {};

/* reductions over the `g` waves of a row, the waves' partials combined from
 * one LDS read per lane (16 cells, then the row of 16 lanes) in a fixed order */
__device__ __forceinline__ float row16_max(float v) {
	v = fmaxf(v, dpp_f32<DPP_QUAD_1032>(v));
	v = fmaxf(v, dpp_f32<DPP_QUAD_2301>(v));
	v = fmaxf(v, dpp_f32<DPP_ROW_HALF_MIRROR>(v));
	v = fmaxf(v, dpp_f32<DPP_ROW_MIRROR>(v));
	return readlane_f32(v, 0);
}
__device__ __forceinline__ float row16_sum(float v) {
	v += dpp_f32<DPP_QUAD_1032>(v);
	v += dpp_f32<DPP_QUAD_2301>(v);
	v += dpp_f32<DPP_ROW_HALF_MIRROR>(v);
	v += dpp_f32<DPP_ROW_MIRROR>(v);
	return readlane_f32(v, 0);
}
__device__ __forceinline__ float waves_max(float v, float * cells, int g, int wave, int lane) {
	v = wave_max(v);
	if (g == 1) return v;
	if (lane == 0) cells[wave] = v;
	lds_barrier();
	const int k = lane & 15;
	return row16_max(k < g ? cells[k] : -__builtin_inff());
}
__device__ __forceinline__ void waves_sum2(float & a, float & b, float * cells, int g, int wave, int lane) {
	a = wave_sum(a);
	b = wave_sum(b);
	if (g == 1) return;
	if (lane == 0) { cells[wave] = a; cells[16 + wave] = b; }
	lds_barrier();
	const int k = lane & 15;
	a = row16_sum(k < g ? cells[k] : 0.0f);
	b = row16_sum(k < g ? cells[16 + k] : 0.0f);
}

/* The mean loss of a launch whose workgroups end in any order, without one
 * counter that all of them would queue at: workgroups are counted in groups
 * of consecutive ones (SMX_GROUP_WGS, more where that would be more than
 * SMX_GROUPS groups); the wave that completes a group sums its rows' losses
 * (fp64, fixed order) and counts the group, and the wave that completes the
 * last group sums the groups and resets the counters. The counters are zero
 * between launches, and the handle orders launches that share them. */
#define SMX_GROUPS 256
#define SMX_GROUP_WGS 64
#define SMX_GROUP_STRIDE 32   /* counters 128 bytes apart */
__device__ __attribute__((aligned(4096))) unsigned int g_smx_group_done[(SMX_GROUPS + 1) * SMX_GROUP_STRIDE];
__device__ double g_smx_group_sum[SMX_GROUPS];

struct SmxGroup {
	int first, count, index, n_groups;   /* workgroups */
	__device__ __forceinline__ SmxGroup() {
		const int wg = (int) blockIdx.x, n = (int) gridDim.x;
		int per = (n + SMX_GROUPS - 1) / SMX_GROUPS;
		if (per < SMX_GROUP_WGS) per = SMX_GROUP_WGS;
		n_groups = (n + per - 1) / per;
		index = wg / per;
		first = index * per;
		count = (n - first) < per ? (n - first) : per;
	}
};

/* counts this wave's earlier stores as made (lane 0's, once they are
 * complete); the count before it, valid in lane 0 */
__device__ __forceinline__ unsigned smx_arrive(unsigned * counter, int lane) {
	unsigned d = 0u;
	if (lane == 0) {
		__asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
		d = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	}
	return d;
}
__device__ __forceinline__ double wave_sum_f64(double s) {
	for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
	return s;
}
/* a wave whose workgroup was the `arrived`-th (from 0, in lane 0) of its group;
 * workgroup b has rows b * rows_per_wg and the next ones */
__device__ __forceinline__ void smx_rows_mean(const SmxGroup & g, unsigned arrived, int rows_per_wg, int n_rows, const float * loss, float * mean_loss, int lane) {
	unsigned * done = g_smx_group_done + g.index * SMX_GROUP_STRIDE;
	if ((int) __builtin_amdgcn_readfirstlane(arrived) != g.count - 1) return;
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
	double s = 0.0;
	const int r0 = g.first * rows_per_wg;
	for (int k = lane; k < g.count * rows_per_wg; k += 64)
		if (r0 + k < n_rows) s += (double) __hip_atomic_load(loss + r0 + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	s = wave_sum_f64(s);
	if (lane == 0) __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	if (g.n_groups > 1) {
		unsigned * all = g_smx_group_done + SMX_GROUPS * SMX_GROUP_STRIDE;
		if (lane == 0) __hip_atomic_store(&g_smx_group_sum[g.index], s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		if ((int) __builtin_amdgcn_readfirstlane(smx_arrive(all, lane)) != g.n_groups - 1) return;
		__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
		s = 0.0;
		for (int k = lane; k < g.n_groups; k += 64) s += __hip_atomic_load(&g_smx_group_sum[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		s = wave_sum_f64(s);
		if (lane == 0) __hip_atomic_store(all, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	}
	if (lane == 0) *mean_loss = (float) (s / (double) n_rows);
}

/* the window's elements outside the row become -inf, in place (fp8, which has
 * no infinity in E4M3, masks the unpacked values instead) */
template <typename T>
__device__ __forceinline__ void smx_mask_chunk(R16 & r, uint32_t pos, uint32_t h, uint32_t end) {
	constexpr int PW = 4 / (int) sizeof(T);   /* elements per word */
#pragma unroll
	for (int i = 0; i < 4; i++) {
		uint32_t keep = 0u;
#pragma unroll
		for (int e = 0; e < PW; e++) {
			const uint32_t p = pos + (uint32_t) (i * PW + e);
			if (p >= h && p < end) keep |= (PW == 1 ? 0xffffffffu : 0xffffu << (16 * e));
		}
		r.w[i] = (r.w[i] & keep) | (SmxWord<T>::NEG_INF & ~keep);
	}
}

/* d = rnd(x - m) of a pair of fp8 values, in the 16-bit output type: opaque,
 * so that both halves come from one packed convert */
template <typename TO>
__device__ __forceinline__ void smx_round2(const float * x_m, float * d) {
	uint32_t w = SmxWord<TO>::pack(x_m);
	__asm__ volatile("" : "+v"(w));
	SmxWord<TO>::unpack(w, d);
}

/*
 * One row per `g` waves (smx_rows_waves: a wave alone, or a workgroup of g),
 * CH 16-byte chunks per thread, loaded at once, reduced twice and written;
 * no loop over rows: several workgroups share a CU, so one row's loads and
 * stores run under another's arithmetic, and a finished row's stores drain
 * behind its successor.
 * KEEP (CH * elements per chunk floats fit the registers): the exponentials
 * of the sum pass stay in registers in fp32 and the output pass multiplies
 * them by 1 / sum, one exponential less per element than forming them again
 * from the rounded differences, which the longest rows (CH = 16) do.
 */
template <typename T, typename TO, bool FUSED, int CH>
__device__ __forceinline__ void smx_rows(int n_rows, int n_cols, const T * X, TO * out, const uint32_t * labels, float * loss, float * mean_loss) {
	using C = SmxChunk<T>;
	constexpr int VEC = C::N;
	constexpr int CB = VEC * (int) sizeof(T);   /* bytes of a chunk */
	constexpr int OB = VEC * (int) sizeof(TO);
	constexpr bool KEEP = CH * VEC <= 64;
	constexpr bool F8 = IsFp8<T>::value;
	static_assert(OB == 16, "a chunk's outputs are one 16-byte store");
	__shared__ float mcells[16];
	__shared__ float scells[32];
	__shared__ float xlab_cell[SMX_ROWS_PER_WG];
	const int lane = threadIdx.x & 63;
	const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int g = smx_rows_waves(CH, n_rows, n_cols, (int) sizeof(T), (unsigned long long) (uintptr_t) X, (unsigned long long) (uintptr_t) out);
	const int wave = (g == 1) ? 0 : wv;
	const int cell = (g == 1) ? wv : 0;
	const int nt = 64 * g;
	const int t = wave * 64 + lane;
	const SmxGroup grp;
	unsigned arrived = 0u;
	const bool mean = FUSED && loss && mean_loss;
	const int row = (g == 1) ? (int) blockIdx.x * SMX_ROWS_PER_WG + wv : (int) blockIdx.x;
	if (row < n_rows) {   /* whole waves: no barrier where g == 1 */
	const SmxWindow w = smx_window<T, TO>(X, out, n_cols, row);
	const int nch = (w.chunks + nt - 1) / nt;
	const uint32_t voff = (uint32_t) t * OB;
	const __amdgpu_buffer_rsrc_t rin = make_rsrc(w.in, (uint32_t) w.chunks * CB);
	const __amdgpu_buffer_rsrc_t rout = make_rsrc(w.out, (uint32_t) w.chunks * OB);

	typename C::raw x[CH];
#pragma unroll
	for (int c = 0; c < CH; c++)
		if (c < nch) x[c] = C::load(rin, (uint32_t) t * CB, (uint32_t) (c * nt) * CB);
	const uint32_t lab = FUSED ? load_scalar(labels + row) : 0xffffffffu;
	const bool lab_ok = FUSED && lab < (uint32_t) n_cols;
	/* the label's chunk, its thread and its element there */
	const uint32_t lab_pos = lab_ok ? lab + w.h : 0u;
	const int lab_chunk = (int) (lab_pos / VEC);
	const int c_lab = lab_ok ? lab_chunk / nt : -1;
	const int t_lab = lab_chunk - (lab_ok ? c_lab * nt : 0);
	const int le = (int) (lab_pos % VEC);
	/* Elements outside the row are -inf, which changes neither the max nor
	 * the sums. Only the first and the last chunk of a thread can hold any (h
	 * is below one line). */
	auto edge = [&](int c) { return c == 0 || c == nch - 1; };
	auto partial = [&](int c) {
		const uint32_t pos = (uint32_t) (c * nt + t) * VEC;
		return pos < w.h || pos + VEC > w.end;
	};
	/* fp8: a chunk's values, unpacked anew in every pass */
	auto values = [&](int c, float (&f)[VEC]) {
		if constexpr (F8) C::opaque(x[c]);
		C::unpack(x[c], f);
		if (edge(c) && partial(c)) {
			const uint32_t pos = (uint32_t) (c * nt + t) * VEC;
#pragma unroll
			for (int e = 0; e < VEC; e++)
				if (pos + e < w.h || pos + e >= w.end) f[e] = -__builtin_inff();
		}
	};

	float m = -__builtin_inff();
#pragma unroll
	for (int c = 0; c < CH; c++) {
		if (c < nch) {
			if constexpr (F8) {
				float f[VEC];
				values(c, f);
#pragma unroll
				for (int e = 0; e < VEC; e++) m = __builtin_elementwise_maximum(m, f[e]);
			}
			else {
				if (edge(c) && partial(c)) smx_mask_chunk<T>(x[c], (uint32_t) (c * nt + t) * VEC, w.h, w.end);
				m = chunk_max<T>(x[c], m);
			}
		}
	}
	m = waves_max(m, mcells, g, wave, lane);

	float ef[KEEP ? CH : 1][VEC];
	float sd0 = 0.0f, sd1 = 0.0f, sx = 0.0f;
#pragma unroll
	for (int c = 0; c < CH; c++) {
		if (c < nch) {
			const bool lab_here = FUSED && c == c_lab && t == t_lab;
			float x_m[VEC], d[VEC];
			typename C::raw o;
			if constexpr (F8) {
				float f[VEC];
				values(c, f);
#pragma unroll
				for (int e = 0; e < VEC; e += 2) {
					x_m[e] = f[e] - m;
					x_m[e + 1] = f[e + 1] - m;
					smx_round2<TO>(x_m + e, d + e);
				}
				o = x[c];
			}
			else {
				using W = SmxWord<T>;
#pragma unroll
				for (int i = 0; i < 4; i++) o.w[i] = W::diff(x[c].w[i], m, x_m + i * W::N, d + i * W::N);
			}
			if (lab_here) {
				float f[VEC];
				C::unpack(x[c], f);
				float xl = f[0];
#pragma unroll
				for (int e = 1; e < VEC; e++)
					if (e == le) xl = f[e];
				xlab_cell[cell] = xl;
			}
			float ev[VEC];
#pragma unroll
			for (int e = 0; e < VEC; e++) {
				ev[e] = exp_fast(d[e]);
				if (e & 1) sd1 += ev[e]; else sd0 += ev[e];
			}
			if (FUSED) {
				/* the loss sum: unrounded differences, without the label's column */
				float tx[VEC];
#pragma unroll
				for (int e = 0; e < VEC; e++) tx[e] = sizeof(T) == 4 ? ev[e] : exp_fast(x_m[e]);
				if (lab_here) {
#pragma unroll
					for (int e = 0; e < VEC; e++)
						if (e == le) tx[e] = 0.0f;
				}
#pragma unroll
				for (int e = 0; e < VEC; e++) sx += tx[e];
			}
			if constexpr (KEEP) {
#pragma unroll
				for (int e = 0; e < VEC; e++) ef[c][e] = ev[e];
			}
			else x[c] = o;   /* the differences, exact in T (fp8: the logits) */
		}
	}
	float sd = sd0 + sd1;
	waves_sum2(sd, sx, scells, g, wave, lane);
	if (FUSED && wave == 0 && loss) {
		wave_lds_sync();   /* the labelled logit, another lane's where g == 1 (g > 1: the sums' barrier) */
		if (lane == 0) store_loss(loss, row, lab_ok ? fused_loss(sx, m, xlab_cell[cell]) : __builtin_nanf(""));
		/* a workgroup of one row counts it before the outputs, so that the
		 * store, the count and the sums that follow it run beside them */
		if (mean && g > 1) arrived = smx_arrive(g_smx_group_done + grp.index * SMX_GROUP_STRIDE, lane);
	}
	const float inv = 1.0f / sd;
	const float nlog2s = -__builtin_amdgcn_logf(sd);
#pragma unroll
	for (int c = 0; c < CH; c++) {
		if (c < nch) {
			float f[VEC];
			if constexpr (KEEP) {
#pragma unroll
				for (int e = 0; e < VEC; e++) f[e] = ef[c][e] * inv;
			}
			else {
				if constexpr (F8) {
					C::opaque(x[c]);
					C::unpack(x[c], f);
#pragma unroll
					for (int e = 0; e < VEC; e += 2) {
						f[e] -= m;
						f[e + 1] -= m;
						smx_round2<TO>(f + e, f + e);
					}
				}
				else C::unpack(x[c], f);
#pragma unroll
				for (int e = 0; e < VEC; e++) f[e] = __builtin_amdgcn_exp2f(fmaf(f[e], SMX_LOG2E, nlog2s));
			}
			R16 o = pack16<TO>(f);
			if (FUSED && c == c_lab && t == t_lab) {   /* rnd(y) - 1 */
				unpack16<TO>(o, f);
#pragma unroll
				for (int e = 0; e < VEC; e++)
					if (e == le) f[e] -= 1.0f;
				o = pack16<TO>(f);
			}
			if (edge(c)) {
				const uint32_t pos = (uint32_t) (c * nt + t) * VEC;
				if (pos >= w.h && pos + VEC <= w.end) buf_store16_nt(rout, voff, (uint32_t) (c * nt) * OB, o);
				else {
					TO * p = reinterpret_cast<TO *>(w.out);
					unpack16<TO>(o, f);
#pragma unroll
					for (int e = 0; e < VEC; e++)
						if (pos + e >= w.h && pos + e < w.end) p[pos + e] = from_f<TO>(f[e]);
				}
			}
			else buf_store16_nt(rout, voff, (uint32_t) (c * nt) * OB, o);
		}
	}
	}
	if (!mean) return;
	if (g == 1) {
		WAIT_VMEM_ALL();   /* this wave's losses are stored */
		__syncthreads();
		if (wv == 0) arrived = smx_arrive(g_smx_group_done + grp.index * SMX_GROUP_STRIDE, lane);
	}
	if (wv == 0) smx_rows_mean(grp, arrived, g == 1 ? SMX_ROWS_PER_WG : 1, n_rows, loss, mean_loss, lane);
}

#define SMX_ROWS_KERNEL(SUFFIX, PSUFFIX, T, VARIANT, CH)                                                               \
	extern "C" __global__ void __launch_bounds__(SMX_THREADS) softmax_##PSUFFIX##_kernel_##VARIANT(int n_rows,         \
			int n_cols, T * X, T * out) {                                                                              \
		smx_rows<T, T, false, CH>(n_rows, n_cols, X, out, nullptr, nullptr, nullptr);                                     \
	}                                                                                                                  \
	extern "C" __global__ void __launch_bounds__(SMX_THREADS) softmax_cross_entropy_loss_##SUFFIX##_kernel_##VARIANT(  \
			int n_rows, int n_cols, T * logits, uint32_t * labels, float * loss, float * mean_loss) {                  \
		smx_rows<T, T, true, CH>(n_rows, n_cols, logits, logits, labels, loss, mean_loss);                                \
	}
#define SMX_ROWS_KERNELS(SUFFIX, PSUFFIX, T)                                                                           \
	SMX_ROWS_KERNEL(SUFFIX, PSUFFIX, T, rows, SMX_ROWS_CH)                                                             \
	SMX_ROWS_KERNEL(SUFFIX, PSUFFIX, T, wide_rows, SMX_WIDE_ROWS_CH)

SMX_ROWS_KERNELS(fp32, fp32_fp32, float)
SMX_ROWS_KERNELS(fp16, fp16_fp16, f16_t)
SMX_ROWS_KERNELS(bf16, bf16_bf16, bf16_t)

#define SMX_FP8_ROWS_KERNEL(PSUFFIX, T, TO, VARIANT, CH)                                                               \
	extern "C" __global__ void __launch_bounds__(SMX_THREADS) softmax_##PSUFFIX##_kernel_##VARIANT(int n_rows,         \
			int n_cols, T * X, TO * out) {                                                                             \
		smx_rows<T, TO, false, CH>(n_rows, n_cols, X, out, nullptr, nullptr, nullptr);                                 \
	}
#define SMX_FP8_ROWS_KERNELS(PSUFFIX, T, TO)                                                                           \
	SMX_FP8_ROWS_KERNEL(PSUFFIX, T, TO, rows, SMX_ROWS_CH)                                                             \
	SMX_FP8_ROWS_KERNEL(PSUFFIX, T, TO, wide_rows, SMX_WIDE_ROWS_CH)

SMX_FP8_ROWS_KERNELS(fp8e4m3_fp16, fp8e4m3_t, f16_t)
SMX_FP8_ROWS_KERNELS(fp8e4m3_bf16, fp8e4m3_t, bf16_t)
SMX_FP8_ROWS_KERNELS(fp8e5m2_fp16, fp8e5m2_t, f16_t)
SMX_FP8_ROWS_KERNELS(fp8e5m2_bf16, fp8e5m2_t, bf16_t)
