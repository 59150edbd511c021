/*
 * Softmax and fused softmax + cross-entropy for rows of up to 131,072 16-bit
 * or 65,536 fp32 columns at any alignment: the "_rows" and "_wide_rows"
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
 */

/* The 16-byte chunks that cover a row: the window starts at the 128-byte line
 * (16-byte chunk, where input and output lie differently within their lines)
 * that holds the row's first element, so that every wave's loads and stores
 * are whole lines however long the rows are. Elements [h, end) of the window
 * are the row's; the others belong to the neighbouring rows, are read with it
 * (a chunk never crosses a page) and never written. */
struct SmxWindow {
	const char * in;
	char * out;
	uint32_t h, end;
	int chunks;
};

template <typename T>
__device__ __forceinline__ SmxWindow smx_window(const T * X, T * out, int n_cols, int row) {
	const uint64_t off = (uint64_t) row * (uint64_t) n_cols * sizeof(T);
	const uint64_t a = (uint64_t) (uintptr_t) X + off, o = (uint64_t) (uintptr_t) out + off;
	const uint64_t mask = ((a ^ o) & 127u) ? 15u : 127u;
	SmxWindow w;
	w.in = reinterpret_cast<const char *>(a & ~mask);
	w.out = reinterpret_cast<char *>(o & ~mask);
	w.h = (uint32_t) (a & mask) / (uint32_t) sizeof(T);
	w.end = w.h + (uint32_t) n_cols;
	w.chunks = (int) ((w.end + VecOf<T>::N - 1) / VecOf<T>::N);
	return w;
}

/* the window's elements outside the row become -inf */
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
__device__ unsigned int g_smx_group_done[(SMX_GROUPS + 1) * SMX_GROUP_STRIDE];
__device__ double g_smx_group_sum[SMX_GROUPS];

struct SmxGroup {
	int first, count, index, n_groups;
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
template <typename T, bool FUSED, int CH>
__device__ __forceinline__ void smx_rows(int n_rows, int n_cols, const T * X, T * out, const uint32_t * labels, float * loss, float * mean_loss) {
	constexpr int VEC = VecOf<T>::N;
	constexpr bool KEEP = CH * VEC <= 64;
	using W = SmxWord<T>;
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
	const SmxWindow w = smx_window<T>(X, out, n_cols, row);
	const int nch = (w.chunks + nt - 1) / nt;
	const uint32_t voff = (uint32_t) t * 16u;
	const __amdgpu_buffer_rsrc_t rin = make_rsrc(w.in, (uint32_t) w.chunks * 16u);
	const __amdgpu_buffer_rsrc_t rout = make_rsrc(w.out, (uint32_t) w.chunks * 16u);

	R16 x[CH];
#pragma unroll
	for (int c = 0; c < CH; c++)
		if (c < nch) x[c] = buf_load16_nt(rin, voff, (uint32_t) (c * nt) * 16u);
	const uint32_t lab = FUSED ? load_scalar(labels + row) : 0xffffffffu;
	const bool lab_ok = FUSED && lab < (uint32_t) n_cols;
	/* the label's chunk, its thread and its element there */
	const uint32_t lab_pos = lab_ok ? lab + w.h : 0u;
	const int lab_chunk = (int) (lab_pos / VEC);
	const int c_lab = lab_ok ? lab_chunk / nt : -1;
	const int t_lab = lab_chunk - (lab_ok ? c_lab * nt : 0);
	const int le = (int) (lab_pos % VEC);
	/* only the first and the last chunk of a thread can hold elements
	 * outside the row (h is below one line, 8 chunks) */
	auto edge = [&](int c) { return c == 0 || c == nch - 1; };

	float m = -__builtin_inff();
#pragma unroll
	for (int c = 0; c < CH; c++) {
		if (c < nch) {
			if (edge(c)) {
				const uint32_t pos = (uint32_t) (c * nt + t) * VEC;
				if (pos < w.h || pos + VEC > w.end) smx_mask_chunk<T>(x[c], pos, w.h, w.end);
			}
			m = chunk_max<T>(x[c], m);
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
			R16 o;
#pragma unroll
			for (int i = 0; i < 4; i++) o.w[i] = W::diff(x[c].w[i], m, x_m + i * W::N, d + i * W::N);
			if (lab_here) {
				float f[VEC];
				unpack16<T>(x[c], f);
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
			else x[c] = o;
		}
	}
	float sd = sd0 + sd1;
	waves_sum2(sd, sx, scells, g, wave, lane);
	if (FUSED && wave == 0 && loss) {
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
				unpack16<T>(x[c], f);
#pragma unroll
				for (int e = 0; e < VEC; e++) f[e] = __builtin_amdgcn_exp2f(fmaf(f[e], SMX_LOG2E, nlog2s));
			}
			R16 o = pack16<T>(f);
			if (FUSED && c == c_lab && t == t_lab) {   /* rnd(y) - 1 */
				unpack16<T>(o, f);
#pragma unroll
				for (int e = 0; e < VEC; e++)
					if (e == le) f[e] -= 1.0f;
				o = pack16<T>(f);
			}
			if (edge(c)) {
				const uint32_t pos = (uint32_t) (c * nt + t) * VEC;
				if (pos >= w.h && pos + VEC <= w.end) buf_store16_nt(rout, voff, (uint32_t) (c * nt) * 16u, o);
				else {
					T * p = reinterpret_cast<T *>(w.out);
					unpack16<T>(o, f);
#pragma unroll
					for (int e = 0; e < VEC; e++)
						if (pos + e >= w.h && pos + e < w.end) p[pos + e] = from_f<T>(f[e]);
				}
			}
			else buf_store16_nt(rout, voff, (uint32_t) (c * nt) * 16u, o);
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
		smx_rows<T, false, CH>(n_rows, n_cols, X, out, nullptr, nullptr, nullptr);                                     \
	}                                                                                                                  \
	extern "C" __global__ void __launch_bounds__(SMX_THREADS) softmax_cross_entropy_loss_##SUFFIX##_kernel_##VARIANT(  \
			int n_rows, int n_cols, T * logits, uint32_t * labels, float * loss, float * mean_loss) {                  \
		smx_rows<T, true, CH>(n_rows, n_cols, logits, logits, labels, loss, mean_loss);                                \
	}
#define SMX_ROWS_KERNELS(SUFFIX, PSUFFIX, T)                                                                           \
	SMX_ROWS_KERNEL(SUFFIX, PSUFFIX, T, rows, SMX_ROWS_CH)                                                             \
	SMX_ROWS_KERNEL(SUFFIX, PSUFFIX, T, wide_rows, SMX_WIDE_ROWS_CH)

SMX_ROWS_KERNELS(fp32, fp32_fp32, float)
SMX_ROWS_KERNELS(fp16, fp16_fp16, f16_t)
SMX_ROWS_KERNELS(bf16, bf16_bf16, bf16_t)
