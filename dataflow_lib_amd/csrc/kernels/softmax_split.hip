/*
 * Softmax and fused softmax + cross-entropy of a few long rows (the "_split"
 * kernels, smx_kernel_for): each row is split over up to SMX_SPLIT_MAX
 * workgroups, since a row on one CU takes 17-24 us of that CU's arithmetic
 * whatever the other 255 do.
 *
 * Two launches instead of workgroups that wait for each other: the first finds
 * the row's max in every workgroup (all of them read the row, from the L2 of
 * the XCD that they share, which costs less than another launch), sums the
 * exponentials of its own slice and leaves max and sums in the code object's
 * memory; the second adds the slices' sums in order and writes its slice's
 * outputs. Same arithmetic as the other softmax kernels. Measured on MI355X,
 * one CU per row -> split, bf16 softmax / fused loss:
 *    1 x 128256  16.4 -> 8.5 us   22.5 ->  9.4 us
 *   16 x 128256  18.7 -> 9.6 us   24.4 -> 11.2 us
 *   64 x 128256  19.5 -> 13.8 us  25.2 -> 16.9 us
 * of which 7.4 us are what two launches take.
 * A slice is `k` sets of SMX_THREADS chunks (chunk = 16 bytes, fp8 8).
 */
struct SmxSplitPart {
	float m, sd, sx, unused;
};
/* a row's parts in two whole lines: where the compiler's placement had them in
 * three, 16 x 128256 bf16 took 10.05 us instead of 9.87 (and on a page, with
 * g_smx_group_done: fused 11.47 us on 256 bytes, 11.20 on 4096) */
__device__ __attribute__((aligned(4096))) SmxSplitPart g_smx_split[SMX_SPLIT_ROWS * SMX_SPLIT_MAX];
__device__ float g_smx_split_xlab[SMX_SPLIT_ROWS];   /* a row's labelled logit */

/* rounded differences of a chunk in the output type */
template <typename TO, int VEC>
__device__ __forceinline__ void smx_split_round(const float (&x_m)[VEC], float (&d)[VEC]) {
	if constexpr (sizeof(TO) == 4) {
#pragma unroll
		for (int e = 0; e < VEC; e++) d[e] = x_m[e];
	}
	else {
#pragma unroll
		for (int e = 0; e < VEC; e += 2) smx_round2<TO>(x_m + e, d + e);
	}
}

/* What a workgroup of either launch works on. Workgroups are dealt to the
 * XCDs round-robin: a row's slices go to one XCD. */
template <typename T, typename TO>
struct SmxSplit {
	using C = SmxChunk<T>;
	static constexpr int VEC = C::N;
	static constexpr int CB = VEC * (int) sizeof(T), OB = VEC * (int) sizeof(TO);
	int slices, k, row, slice, tid;
	SmxWindow w;
	__device__ __forceinline__ SmxSplit(int n_rows, int n_cols, const T * X, TO * out) {
		const int sets = smx_split_sets(n_cols, (int) sizeof(T), (unsigned long long) (uintptr_t) X, (unsigned long long) (uintptr_t) out);
		slices = smx_split_slices(n_rows, sets);
		k = (sets + slices - 1) / slices;
		const int xcd = (int) blockIdx.x % SMX_SPLIT_XCDS, local = (int) blockIdx.x / SMX_SPLIT_XCDS;
		row = local / slices * SMX_SPLIT_XCDS + xcd;
		slice = local % slices;
		tid = (int) threadIdx.x;
		if (row < n_rows) w = smx_window<T, TO>(X, out, n_cols, row);
	}
	__device__ __forceinline__ uint32_t chunk(int set) const { return (uint32_t) (set * SMX_THREADS + tid); }
	/* values of a loaded chunk; elements outside the row are -inf */
	__device__ __forceinline__ void values(const typename C::raw & x, int set, float (&f)[VEC]) const {
		C::unpack(x, f);
		const uint32_t pos = chunk(set) * VEC;
		if (pos < w.h || pos + VEC > w.end) {
#pragma unroll
			for (int e = 0; e < VEC; e++)
				if (pos + e < w.h || pos + e >= w.end) f[e] = -__builtin_inff();
		}
	}
};

template <typename T, typename TO, bool FUSED>
__device__ __forceinline__ void smx_split_part(int n_rows, int n_cols, const T * X, TO * out, const uint32_t * labels) {
	using S = SmxSplit<T, TO>;
	using C = SmxChunk<T>;
	constexpr int VEC = S::VEC;
	constexpr int U = 8;
	__shared__ float mcells[16];
	__shared__ float scells[32];
	const S s(n_rows, n_cols, X, out);
	if (s.row >= n_rows) return;
	const int lane = s.tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(s.tid >> 6);
	const __amdgpu_buffer_rsrc_t rin = make_rsrc(s.w.in, (uint32_t) s.w.chunks * S::CB);
	const int sets = (s.w.chunks + SMX_THREADS - 1) / SMX_THREADS;
	typename C::raw mine[SMX_SPLIT_K];
#pragma unroll
	for (int j = 0; j < SMX_SPLIT_K; j++)
		if (j < s.k) mine[j] = C::load_again(rin, s.chunk(s.slice * s.k + j) * S::CB, 0);
	float m = -__builtin_inff();
	for (int c0 = 0; c0 < sets; c0 += U) {
		typename C::raw v[U];
#pragma unroll
		for (int j = 0; j < U; j++) v[j] = C::load_again(rin, s.chunk(c0 + j) * S::CB, 0);   /* past the window: zeros, masked below */
#pragma unroll
		for (int j = 0; j < U; j++) {
			float f[VEC];
			s.values(v[j], c0 + j, f);
#pragma unroll
			for (int e = 0; e < VEC; e++) m = __builtin_elementwise_maximum(m, f[e]);
		}
	}
	m = waves_max(m, mcells, SMX_THREADS / 64, wave, lane);

	const uint32_t lab = FUSED ? load_scalar(labels + s.row) : 0xffffffffu;
	const uint32_t lab_pos = (FUSED && lab < (uint32_t) n_cols) ? lab + s.w.h : 0xffffffffu;
	float sd = 0.0f, sx = 0.0f;
#pragma unroll
	for (int j = 0; j < SMX_SPLIT_K; j++) {
		if (j < s.k) {
			const int set = s.slice * s.k + j;
			float f[VEC], x_m[VEC], d[VEC];
			s.values(mine[j], set, f);
#pragma unroll
			for (int e = 0; e < VEC; e++) x_m[e] = f[e] - m;
			smx_split_round<TO, VEC>(x_m, d);
			const uint32_t pos = s.chunk(set) * VEC;
#pragma unroll
			for (int e = 0; e < VEC; e++) {
				sd += exp_fast(d[e]);
				/* the loss sum: unrounded differences, without the label's column */
				if (FUSED) {
					if (pos + e == lab_pos) g_smx_split_xlab[s.row] = f[e];
					else sx += exp_fast(x_m[e]);
				}
			}
		}
	}
	waves_sum2(sd, sx, scells, SMX_THREADS / 64, wave, lane);
	if (s.tid == 0) g_smx_split[s.row * SMX_SPLIT_MAX + s.slice] = SmxSplitPart{m, sd, sx, 0.0f};
}

template <typename T, typename TO, bool FUSED>
__device__ __forceinline__ void smx_split_out(int n_rows, int n_cols, const T * X, TO * out, const uint32_t * labels, float * loss, float * mean_loss) {
	using S = SmxSplit<T, TO>;
	using C = SmxChunk<T>;
	constexpr int VEC = S::VEC;
	const S s(n_rows, n_cols, X, out);
	if (s.row >= n_rows) return;
	const int lane = s.tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(s.tid >> 6);
	const __amdgpu_buffer_rsrc_t rin = make_rsrc(s.w.in, (uint32_t) s.w.chunks * S::CB);
	const __amdgpu_buffer_rsrc_t rout = make_rsrc(s.w.out, (uint32_t) s.w.chunks * S::OB);
	typename C::raw x[SMX_SPLIT_K];
#pragma unroll
	for (int j = 0; j < SMX_SPLIT_K; j++)
		if (j < s.k) x[j] = C::load(rin, s.chunk(s.slice * s.k + j) * S::CB, 0);
	/* the row's max and sums, every wave for itself, in slice order */
	const SmxSplitPart p = g_smx_split[s.row * SMX_SPLIT_MAX + ((lane & 15) < s.slices ? (lane & 15) : 0)];
	const bool live = (lane & 15) < s.slices;
	const float m = readlane_f32(p.m, 0);
	const float sd = row16_sum(live ? p.sd : 0.0f);
	const float sx = row16_sum(live ? p.sx : 0.0f);
	const float inv = 1.0f / sd;
	const uint32_t lab = FUSED ? load_scalar(labels + s.row) : 0xffffffffu;
	const bool lab_ok = FUSED && lab < (uint32_t) n_cols;
	const uint32_t lab_pos = lab_ok ? lab + s.w.h : 0xffffffffu;
	SmxGroup rows;   /* one group of all rows */
	rows.first = rows.index = 0;
	rows.count = n_rows;
	rows.n_groups = 1;
	unsigned arrived = 0u;
	const bool owner = FUSED && s.slice == 0 && wave == 0 && loss;
	if (owner) {
		if (lane == 0) store_loss(loss, s.row, lab_ok ? fused_loss(sx, m, g_smx_split_xlab[s.row]) : __builtin_nanf(""));
		if (mean_loss) arrived = smx_arrive(g_smx_group_done, lane);
	}
#pragma unroll
	for (int j = 0; j < SMX_SPLIT_K; j++) {
		if (j < s.k) {
			const int set = s.slice * s.k + j;
			float f[VEC], d[VEC];
			s.values(x[j], set, f);
#pragma unroll
			for (int e = 0; e < VEC; e++) f[e] -= m;
			smx_split_round<TO, VEC>(f, d);
#pragma unroll
			for (int e = 0; e < VEC; e++) f[e] = exp_fast(d[e]) * inv;
			R16 o = pack16<TO>(f);
			const uint32_t pos = s.chunk(set) * VEC;
			if (FUSED && lab_pos - pos < (uint32_t) VEC) {   /* rnd(y) - 1 */
				unpack16<TO>(o, f);
#pragma unroll
				for (int e = 0; e < VEC; e++)
					if (pos + e == lab_pos) f[e] -= 1.0f;
				o = pack16<TO>(f);
			}
			if (pos >= s.w.h && pos + VEC <= s.w.end) buf_store16_nt(rout, s.chunk(set) * S::OB, 0, o);
			else {
				TO * q = reinterpret_cast<TO *>(s.w.out);
				unpack16<TO>(o, f);
#pragma unroll
				for (int e = 0; e < VEC; e++)
					if (pos + e >= s.w.h && pos + e < s.w.end) q[pos + e] = from_f<TO>(f[e]);
			}
		}
	}
	if (owner && mean_loss) smx_rows_mean(rows, arrived, 1, n_rows, loss, mean_loss, lane);
}

#define SMX_SPLIT_SOFTMAX(PSUFFIX, T, TO)                                                                              \
	extern "C" __global__ void __launch_bounds__(SMX_THREADS) softmax_##PSUFFIX##_kernel_split(int n_rows, int n_cols, \
			T * X, TO * out) {                                                                                         \
		smx_split_part<T, TO, false>(n_rows, n_cols, X, out, nullptr);                                                 \
	}                                                                                                                  \
	extern "C" __global__ void __launch_bounds__(SMX_THREADS) softmax_##PSUFFIX##_kernel_split_out(int n_rows,         \
			int n_cols, T * X, TO * out) {                                                                             \
		smx_split_out<T, TO, false>(n_rows, n_cols, X, out, nullptr, nullptr, nullptr);                                \
	}
#define SMX_SPLIT_KERNELS(SUFFIX, PSUFFIX, T)                                                                          \
	SMX_SPLIT_SOFTMAX(PSUFFIX, T, T)                                                                                   \
	extern "C" __global__ void __launch_bounds__(SMX_THREADS) softmax_cross_entropy_loss_##SUFFIX##_kernel_split(      \
			int n_rows, int n_cols, T * logits, uint32_t * labels, float * loss, float * mean_loss) {                  \
		smx_split_part<T, T, true>(n_rows, n_cols, logits, logits, labels);                                            \
	}                                                                                                                  \
	extern "C" __global__ void __launch_bounds__(SMX_THREADS) softmax_cross_entropy_loss_##SUFFIX##_kernel_split_out(  \
			int n_rows, int n_cols, T * logits, uint32_t * labels, float * loss, float * mean_loss) {                  \
		smx_split_out<T, T, true>(n_rows, n_cols, logits, logits, labels, loss, mean_loss);                            \
	}

SMX_SPLIT_KERNELS(fp32, fp32_fp32, float)
SMX_SPLIT_KERNELS(fp16, fp16_fp16, f16_t)
SMX_SPLIT_KERNELS(bf16, bf16_bf16, bf16_t)
SMX_SPLIT_SOFTMAX(fp8e4m3_fp16, fp8e4m3_t, f16_t)
SMX_SPLIT_SOFTMAX(fp8e4m3_bf16, fp8e4m3_t, bf16_t)
SMX_SPLIT_SOFTMAX(fp8e5m2_fp16, fp8e5m2_t, f16_t)
SMX_SPLIT_SOFTMAX(fp8e5m2_bf16, fp8e5m2_t, bf16_t)
