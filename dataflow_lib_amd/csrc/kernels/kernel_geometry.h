/*
 * Geometry shared by the kernels and the launch-configuration library (plain
 * C on the host side), so both sides agree on paths, limits and layouts.
 *
 * RMSNorm vector path: each row is split over TPR threads ("a row slot");
 * thread t of the slot owns the 16-byte chunks t and t + TPR of the row
 * (RMS_CH = 2 chunks), so it always touches the same columns whatever row it
 * is on. TPR = 64 * ceil(ceil(chunks_per_row / 2) / 64), at most 1024.
 * RMSNorm element path (unaligned pointers, ragged rows, or rows longer than
 * 2 x 1024 chunks): TPR = 256 and a strided loop over the columns.
 * A workgroup holds `slots` row slots (blockDim.x = slots * TPR).
 */
#ifndef KERNEL_GEOMETRY_H
#define KERNEL_GEOMETRY_H

#define RMS_CH 2
#define RMS_MAX_TPR 1024
#define RMS_STREAM_TPR 256
/* element-path workgroups (one 256-thread row slot each) per CU, at most */
#define RMS_STREAM_GROUPS_PER_CU 8
/* LDS floats per row slot for the row reductions: [2 parities][32] */
#define RMS_CELLS_PER_SLOT 64
/* launch target: bytes of row loads outstanding per CU (each row slot keeps
 * its current and next row in flight) */
#define RMS_INFLIGHT_BYTES (64 * 1024)
/* dW finish kernel: RMS_FIN_COLS columns per workgroup, partial rows spread over its threads */
#define RMS_FINISH_THREADS 256
#define RMS_FIN_COLS 16   /* columns per finish workgroup */
/* fp32 partial rows for the two-pass dW reduction (16 MiB) */
#define RMS_DW_SCRATCH_FLOATS (4u << 20)

/* softmax / cross-entropy, main kernels: one workgroup per row, rows of up to
 * SMX_THREADS * SMX_MAXCH 16-byte chunks held in registers */
#define SMX_THREADS 1024
#define SMX_MAXCH 16
/* chunks per thread of the next row prefetched into LDS (9 x 16 KB); the
 * other SMX_MAXCH - SMX_PF chunks of the next row are prefetched into VGPRs */
#define SMX_PF 9
/* "_long_rows" kernels (16-bit): the same with more chunks per thread, the
 * next row's chunks past SMX_PF loaded at the top of their own row */
#define SMX_LONG_MAXCH 20

/* softmax / cross-entropy, "_rows" kernels: rows held by 1..16 waves,
 * SMX_ROWS_CH 16-byte chunks per thread; a row that one wave holds shares its
 * workgroup with SMX_ROWS_PER_WG - 1 others */
#define SMX_ROWS_CH 8
#define SMX_WIDE_ROWS_CH 16
#define SMX_ROWS_PER_WG 4

/* softmax / cross-entropy, "_split" kernels: few rows of many chunks, each over
 * up to SMX_SPLIT_MAX workgroups of SMX_THREADS, a slice being up to
 * SMX_SPLIT_K sets of SMX_THREADS chunks */
#define SMX_SPLIT_ROWS 64
#define SMX_SPLIT_MAX 16
#define SMX_SPLIT_K 4
#define SMX_SPLIT_XCDS 8

/* RoPE, head_dim <= 512. Vector path: one ROPE_SLOT_THREADS workgroup per
 * token at a time (persistent over tokens, next token prefetched), thread t
 * owning Q chunks t + 256 j (j < ROPE_QJ) and K chunks t + 256 j (j < ROPE_KJ)
 * of 16 bytes. Element path (unaligned rows or head_dim not a multiple of the
 * vector): one wave per token, ROPE_WAVES waves per workgroup. */
#define ROPE_MAX_HEAD_DIM 512
#define ROPE_WAVES 4
#define ROPE_SLOT_THREADS 256
#define ROPE_QJ 4
#define ROPE_KJ 2
/* vector path workgroups per CU at most: the RoPE kernels' registers allow
 * four, the fused KV-cache variant's three, and the launch takes the smaller
 * of this and what the kernel's registers leave resident */
#define ROPE_SLOT_WG_PER_CU 4
#define ROPE_WIDE_THREADS 512
#define ROPE_WIDE_WG_PER_CU 2

/* fp8 x 16-bit RMSNorm backward (fp8_ops.hip): rows in 8-element chunks
 * (8 bytes of each fp8 operand, 16 of each 16-bit one); a row slot of TPR
 * threads covers a row, thread t owning chunks t + TPR k (k < F8_CPT), so
 * rows of up to 8 * F8_CPT * 1024 columns take this path. bwd_x: 256-thread
 * workgroups, F8_BWDX_WG_PER_CU per CU; bwd_w: one workgroup of up to 1024
 * threads per CU whose slots add their partial rows in LDS. */
#define F8_CPT 2
#define F8_BWDX_WG_PER_CU 4

/* embedding / copy_to_seq_context: one wave per row, 4 waves per workgroup */
#define GS_WAVES 4

/* SwiGLU: grid-stride, one 512-thread workgroup per CU; per thread and
 * stream, U 16-byte chunks computed per step while the next U load. Measured
 * on MI355X at 8192 x 14336 bf16 over 1-4 workgroups of 256-1024 threads
 * per CU and U = 1, 2, 4: the forward (2 reads + 1 write) is fastest with
 * U = 2 (116 us), the backward (3 reads + 2 writes) with U = 1 (194 us
 * against 201 us with U = 2) */
#define SWIGLU_FWD_UNROLL 2
#define SWIGLU_BWD_UNROLL 1
#define SWIGLU_THREADS 512
#define SWIGLU_WG_PER_CU 1

#ifdef __HIPCC__
#define GEOM_FN __host__ __device__ __forceinline__
#define GEOM_CONST constexpr GEOM_FN
#else
#define GEOM_FN static inline
#define GEOM_CONST GEOM_FN
#endif

/* RMSNorm: 16-byte chunks per row, or 0 when the element path must be used */
GEOM_FN int rms_vec_chunks(int n_cols, int elem_bytes, unsigned long long ptr_or) {
	const int vec = 16 / elem_bytes;
	if (n_cols <= 0 || (n_cols % vec) != 0 || (ptr_or & 15ull) != 0ull) return 0;
	const int nv = n_cols / vec;
	if ((nv + RMS_CH - 1) / RMS_CH > RMS_MAX_TPR) return 0;
	return nv;
}

/* element path: threads per row slot. The dW modes (whose slots each keep an
 * n_cols-float partial row in LDS, so that only one slot fits per workgroup
 * once rows are long) use one slot of RMS_MAX_TPR threads from
 * RMS_STREAM_WIDE_COLS columns on */
#define RMS_STREAM_WIDE_COLS 4096
GEOM_FN int rms_stream_tpr(int dw_mode, int n_cols) {
	return (dw_mode && n_cols >= RMS_STREAM_WIDE_COLS) ? RMS_MAX_TPR : RMS_STREAM_TPR;
}

GEOM_FN int rms_tpr_for(int nv) {
	if (nv == 0) return RMS_STREAM_TPR;
	const int t = (nv + RMS_CH - 1) / RMS_CH;
	return ((t + 63) / 64) * 64;
}

/* Row slots per CU for the row-streaming RMSNorm ops: each slot keeps two rows
 * of `arrays` input rows in flight (the current one and the prefetched next
 * one), and about RMS_INFLIGHT_BYTES outstanding per CU measured best: more
 * concurrent row streams only add DRAM page misses. */
GEOM_FN long rms_slots_per_cu(int n_cols, long elem, int arrays) {
	const long per_slot = 2L * (long) n_cols * elem * (long) arrays;
	const long s = per_slot > 0 ? (long) RMS_INFLIGHT_BYTES / per_slot : 1;
	return s < 1 ? 1 : (s > 32 ? 32 : s);
}

/* Launch shape of the dW ops (bwd_w: arrays = 2, fused bwd: arrays = 3) for
 * n_rows >= 1 and n_cols >= 1: one workgroup per CU holding the CU's row
 * slots, so each workgroup writes one fp32 partial row. nv is
 * rms_vec_chunks(); max_lds the LDS bytes a workgroup may use; scratch_floats
 * the size of the partial-row buffer. Fills grid, block and dynamic LDS bytes
 * and returns 0, or -1 when the LDS cannot hold a row's partial sums, -2 when
 * one partial row does not fit the buffer. */
GEOM_FN int rms_dw_geometry(int n_rows, int n_cols, long elem, int nv, int arrays, long cu_count, long max_lds,
							long scratch_floats, unsigned * grid, unsigned * block, unsigned * lds) {
	const int tpr = (nv > 0) ? rms_tpr_for(nv) : rms_stream_tpr(1, n_cols);
	const long by_slots = rms_slots_per_cu(n_cols, elem, arrays);
	const long by_threads = (RMS_MAX_TPR / tpr) < 1 ? 1 : (RMS_MAX_TPR / tpr);
	int slots = (int) (by_slots < by_threads ? by_slots : by_threads);
	long bytes = 0;
	for (; slots >= 1; slots--) {
		const long colbuf = (nv > 0) ? (long) n_cols : (long) slots * n_cols;
		bytes = ((long) RMS_CELLS_PER_SLOT * slots + colbuf) * (long) sizeof(float);
		if (bytes <= max_lds) break;
	}
	if (slots < 1) return -1;
	const long max_parts = scratch_floats / (long) n_cols;
	if (max_parts < 1) return -2;
	long g = ((long) n_rows + slots - 1) / slots;
	if (g > cu_count) g = cu_count;
	if (g > max_parts) g = max_parts;
	*grid = (unsigned) g;
	*block = (unsigned) (slots * tpr);
	*lds = (unsigned) bytes;
	return 0;
}

/* fp8 x 16-bit RMSNorm backward: threads per row slot for the chunked path,
 * or 0 when rows must take the element path */
GEOM_FN int f8_row_tpr(int n_cols) {
	if (n_cols <= 0 || (n_cols % 8) != 0) return 0;
	const int t = (n_cols / 8 + F8_CPT - 1) / F8_CPT;
	const int tpr = ((t + 63) / 64) * 64;
	return tpr <= 1024 ? tpr : 0;
}

/* fp8 -> 16-bit softmax, long rows (fp8_ops.hip, softmax_fp8_pf): one
 * SMX_THREADS workgroup per CU holding the row in registers (F8_PF_PIECES
 * 8-byte pieces per thread) while the next row streams in, half into LDS and
 * half into registers; rows of a multiple of 16 columns up to
 * 8 * F8_PF_PIECES * SMX_THREADS. smx_kernel_for sends it more than 512 rows
 * of more than 8192 pieces; the shorter rows that reach the main kernel (2^26
 * of them and more) are left out by F8_PF_MIN_COLS */
#define F8_PF_PIECES 16
#define F8_PF_MIN_COLS 32768
GEOM_FN int f8_smx_pf_ok(int n_cols) {
	return n_cols >= F8_PF_MIN_COLS && (n_cols % 16) == 0 && n_cols / 8 <= F8_PF_PIECES * SMX_THREADS;
}

/* softmax register-row paths: the fewest chunks per thread, of its own, that a
 * row there has. The main kernels test it (smx); the "_long_rows" ones rely on
 * smx_kernel_for. */
GEOM_CONST int smx_regs_atleast(int elem_bytes, int maxch) {
	return maxch > SMX_MAXCH ? SMX_MAXCH + 1 : (elem_bytes == 4 ? 6 : 8);
}

/* softmax "_rows" kernels: what a row's window (SmxWindow) starts on, less one:
 * a 128-byte line, or 16 bytes where input and output lie differently within
 * their lines and where the line's other elements would not fit beside the
 * longest rows */
GEOM_FN unsigned smx_rows_line(int n_cols, int elem_bytes, unsigned long long x, unsigned long long out) {
	if (elem_bytes == 1) return n_cols > 8 * 1024 * SMX_WIDE_ROWS_CH - 128 ? 15u : 127u;
	return ((x ^ out) & 127ull) ? 15u : 127u;
}

/* The chunks (16 bytes, fp8 logits 8) a row's window can have, or 0 when input
 * and output lie differently within a chunk (fp8 logits: are not both 16-byte
 * aligned) */
GEOM_FN int smx_rows_chunks(int n_cols, int elem_bytes, unsigned long long x, unsigned long long out) {
	const long bytes = (long) n_cols * elem_bytes;
	const long chunk = elem_bytes == 1 ? 8 : 16;
	const long line = (long) smx_rows_line(n_cols, elem_bytes, x, out);
	if (elem_bytes == 1 ? ((x | out) & 15ull) != 0ull : ((x ^ out) & 15ull) != 0ull || ((x | out) % (unsigned) elem_bytes) != 0ull) return 0;
	const long off = (bytes | (long) (x & 127ull)) & line;   /* rows start at multiples of its lowest bit */
	const long slack = off == 0 ? 0 : (off % chunk == 0 ? line + 1 - chunk : line);
	return (int) ((bytes + slack + chunk - 1) / chunk);
}

/* Waves per row for a kernel of ch chunks per thread, or 0 when 16 waves do
 * not hold the row. */
GEOM_FN int smx_rows_waves(int ch, int n_rows, int n_cols, int elem_bytes, unsigned long long x, unsigned long long out) {
	const int chunks = smx_rows_chunks(n_cols, elem_bytes, x, out);
	if (chunks == 0 || chunks > 16 * 64 * ch) return 0;
	int g = (chunks + 64 * ch - 1) / (64 * ch);
	/* few rows: more waves each, until the chip has 8 per CU */
	while (g <= 8 && (long) n_rows * g < 2048 && chunks > 64 * g) g *= 2;
	return g;
}

/* "_split" kernels: a row's sets of SMX_THREADS chunks, and the workgroups a
 * row is split over: as many as give the chip a workgroup per CU */
GEOM_FN int smx_split_sets(int n_cols, int elem_bytes, unsigned long long x, unsigned long long out) {
	return (smx_rows_chunks(n_cols, elem_bytes, x, out) + SMX_THREADS - 1) / SMX_THREADS;
}
GEOM_FN int smx_split_slices(int n_rows, int sets) {
	int s = 256 / n_rows;
	if (s > SMX_SPLIT_MAX) s = SMX_SPLIT_MAX;
	if (s > sets) s = sets;
	if (s < 1) return 1;
	/* no more than the slices' sets need */
	const int k = (sets + s - 1) / s;
	return (sets + k - 1) / k;
}

/* streaming kernels: rows of 2^28 chunks (4 GiB), which 32-bit offsets do not
 * reach, less more than the four sets of chunks that a pass runs past the row */
#define SMX_STREAM_MAX_CHUNKS ((1 << 28) - (1 << 13))

/* Which kernel a softmax / cross-entropy call takes. In order:
 * - SMX_SPLIT for at most SMX_SPLIT_ROWS rows (half as many of 8 sets) of more
 *   than seven (fp32: eight) sets of SMX_THREADS chunks, in slices of at most
 *   SMX_SPLIT_K: two launches, so shorter rows stay on one CU (softmax 16 x
 *   65536 bf16 9.5 -> 7.9 us, but 16 x 50257 8.9 -> 10.6, fp32 64 x 32000 7.6
 *   -> 8.5), and so do more rows, whose slices are long and
 *   whose maxima are then found too often over (128 x 128256 20.8 us either
 *   way, fp16 21.9 -> 27.0);
 * - SMX_LONG_ROWS for aligned 16-bit rows of 17 to 20 chunks per thread, by the
 *   row's own chunks, which that kernel counts and relies on
 *   (smx_regs_atleast), not by its window's: a window may have up to seven
 *   more, and with 16 chunks per thread of its own (131,024 to 131,072
 *   columns) the row is the main kernel's;
 * - SMX_ROWS (8 chunks per thread) while the row needs at most 8 waves (16-bit)
 *   or 4 (fp32), so that at least two rows share a CU, and up to 16 waves when
 *   no two rows have to share one (16 x 50257 bf16: 9.4 us, wide 11.7);
 * - SMX_WIDE_ROWS (16 chunks) up to twice that: 1024 x 50257 bf16 41.4 us
 *   against 50.7 with 13 waves of 8 chunks, of which a CU holds one workgroup;
 *   fp32 8192 x 16384 184.2 against 199.9;
 * - rows of more than 8192 chunks, and fp32 rows of more than 6144 when there
 *   are many of them, go to the main kernel, which overlaps one row with the
 *   next on the same CU (1024 x 100000 bf16 78.5 us, wide 98.3; 4096 x 32000
 *   fp32 169.4, wide 184.1), unless they are unaligned, which it does not
 *   hold in registers (1024 x 128257 bf16 557 us, wide 116);
 * - unaligned rows of more than 16 chunks per thread to SMX_ANY_ROWS, which
 *   streams them as the main kernel does aligned ones, but for rows of
 *   SMX_STREAM_MAX_CHUNKS chunks and more, which go element by element in the
 *   main kernel;
 * - rows that would make a launch of the row kernels, which take all rows at
 *   once, 2^32 threads or more (from 2^26 rows of one wave on), to the main
 *   kernel, which walks them;
 * - fp8 logits the same way: 12 waves of 8 chunks still share a CU with
 *   another row (1024 x 48000 27.7 us, wide 30.3; 1024 x 50256 43.0, wide
 *   31.6), and the main kernel overlaps rows from some 512 on (300 x 128256
 *   41.4 us, wide 34.7; 1024 x 100000 68.4, wide 78.9).
 */
#define SMX_MAIN 0
#define SMX_ROWS 1
#define SMX_WIDE_ROWS 2
#define SMX_LONG_ROWS 3
#define SMX_SPLIT 4
#define SMX_ANY_ROWS 5
#define SMX_FEW_ROWS 256   /* no more rows than CUs: each row has a CU to itself */
GEOM_FN int smx_kernel_for(int n_rows, int n_cols, int elem_bytes, unsigned long long x, unsigned long long out) {
	const int chunks = smx_rows_chunks(n_cols, elem_bytes, x, out);
	const int few = n_rows <= SMX_FEW_ROWS;
	/* the main kernel holds the row in registers too */
	const int main_regs = ((x | out) & 15ull) == 0ull && ((long) n_cols * elem_bytes) % 16 == 0;
	if (chunks > (elem_bytes == 4 ? 8 : 7) * SMX_THREADS && n_rows <= (chunks > 8 * SMX_THREADS ? SMX_SPLIT_ROWS : SMX_SPLIT_ROWS / 2)) {
		const int sets = (chunks + SMX_THREADS - 1) / SMX_THREADS;
		const int slices = smx_split_slices(n_rows, sets);
		if ((sets + slices - 1) / slices <= SMX_SPLIT_K) return SMX_SPLIT;
	}
	const long own = (long) n_cols * elem_bytes / 16;
	if (main_regs && elem_bytes == 2 && own > 1024 * SMX_MAXCH && own <= 1024 * SMX_LONG_MAXCH) return SMX_LONG_ROWS;
	if (chunks == 0) return SMX_MAIN;
	if (chunks > 1024 * SMX_WIDE_ROWS_CH) return (main_regs || elem_bytes == 1 || chunks >= SMX_STREAM_MAX_CHUNKS) ? SMX_MAIN : SMX_ANY_ROWS;
	const int waves = (chunks + 64 * SMX_ROWS_CH - 1) / (64 * SMX_ROWS_CH);   /* at most: the wide kernel takes half */
	if (64ll * waves * ((long long) n_rows + SMX_ROWS_PER_WG - 1) >= 1ll << 32) return SMX_MAIN;
	if (elem_bytes == 1) {
		if (chunks <= (few ? 1024 : 768) * SMX_ROWS_CH) return SMX_ROWS;
		return (chunks <= 1024 * SMX_ROWS_CH || n_rows <= 2 * SMX_FEW_ROWS || !f8_smx_pf_ok(n_cols)) ? SMX_WIDE_ROWS : SMX_MAIN;
	}
	if (chunks <= 1024 * SMX_ROWS_CH && (few || chunks <= (elem_bytes < 4 ? 512 : 256) * SMX_ROWS_CH)) return SMX_ROWS;
	if (!main_regs) return SMX_WIDE_ROWS;
	if (elem_bytes == 4 && chunks > 6144 && n_rows >= 8 * SMX_FEW_ROWS) return SMX_MAIN;
	return chunks <= 1024 * SMX_ROWS_CH ? SMX_WIDE_ROWS : SMX_MAIN;
}

/* RoPE vector path: fp8 rows are half as long as bf16 ones, so the main kernel
 * takes two tokens at a time when their Q and K chunks fit its registers. */
#define ROPE_TG_QJ 2   /* Q chunks per thread in a step of several tokens */
GEOM_FN int rope_fp8_pairs(int model_dim, int kv_dim) {
	return 2 * (model_dim / 16) <= ROPE_SLOT_THREADS * ROPE_TG_QJ && 2 * (kv_dim / 16) <= ROPE_SLOT_THREADS * ROPE_KJ;
}

/* Tokens per step of the "_multi" kernels, or 1 where the main kernel runs:
 * four, else two, that fit ROPE_TG_QJ Q chunks per thread, from a step per CU
 * on; else two of ROPE_QJ. A step's fp64 sin/cos tables take a wave about a
 * microsecond, which rows of 1-2 KB do not hide: 8192 x (16 + 4) x 64 bf16 15.0
 * -> 8.9 us with four (42 MB: 4.7 TB/s), 16384 x (8 + 8) x 64 26.2 -> 13.5,
 * with the KV cache 22.2 -> 12.9 and 43.7 -> 21.8; two tokens of 8 KB rows gain
 * once every CU has several steps (x (32 + 8) x 128, main -> two: 1024 tokens
 * 5.4 -> 5.5 us, 1531 7.4 -> 6.6, 2048 9.4 -> 8.6, 8192 29.6 -> 29.2, with the
 * KV cache 7.1 -> 7.5, 9.4 -> 8.9, 12.3 -> 10.8, 37.8 -> 36.1). fp8 takes two
 * in its main kernel already. */
GEOM_FN int rope_tokens_per_group(long n_tokens, int model_dim, int kv_dim, int elem_bytes) {
	const int nvq = model_dim * elem_bytes / 16, nvk = kv_dim * elem_bytes / 16;
	int tg = 4;
	for (; tg > 1; tg /= 2) {
		if (tg * nvq <= ROPE_SLOT_THREADS * ROPE_TG_QJ && tg * nvk <= ROPE_SLOT_THREADS * ROPE_KJ && n_tokens >= tg * 256L) break;
	}
	if (elem_bytes == 1) return tg == 4 ? 4 : 1;
	if (tg == 1 && 2 * nvq <= ROPE_SLOT_THREADS * ROPE_QJ && 2 * nvk <= ROPE_SLOT_THREADS * ROPE_KJ && n_tokens >= 1280) return 2;
	return tg;
}

/* RoPE: whether the vector (slot) path applies with workgroups of `threads` */
GEOM_FN int rope_slot_ok(int threads, int model_dim, int kv_dim, int head_dim, int elem_bytes, unsigned long long ptr_or) {
	const int vec = 16 / elem_bytes;
	if ((head_dim % vec) != 0 || (ptr_or & 15ull) != 0ull) return 0;
	return (model_dim / vec) <= threads * ROPE_QJ && (kv_dim / vec) <= threads * ROPE_KJ;
}

#endif
