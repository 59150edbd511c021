/* The launch rule of the softmax kernels against what their rows really take,
 * over storage types, lengths and places in memory: every row's window fits
 * the chunks that smx_rows_chunks promised, the output window starts on a
 * chunk, the chosen row kernel's waves hold the row, split rows have enough
 * slices, and a row sent to the "_long_rows" kernels has, by its own chunks,
 * as many per thread as they rely on and no more than they hold. Prints what
 * does not hold; the exit status is the number of such cases (at most 99). */
#include <stdio.h>
#include <stdint.h>

#include "kernel_geometry.h"

/* Which kernel, and which of the main kernels' paths (as they choose it), a
 * softmax call takes: an index into ROUTES of test_geometry.py. */
int smx_route(int n_rows, int n_cols, int elem, unsigned long long x, unsigned long long out) {
	const int kernel = smx_kernel_for(n_rows, n_cols, elem, x, out);
	if (kernel != SMX_MAIN) return kernel;
	const int aligned = ((x | out) & 15) == 0;
	if (elem == 1) return aligned && f8_smx_pf_ok(n_cols) ? SMX_MAIN : 7;
	const long nv = (long) n_cols * elem / 16, nch = (nv + SMX_THREADS - 1) / SMX_THREADS;
	if (!aligned || (long) n_cols * elem % 16 != 0) return 7;
	if (nch <= SMX_MAXCH && nch >= smx_regs_atleast(elem, SMX_MAXCH)) return SMX_MAIN;
	return nv < SMX_STREAM_MAX_CHUNKS ? 6 : 7;
}

/* every length up to 700 and around those where a row takes another kernel
 * (the sweep stops at each range's start), about every 2000th between */
static int next_length(int n) {
	static const int edges[] = {16300, 24500, 32700, 57300, 65400, 98200, 130900, 163700};
	const int width = 250, n_edges = (int) (sizeof(edges) / sizeof(edges[0]));
	if (n < 700) return n + 1;
	for (int i = 0; i < n_edges; i++) {
		if (n >= edges[i] && n < edges[i] + width) return n + 1;
		if (n < edges[i] && n + 1997 > edges[i]) return edges[i];
	}
	return n + 1997;
}

int main(void) {
	static const unsigned long long offsets[] = {0, 16, 64, 112, 2, 6, 34, 128, 4, 12, 8, 1, 5};
	static const int row_counts[] = {1, 7, 64, 200, 257, 5000, 1 << 25, (1 << 26) - 4, 1 << 26, 2147483647};
	const int n_counts = (int) (sizeof(row_counts) / sizeof(row_counts[0]));
	const int n_off = (int) (sizeof(offsets) / sizeof(offsets[0]));
	long bad = 0;
	for (int e = 1; e <= 4; e *= 2) {
		const int oe = e == 1 ? 2 : e;
		const long chunk = e == 1 ? 8 : 16;
		for (int i = 0; i < n_off * n_off; i++) {
			const unsigned long long x = 4096 + offsets[i / n_off], o = 8192 + offsets[i % n_off];
			if (x % e || o % oe) continue;
			for (int n = 1; n < 540000; n = next_length(n)) {
				const int bound = smx_rows_chunks(n, e, x, o);
				if (!bound) continue;
				const unsigned line = smx_rows_line(n, e, x, o);
				for (int r = 0; r < 130; r++) {
					const unsigned long long a = x + (unsigned long long) r * n * e, h = a & line;
					const long need = ((long) h + (long) n * e + chunk - 1) / chunk;
					const unsigned long long out = o + (unsigned long long) r * n * oe - (h / e) * oe;
					if (need > bound || (out & 15)) {
						if (bad++ < 10) printf("elem %d, %d columns, x+%llu out+%llu, row %d: %ld chunks of %d, out %llu\n", e, n, x - 4096, o - 8192, r, need, bound, out & 15);
					}
				}
				for (int k = 0; k < n_counts; k++) {
					const int kernel = smx_kernel_for(row_counts[k], n, e, x, o);
					if (kernel == SMX_SPLIT) {
						const int sets = smx_split_sets(n, e, x, o), s = smx_split_slices(row_counts[k], sets);
						const int per = (sets + s - 1) / s;
						if (row_counts[k] > SMX_SPLIT_ROWS || s < 1 || s > SMX_SPLIT_MAX || per > SMX_SPLIT_K || (long) s * per * SMX_THREADS < bound) {
							if (bad++ < 10) printf("elem %d, %d rows of %d columns: %d slices of %d sets\n", e, row_counts[k], n, s, per);
						}
					}
					if (kernel == SMX_LONG_ROWS) {
						const long nv = (long) n * e / 16, nch = (nv + SMX_THREADS - 1) / SMX_THREADS;
						if (e != 2 || ((x | o) & 15) || (long) n * e % 16 || nch < smx_regs_atleast(e, SMX_LONG_MAXCH) || nch > SMX_LONG_MAXCH) {
							if (bad++ < 10) printf("elem %d, %d long rows of %d columns, x+%llu out+%llu: %ld chunks per thread\n", e, row_counts[k], n, x - 4096, o - 8192, nch);
						}
					}
					if (kernel != SMX_ROWS && kernel != SMX_WIDE_ROWS) continue;
					const int ch = kernel == SMX_ROWS ? SMX_ROWS_CH : SMX_WIDE_ROWS_CH;
					const int g = smx_rows_waves(ch, row_counts[k], n, e, x, o);
					if (g < 1 || g > 16 || (long) g * 64 * ch < bound) {
						if (bad++ < 10) printf("elem %d, %d rows of %d columns: %d waves of %d chunks for %d\n", e, row_counts[k], n, g, ch, bound);
					}
					/* all rows in one launch, whose threads fit 32 bits */
					const long long threads = g == 1 ? ((long long) row_counts[k] + SMX_ROWS_PER_WG - 1) / SMX_ROWS_PER_WG * 64 * SMX_ROWS_PER_WG : (long long) row_counts[k] * 64 * g;
					if (threads >= 1ll << 32) {
						if (bad++ < 10) printf("elem %d, %d rows of %d columns: a launch of %lld threads\n", e, row_counts[k], n, threads);
					}
				}
			}
		}
	}
	/* rows of gigabytes: the "_any_rows" kernels' byte offsets and element
	 * indexes, which run up to four sets of chunks past the row, in 32 bits */
	static const int huge[] = {1 << 28, (1 << 29) + 3, (1 << 30) - 32769, (1 << 30) - 1, 1 << 30, (1 << 30) + 5, 2147483647 - 65600, 2147483647 - 64, 2147483647};
	for (int i = 0; i < (int) (sizeof(huge) / sizeof(huge[0])); i++) {
		for (int e = 2; e <= 4; e *= 2) {
			for (unsigned long long off = 0; off < 128; off += e) {
				const int n = huge[i];
				if (smx_kernel_for(1, n, e, 4096 + off, 8192 + off) != SMX_ANY_ROWS) continue;
				const long long last = ((long long) n * e + 127) / 16 + 1 + 4 * SMX_THREADS;
				if (last * 16 >= 1ll << 32 || last * (16 / e) >= 1ll << 31) {
					if (bad++ < 10) printf("elem %d, a row of %d columns +%llu: byte %lld, element %lld\n", e, n, off, last * 16, last * (16 / e));
				}
			}
		}
	}
	return bad > 99 ? 99 : (int) bad;
}
