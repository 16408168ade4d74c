/* cswap_test_hooks.h -- entry points that exist for the library's own tests only.
 *
 * They are exported by libcswap_hip.so but are not part of its interface: they
 * force failure paths that cannot be provoked from outside, or expose a host-side
 * calculation so that it can be checked for parts this build never runs on.
 * Nothing here has a counterpart in the reference.  Do not call them from
 * production code: their effect is process-wide.
 */
#ifndef CSWAP_TEST_HOOKS_H
#define CSWAP_TEST_HOOKS_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

/* The single-pass ZVC kernels wait, bounded, for status words of other workgroups.
 * spin_limit: how many times in all a wavefront asks again before it gives up
 * (0 = the default, some tens of milliseconds' worth).  skip, bits: 1 the count of the first
 * tile is never published, so that everything after it waits in vain; 2 (small form)
 * the first tile never says that it has its offset, so that whoever clears its count
 * waits in vain; 4 (small form) the last tile takes the workspace for unusable, as one does
 * that starts after another's wait has run out.  (0, 0) restores normal operation. */
void cswap_zvc_debug_set_lookback(unsigned spin_limit, unsigned skip);

/* Data workgroups the pipeline kernel of cswap_zvc_compress_fused is launched with for a
 * tensor of `tiles` tiles on a part with `compute_units` compute units (the scanner's
 * workgroup comes on top).  Host only. */
int cswap_test_zvc_stream_groups(int tiles, int compute_units);

/* 1 if the expansion of many short chunks that start on no 16-byte boundary stores a tensor of this many
 * bytes with the nontemporal hint.  Host only. */
int cswap_test_zvc_packed_hint(size_t bytes);

/* Which of the encoder's one-lane-per-block kernels a 3-D field of 32-bit elements with contiguous
 * x-rows runs where no other form takes it: 0 the general one, 1 the one for rows at any element,
 * 2 the general one with the nontemporal load hint; or an error code.  sy, sz: strides in elements
 * (0 = packed), misaligned: elements that the field starts past a 16-byte boundary.  3: as floats it
 * runs the form with four lanes per block on a part with `compute_units` of them (0: that form is not
 * asked about).  Host only. */
int cswap_test_zfp_encode_route(size_t nx, size_t ny, size_t nz, ptrdiff_t sy, ptrdiff_t sz, unsigned misaligned,
                                unsigned maxbits, int compute_units);

/* 1 if a 3-D field of floats with contiguous, 16-byte aligned x-rows is decoded by the form with four lanes per block on a
 * part with `compute_units` of them.  sy, sz: strides in elements (0 = packed).  Host only. */
int cswap_test_zfp_decode_quad(size_t nx, size_t ny, size_t nz, ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits,
                               int compute_units);

/* 1 if the decoder stores a field of 16-byte aligned rows with the nontemporal hint.  base: the field's address
 * (its alignment counts), pitch, plane: bytes from row to row and from plane to plane, bytes: of the field.  Host only. */
int cswap_test_zfp_store_hint(unsigned long long base, unsigned long long pitch, unsigned long long plane,
                              unsigned long long bytes, unsigned maxbits);

/* How the decoder's kernel for whole-word rates with one lane per block stores a 3-D field of floats with contiguous x-rows:
 * 0 row by row, 1 as runs through LDS, 2 as runs with the nontemporal hint; or an error code.  sy, sz: strides in
 * elements (0 = packed), base: the field's distance from a 128-byte line.  Host only. */
int cswap_test_zfp_decode_runs(size_t nx, size_t ny, size_t nz, ptrdiff_t sy, ptrdiff_t sz, unsigned base);

#ifdef __cplusplus
}
#endif
#endif
