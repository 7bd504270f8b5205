// sph_kernels.hpp -- host launchers of the gfx950 kernels (sph_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "sph_common.hpp"

namespace sph {

// state masks for the box state filter of the passes
constexpr int MASK_STEP = (1 << BOX_INIT) | (1 << BOX_RUN);
constexpr int MASK_RUN = (1 << BOX_RUN);
constexpr int MASK_INIT = (1 << BOX_INIT);
constexpr int MASK_ALL = (1 << BOX_INIT) | (1 << BOX_RUN) | (1 << BOX_DONE);

// build stage: plan, keys, sort, permutation, cell starts and lists of the
// building boxes
void launch_build_plan(const ArenaView &A, int force_mask, hipStream_t st);
void launch_keys(const ArenaView &A, int force_mask, hipStream_t st);
// cells != 0: also the cell starts from the sorted keys (radix-sort path)
void launch_permute(const ArenaView &A, int force_mask, int cells, hipStream_t st);
// arenas whose boxes all fit box_sort_fits: per-box counting sort in place of
// keys + radix sort + cell starts (same order)
void launch_box_sort(const ArenaView &A, int force_mask, int nbox, hipStream_t st);
bool box_sort_fits(int ncells, int n);
void launch_build_lists(const ArenaView &A, int force_mask, int fp32, hipStream_t st);
// advance != 0: also counts the step before this one (a plain step of a single
// box launched without k_box_step)
void launch_density(const ArenaView &A, int fp32, int state_mask, int unroll, hipStream_t st, int advance = 0);
void launch_grad(const ArenaView &A, int fp32, int state_mask, int diag, int unroll, hipStream_t st);
// step != 0: the stepping launch, which also takes each running slot's
// leapfrog step into the second state buffers (and carries the other live
// slots over); the runtime swaps the buffers after it
void launch_rates(const ArenaView &A, int fp32, int state_mask, int unroll, int step, hipStream_t st);
// the step pass as a launch of its own, after launch_rates(step = 0)
void launch_leapfrog(const ArenaView &A, int fp32, hipStream_t st);
void launch_box_step(const ArenaView &A, int nbox, hipStream_t st);
void launch_upload(const ArenaView &A, int off, int n, int field, const double *src, hipStream_t st);
// slots [off, off + n) to box b (-1: free); src: host-mapped r, v, m of the
// caller's particles i0 .. i0 + n - 1, or null
void launch_assign_slots(const ArenaView &A, int off, int n, int b, int i0, const double *src, hipStream_t st);
struct PutSpans {
    unsigned *dst[3];
    const unsigned *src[3];
    int words[3];
};
void launch_put(const PutSpans &P, hipStream_t st);
void launch_to_host(size_t n, const double *src, double *dst, hipStream_t st);
void launch_fetch(const ArenaView &A, int n, const int *inv, double *dst, int dyn_words, hipStream_t st);
void launch_download(const ArenaView &A, int box, int n, int field, double *dst, hipStream_t st);
void launch_inverse(const int *ids, int off, int n, int *inv, hipStream_t st);
// sorted partners of particle i in rows[i * pair_row()] on, their number in
// count[i]; over[0] is set when one has more than a row holds (then
// launch_pairs_long fills segments at offs instead), over[1] is cleared for
// launch_offsets_wrap, which sets it when the counts' sum passed 32 bits
int pair_row();
void launch_offsets_wrap(int n, const unsigned *offs, const unsigned *grand, unsigned *wrapped, hipStream_t st);
void launch_pairs(const ArenaView &A, int box, int n, unsigned *count, int *rows, unsigned *over, hipStream_t st);
void launch_pairs_long(const ArenaView &A, int box, int n, const int *inv, const unsigned *offs, int *jbuf, hipStream_t st);
// stride: pair_row() for rows, 0 for segments
void launch_pairs_emit(int n, const unsigned *offs, const unsigned *count, const int *jbuf, int stride,
                       long long *iap, long long cap, hipStream_t st);
void launch_separations(const ArenaView &A, int box, const int *inv, long long np,
                        const long long *iap, double *drij, double *rij, double *rsq, double *dv,
                        hipStream_t st);
void launch_lucy(long long np, const double *r, const double *dx, double h, int dim, double *w,
                 double *dwdx, hipStream_t st);
void launch_min_image(long long np, double *dr, double Lx, double Ly, hipStream_t st);
void launch_set_u(const ArenaView &A, int box, int n, const double *T, double T0, hipStream_t st);
// part: energy_blocks(n) block sums of the box's n slots
int energy_blocks(int n);
void launch_energy_now(const ArenaView &A, int box, int n, double2 *part, double *out3, hipStream_t st);
void launch_fp32_accumulate(long long n, const double *x, int unroll, double *out2, hipStream_t st);
// Device scratch of a rendering of n particles (n >= 1 counts; the arrays of
// one call, nothing in them need be cleared): SPLASH_HEAD_BYTES of head, n
// records twice, n keys and values, the sort's counters and C.max_cells + 1
// cell starts.
constexpr size_t SPLASH_HEAD_BYTES = 1024;
// Up to this many particles a rendering takes no launch for their largest
// smoothing length and at most 256 cells (one pass of the cell sort).
constexpr int64_t SPLASH_FEW = 1024;
struct SplashScratch {
    void *head;
    double4 *rec, *rec_sorted;
    unsigned *keys, *k_out, *v_out, *k_alt, *v_alt;
    void *sort_tmp;
    int *cs;
};
void launch_splash(long long n, const double *r, const double *m, const double *rho, const double *a,
                   const double *h, const SplashGrid &C, const SplashScratch &W, int nx, const double *x, int ny,
                   const double *y, double *Z, hipStream_t st);

}  // namespace sph
