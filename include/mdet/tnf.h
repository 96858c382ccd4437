/*
 * mdet TNF path: C ABI of the MI355X (gfx950) implementation of MdeT's
 * tetranucleotide-frequency contig-graph path.
 *
 * The reference has no library boundary: its path is a set of functions and
 * globals inside one CUDA program.  Each entry point below names the reference
 * interface it replaces (file:line in jonathanavc/MdeT).
 *
 * Conventions
 *   - Every function returns 0 (MDET_OK) or a negative MDET_E_* code; the
 *     message of the last failure on the calling thread is mdet_last_error().
 *     (The reference prints and exit(1)s, cuda/Cuda2.cu:341-354; the C++
 *     drop-in in mdet/tnf.hpp restores that behaviour.)
 *   - Arrays named *_dev are device (HBM) pointers; all others are host.
 *   - A context owns one HIP stream and the scratch memory of the calls made
 *     on it; one host thread drives a context at a time.  Calls are ordered
 *     on the context's stream; results are valid after mdet_ctx_sync().
 *   - Plain C types only: no HIP or torch types cross this boundary.
 */
#ifndef MDET_TNF_H
#define MDET_TNF_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define MDET_OK 0
#define MDET_E_INVALID (-1)  /* bad argument */
#define MDET_E_HIP (-2)      /* HIP runtime error (message names the call) */
#define MDET_E_NOMEM (-3)    /* device allocation failed */
#define MDET_E_RANGE (-4)    /* input outside the supported domain */
#define MDET_E_STATE (-5)    /* object not ready for this call */
#define MDET_E_CAPACITY (-6) /* caller buffer too small (message says how big) */

#define MDET_NTNF 136 /* canonical tetranucleotides per TNF row */

/* ------------------------------------------------------------- general -- */
const char *mdet_version(void);
/* Message of the last failed call on this thread ("" if none). */
const char *mdet_last_error(void);

/* The 136 column 4-mers of a TNF row, 4 chars each, in the reference's order
 * (openmp/TNF.cpp:14-24 TN[]); out needs 545 bytes. */
int mdet_tnf_columns(char *out, uint64_t cap);
/* For each 2-bit 4-mer code (A=0 C=1 G=2 T=3, first base in the low bits:
 * code = b0 | b1<<2 | b2<<4 | b3<<6) the TNF column it counts into.
 * Replaces the lookup table TNmap_d (cuda/Cuda2.cu:149-159), re-derived for
 * this library's base code. */
int mdet_column_of_code(int16_t *out256);

/* ------------------------------------------------------------- context -- */
typedef struct mdet_ctx mdet_ctx;
/* One context per (device, host thread).  Replaces the implicit per-thread
 * device binding of cuda/Cuda2.cu:890-891. */
int mdet_ctx_create(int device, mdet_ctx **out);
int mdet_ctx_destroy(mdet_ctx *ctx);
int mdet_ctx_sync(mdet_ctx *ctx);
/* The context's hipStream_t, as an opaque pointer. */
void *mdet_ctx_stream(mdet_ctx *ctx);

/* Device memory and copies on the context's stream, for callers without
 * HIP headers (the C++ drop-in, Python tests).  Copies are synchronous. */
int mdet_dev_alloc(mdet_ctx *ctx, uint64_t bytes, void **out_dev);
int mdet_dev_free(mdet_ctx *ctx, void *dev);
int mdet_copy_h2d(mdet_ctx *ctx, void *dst_dev, const void *src, uint64_t bytes);
int mdet_copy_d2h(mdet_ctx *ctx, void *dst, const void *src_dev, uint64_t bytes);
/* Free and total device memory of the context's device (hipMemGetInfo). */
int mdet_dev_mem_info(mdet_ctx *ctx, uint64_t *free_bytes, uint64_t *total_bytes);

/* ---------------------------------------------------------- host ingest -- */
/* FASTA with kseq semantics (extra/kseq.h:190-229, as used by
 * openmp/TNF.cpp:102-143): multi-line records joined, empty lines skipped,
 * a trailing '\r' stripped per line, name = header up to the first blank.
 * Pass 1 counts records and sequence bytes; pass 2 fills
 * name_off/name_len[n_records] (offsets into buf), the joined sequences into
 * seq_out and seq_off[n_records+1]. */
int mdet_fasta_scan(const char *buf, uint64_t size, uint64_t *n_records, uint64_t *total_seq);
int mdet_fasta_read(const char *buf, uint64_t size, uint64_t n_records, uint64_t *name_off,
                    uint64_t *name_len, char *seq_out, uint64_t *seq_off);

/* 2-bit packing.  Bases of all contigs are concatenated (contig r occupies
 * global bases [seq_off[r], seq_off[r+1])), 16 per uint32 word, base p at
 * bits 2*(p%16) of word p/16.  Every byte that is not A/C/G/T/a/c/g/t is an
 * N: stored as 0 and listed in runs[2*k], runs[2*k+1] = [start, end) global
 * base ranges, sorted and disjoint.  On MDET_E_CAPACITY *n_runs holds the
 * capacity needed.  The packed stream replaces the char buffer the reference
 * scans (cuda/Cuda2.cu:1826-1844; get_TNF's seqs_d, cuda/Cuda.cu:222). */
int mdet_pack_ascii(const char *seq, const uint64_t *seq_off, uint64_t n, uint32_t *packed,
                    uint64_t packed_words, uint64_t *runs, uint64_t runs_cap, uint64_t *n_runs);

/* The same packing on the device: seq_dev[n_bases] are the joined ASCII bases
 * of all contigs (device memory), packed_dev receives ceil(n_bases/16) words
 * and runs_dev the N runs (runs_cap runs of two uint64), both identical to
 * mdet_pack_ascii's; *n_runs (host) receives the run count, and
 * MDET_E_CAPACITY is returned if it exceeds runs_cap (call again with a larger
 * buffer).  Replaces the host walk over the FASTA bytes of
 * cuda/Cuda2.cu:1436-1572 / 1833-1844 (the reference keeps the text and scans
 * it per contig; here the 2-bit stream is built where it is read). */
int mdet_pack_ascii_dev(mdet_ctx *ctx, const char *seq_dev, uint64_t n_bases, uint32_t *packed_dev,
                        uint64_t packed_words, uint64_t *runs_dev, uint64_t runs_cap, uint64_t *n_runs);

/* log10(min(length, 500000)) in FP64, the per-contig size feature of the
 * pair model (cuda/Cuda2.cu:1535 logSizes).  Computed with the host libm, as
 * the reference does while parsing: the device log10 differs from it in the
 * last bit for ~1.7% of lengths in [1500, 500000], and the FP64 tie-breaker
 * of the pair stage must see the same values as the reference. */
int mdet_logsize_host(const uint64_t *lengths, uint64_t n, double *out);

/* ------------------------------------------------------------ generator -- */
/* Seeded order-3 Markov metagenome (no reference counterpart: the reference
 * ships no data).  Deterministic for a config on any machine/thread count. */
typedef struct mdet_gen_config {
    uint64_t seed;
    uint32_t n_genomes;
    uint32_t n_run_max;  /* N runs have length U{1..n_run_max} */
    double len_median;   /* log-normal contig lengths ... */
    double len_sigma;
    double len_min;      /* ... clipped to [len_min, len_max] */
    double len_max;
    double n_frac;       /* expected fraction of N bases */
    double gc_lo, gc_hi; /* per-genome GC weight ~ U[gc_lo, gc_hi] */
} mdet_gen_config;

int mdet_gen_lengths(const mdet_gen_config *cfg, uint64_t n, uint64_t *lengths, uint32_t *genome);
/* Packs contigs 0..n-1 at base_off[0..n] (lengths as mdet_gen_lengths gives),
 * N runs as in mdet_pack_ascii.  threads <= 0: hardware concurrency (max 16). */
int mdet_gen_packed(const mdet_gen_config *cfg, uint64_t n, const uint64_t *base_off, uint32_t *packed,
                    uint64_t packed_words, uint64_t *runs, uint64_t runs_cap, uint64_t *n_runs,
                    int threads);
/* One contig as ASCII (A/C/G/T/N), identical bases to mdet_gen_packed. */
int mdet_gen_ascii(const mdet_gen_config *cfg, uint64_t contig, char *out, uint64_t len);

/* ------------------------------------------------------------- counting -- */
/* TNF of n contigs from the 2-bit packed stream (device arrays):
 *   packed_dev[ceil(n_bases/16)], runs_dev[2*n_runs] (may be NULL if
 *   n_runs == 0), base_off_dev[n+1] (uint64 global base offsets).
 * For each contig, every window of 4 consecutive bases of the contig that
 * contains no N counts +1 in its canonical column; counts_dev[n*136]
 * (optional, may be NULL) receives the integer counts and tnf_dev[n*136]
 * the row c / sqrt(sum c^2) rounded once from FP64 to FP32 (0/0 = NaN for a
 * contig with no valid window, as openmp/TNF.cpp:208-217).
 * Replaces TNF_CAL (cuda/Cuda2.cu:1823-1864), get_TNF (cuda/Cuda.cu:222-269)
 * and launch_tnf_kernel (cuda/Cuda.cu:1706-1736). */
int mdet_tnf_count(mdet_ctx *ctx, const uint32_t *packed_dev, uint64_t n_bases, const uint64_t *runs_dev,
                   uint64_t n_runs, const uint64_t *base_off_dev, uint32_t n, uint32_t *counts_dev,
                   float *tnf_dev);

/* Same result as mdet_tnf_count, allocating nothing (no hipMalloc, hipFree or
 * allocating library call, no host synchronisation).  No counterpart in the
 * reference: it is for callers that cannot allocate device memory (code under
 * HIP graph capture, tight serving loops, harnesses that forbid it).
 * counts_dev is required here.  The per-chunk metadata lives in a static
 * device array of 2^21 entries (64 MiB, held on every device the library runs
 * on until the process ends), so n_bases may be at most 2^21 x 16384 =
 * 34,359,738,368 (MDET_E_RANGE beyond).  base_off is not read back: it must be
 * non-decreasing with base_off[n] <= n_bases, or the counts are undefined (no
 * access leaves the arrays).  Calls on one device share that array: calls that
 * overlap in time on one device (different streams or contexts) race. */
int mdet_tnf_count_noalloc(mdet_ctx *ctx, const uint32_t *packed_dev, uint64_t n_bases, const uint64_t *runs_dev,
                           uint64_t n_runs, const uint64_t *base_off_dev, uint32_t n, uint32_t *counts_dev,
                           float *tnf_dev);

/* Same result from raw bytes: contig r is seqs_dev[index_dev[r] ..
 * index_dev[n+r]) (get_TNF's [begin | end] index, cuda/Cuda.cu:222-226),
 * case-insensitive ACGT, anything else voids the windows that contain it. */
int mdet_tnf_count_ascii(mdet_ctx *ctx, const char *seqs_dev, const uint64_t *index_dev, uint32_t n,
                         uint32_t *counts_dev, float *tnf_dev);

/* ---------------------------------------------------------------- pairs -- */
/* Precision of the all-pairs distance stage; every mode yields the same edge
 * set (see mdet_tnf_edges). */
#define MDET_EXACT_F32 0   /* FP32 sum of squared differences for every pair that a lower
                            * bound of its distance does not rule out */
#define MDET_BF16_REFINE 1 /* the same with a BF16 MFMA Gram ahead of the FP32 refinement */
#define MDET_F16_REFINE 2  /* the same with an FP16 MFMA Gram */
#define MDET_LEARNED 3     /* learned embedding proposals + FP32 refinement
                            * (mdet_tnf_edges_learned; recall measured, full rows exact) */

typedef struct mdet_edges {
    uint64_t count;
    /* Device arrays owned by the context, valid until the next
     * mdet_tnf_edges call on it or mdet_ctx_destroy.  Sorted by (from, to),
     * from < to.  s = 1 - 1/(1+exp(preProb)) in FP32. */
    const uint32_t *from_dev;
    const uint32_t *to_dev;
    const float *s_dev;
} mdet_edges;

typedef struct mdet_pair_stats {
    uint64_t pairs_total;      /* n(n-1)/2 */
    uint64_t pairs_evaluated;  /* pairs decided (exhaustive modes: pairs_total, most of them by a
                                * lower bound of their distance) */
    uint64_t survivors;        /* pairs passed from the prefilter to FP32 evaluation */
    uint64_t candidates;       /* pairs with FP32 preProb above threshold - band */
    uint64_t adjudicated;      /* pairs decided by the FP64 tie-breaker */
    uint64_t rows_capped;      /* rows with more than max_edges candidates */
    double ms_prefilter;       /* device time of each stage (HIP events) */
    double ms_refine;
    double ms_select;
    double ms_total;
    uint64_t rows_block;       /* rows selected by the block-wide path (more
                                * than 512 candidates, or more than 64
                                * near-ties at the cut) */
    uint64_t rows_global;      /* rows selected in global memory (more than
                                * 4096 candidates, or more than 512 near-ties
                                * at the cut); no size limit */
    /* learned mode, cluster index with the TNF Gram (mdet_tnf_edges_learned):
     * the exact fallback for rows whose proposals fill max_edges */
    uint64_t fallback_rows;    /* full rows evaluated again against every column */
    uint64_t fallback_chunks;  /* 32 x 32 tiles of pairs that this pass's scan lists */
    uint64_t fallback_pairs;   /* its survivors outside the probed cluster pairs, refined */
} mdet_pair_stats;

/*
 * The thresholded, per-row-capped TNF edge list of n contigs:
 *   tnf_dev[n*136] FP32 rows (unit L2 norm), logsize_dev[n] FP64 log10 sizes
 *   with every size >= 1500 (the reference refuses minContig < 1500,
 *   cuda/Cuda2.cu:1329-1332; the model is only monotone in d there).
 * Edge (i, j), i < j, is emitted iff preProb(i,j) > log(1/(1-cutoff) - 1)
 * and j is among the max_edges highest-similarity partners of row i
 * (max_edges == 0: no cap), with preProb as cal_tnf_pre_dist_d computes it.
 * Replaces gen_tnf_graph (cuda/Cuda2.cu:861-970) with get_tnf_graph2
 * (cuda/Cuda2.cu:243-262) and the host heaps of lines 896-946; stats may be
 * NULL.
 */
int mdet_tnf_edges(mdet_ctx *ctx, const float *tnf_dev, const double *logsize_dev, uint32_t n, double cutoff,
                   uint32_t max_edges, int precision, mdet_edges *out, mdet_pair_stats *stats);

/*
 * The prefilters' distance radius: an upper bound, proven and within 1e-7 of
 * the true value, of the largest TNF distance at which a pair of contigs
 * with log sizes in [xlo, xhi] can have preProb > log(1/(1 - cutoff) - 1)
 * (gen_tnf_graph's rule, cuda/Cuda2.cu:884).  No pair farther apart can be an
 * edge, so every prefilter keeps all pairs within it (plus its own rounding
 * margin).  MDET_E_RANGE outside [log10 1500, log10 500000].
 */
int mdet_model_radius(double xlo, double xhi, double cutoff, double *radius);

/*
 * The TNF-only probability graph of the MetaBAT1 variant: every pair (i, j),
 * i < j, whose similarity s = 1 - prob is >= required_min_p, no per-row cap,
 * with prob the variant's TNF distance (cal_tnf_dist_d, cuda/Cuda.cu:103-165:
 * model 1 above the ln 9 floor, else model 2, 0.1 where model 2 is above its
 * floor).  Replaces get_tnf_prob + create_graph (cuda/Cuda.cu:167-198,
 * 1738-1768; with no abundance file cal_dist2 returns the TNF distance,
 * cuda/Cuda.cu:798-814), whose caller caps required_min_p at 0.75
 * (cuda/Cuda.cu:2425-2427).  Inputs and output as mdet_tnf_edges (log sizes
 * of contigs >= 1500 bases; the variant forms log10 of the clamped size on the
 * device, the callers here pass the host value).  The edge count grows fast
 * as required_min_p falls (every pair above s is an edge).
 */
int mdet_tnf_prob_edges(mdet_ctx *ctx, const float *tnf_dev, const double *logsize_dev, uint32_t n,
                        double required_min_p, int precision, mdet_edges *out, mdet_pair_stats *stats);

/* The pairs the last mdet_tnf_edges / mdet_tnf_edges_learned call on ctx
 * evaluated exactly: *count records of 16 bytes {uint32 i, uint32 j,
 * float preProb, uint32 flags} (flags bit 0: decided by the FP64
 * tie-breaker, bit 1: preProb above the threshold), device memory owned by
 * ctx.  These label the training pairs of the learned filter. */
int mdet_last_pairs(mdet_ctx *ctx, const void **records_dev, uint64_t *count);

/* ---------------------------------------------------- learned filter -- */
/* No reference counterpart: the reference evaluates every pair.  An MLP
 * 136 -> 256 -> 256 -> 32 (GELU, BF16 weights, FP32 accumulation) maps a
 * standardised TNF row to an embedding; trained with a contrastive margin
 * loss on pairs the exact path labels, so that a small embedding distance
 * proposes the pairs that can clear the edge threshold. */
typedef struct mdet_mlp mdet_mlp;
int mdet_mlp_create(mdet_ctx *ctx, uint64_t seed, mdet_mlp **out);
int mdet_mlp_destroy(mdet_mlp *mlp);
uint64_t mdet_mlp_param_count(void); /* 109,088 */
/* FP32 master parameters, layout W1[256x136] b1[256] W2[256x256] b2[256]
 * W3[32x256] b3[32] (row-major, out x in); host arrays.  If count is at least
 * twice the parameter count, the second half receives the parameters as the
 * forward pass uses them (weights rounded to BF16). */
int mdet_mlp_get_params(mdet_mlp *mlp, float *out, uint64_t count);
int mdet_mlp_set_params(mdet_mlp *mlp, const float *in, uint64_t count);
/* Input standardisation x' = (tnf - mean) * istd, per column (host arrays). */
int mdet_mlp_set_input_norm(mdet_mlp *mlp, const float *mean136, const float *istd136);
/* Loss L = mean y*D + (1-y)*relu(margin - D), D = |e_i - e_j|^2, over the
 * batch of pairs (pi_dev[b], pj_dev[b], label_dev[b] in {0,1}); grad_out
 * (host, param_count floats) receives dL/dparams at the BF16-rounded weights
 * the forward pass uses; either output may be NULL. */
int mdet_mlp_grad(mdet_mlp *mlp, const float *tnf_dev, const uint32_t *pi_dev, const uint32_t *pj_dev,
                  const float *label_dev, uint32_t batch, float margin, float *grad_out, float *loss_out);
/* One Adam step (beta 0.9 / 0.999) on that loss; loss_out may be NULL. */
int mdet_mlp_train_step(mdet_mlp *mlp, const float *tnf_dev, const uint32_t *pi_dev, const uint32_t *pj_dev,
                        const float *label_dev, uint32_t batch, float lr, float margin, float *loss_out);
/* Embeddings emb_dev[n x 32] of TNF rows tnf_dev[n x 136]. */
int mdet_mlp_embed(mdet_mlp *mlp, const float *tnf_dev, uint32_t n, float *emb_dev);
/* Training of the filter from TNF rows alone (the steps a caller would
 * otherwise script): input standardisation from the rows' column means and
 * standard deviations; one MDET_BF16_REFINE edge-list call whose exactly
 * decided pairs label the data (mdet_last_pairs; positives = preProb above
 * the threshold of cutoff); a training set of n_pairs with positives :
 * negatives = 1 : 4 (positives and twice as many "hard" negatives, evaluated
 * but below the threshold, chosen by a seeded hash of the pair; the rest
 * uniform random pairs labelled against the positives), shuffled; `steps`
 * Adam steps over consecutive batches; with radius_quantile > 0, radius2 =
 * 1.05 x that quantile of the positives' squared embedding distances (for
 * mdet_tnf_edges_learned's radius form).  Zero fields take the defaults
 * shown.  The edge-list buffers of ctx are reused (as by mdet_tnf_edges). */
typedef struct mdet_fit_config {
    uint64_t n_pairs;        /* training pairs (0: 10,000,000) */
    uint32_t steps;          /* Adam steps (0: 20,000) */
    uint32_t batch;          /* pairs per step (0: 512) */
    float lr;                /* (0: 2e-3) */
    float margin;            /* loss margin on the squared distance (0: 4.0) */
    uint64_t seed;           /* sampling and shuffling */
    double radius_quantile;  /* in (0, 1]: calibrate radius2; 0: do not */
    uint32_t loss_every;     /* > 0: record (step, loss) every loss_every steps and at the last */
    uint32_t loss_cap;       /* capacity of loss_curve in (step, loss) entries */
    float *loss_curve;       /* host array of 2 x loss_cap floats, or NULL */
} mdet_fit_config;

typedef struct mdet_fit_result {
    uint64_t labelled;     /* pairs the labelling call decided exactly */
    uint64_t positives;    /* of them above the threshold */
    uint64_t pairs;        /* training pairs built */
    uint32_t loss_points;  /* entries written to loss_curve */
    float radius2;         /* calibrated squared radius, 0 without a quantile */
    double ms_label;       /* host wall time: standardisation, labels and set */
    double ms_train;       /* the Adam steps */
    double ms_calibrate;   /* the radius */
} mdet_fit_result;

/* The training-set step alone, on the host: records[n_records] as
 * mdet_last_pairs gives them (host copy), contigs < n; pi, pj, y receive
 * *count pairs (cap entries each; all three NULL: only *count and
 * *positives are set, MDET_E_CAPACITY if cap is too small).  The sample
 * depends only on the set of records and the seed, not on their order. */
int mdet_fit_training_set(const void *records, uint64_t n_records, uint32_t n, uint64_t n_pairs, uint64_t seed,
                          uint32_t *pi, uint32_t *pj, float *y, uint64_t cap, uint64_t *count, uint64_t *positives);
/* The standardisation step alone: mean and 1/(std + 1e-6) of each column of
 * tnf_dev[n x 136] (population std, NaN read as 0) set as the input norm. */
int mdet_mlp_norm_from_rows(mdet_mlp *mlp, const float *tnf_dev, uint32_t n);
int mdet_mlp_fit(mdet_mlp *mlp, const float *tnf_dev, const double *logsize_dev, uint32_t n, double cutoff,
                 uint32_t max_edges, const mdet_fit_config *cfg, mdet_fit_result *result);

/* Edge list as mdet_tnf_edges, with the pairs to evaluate proposed by the
 * network.  With n_probe > 0 (at most 32): a cluster index over the
 * embeddings (k-means, n_clusters centroids, 0 = n/192, at most 16384), and the
 * pairs of clusters among each other's n_probe nearest centroids.
 *   radius2 == 0 (the default form): within those cluster pairs the BF16 TNF
 *   Gram prefilter of MDET_BF16_REFINE decides.  A row whose proposals fill
 *   its max_edges slots (at least max_edges - max_edges/32 kept: a full row;
 *   the divisor is mdet_learned_set_fallback_margin's)
 *   could have missed a better partner, so full rows are evaluated again
 *   against every column (BF16 Gram, the survivors outside the probed
 *   cluster pairs refined): a full row keeps exactly mdet_tnf_edges's
 *   top-max_edges (mdet_learned_set_fallback turns this off).  Other rows
 *   keep the proposed partners that pass (a subset of theirs; recall
 *   measured).
 *   radius2 > 0: within the probed cluster pairs only pairs whose BF16
 *   embedding distance^2 is below radius2 are evaluated (no fallback).
 * With n_probe == 0 and radius2 > 0: every pair's embedding distance (MFMA
 * Gram over the whole triangle), the same radius rule.  The exact stage
 * (refinement and selection) is the other modes'.  stats->pairs_evaluated
 * counts the candidate pairs, stats->fallback_* the exact completion. */
int mdet_tnf_edges_learned(mdet_ctx *ctx, mdet_mlp *mlp, const float *tnf_dev, const double *logsize_dev, uint32_t n,
                           double cutoff, uint32_t max_edges, float radius2, uint32_t n_clusters, uint32_t n_probe,
                           mdet_edges *out, mdet_pair_stats *stats);
/* The full-row fallback of the default learned form on (enabled != 0, the
 * default of a new context) or off for later calls on ctx.  Off, a full row
 * keeps its proposed partners only, and a missed better partner lets the next
 * proposed one in: edges outside the exhaustive list become possible (faster,
 * for callers that accept that). */
int mdet_learned_set_fallback(mdet_ctx *ctx, int enabled);
/* The full-row margin for later learned calls on ctx: a row is completed
 * against every column when its proposals keep at least max_edges -
 * max_edges / margin_div partners (default 32; margin_div >= 1, 1 completes
 * every row).  A row keeps a wrong edge only if it missed more partners than
 * the margin and exceeds max_edges in truth: a smaller divisor makes that
 * rarer and evaluates more rows (measured at 1M contigs, cutoff 0.95,
 * maxEdges 200: 12 wrong edges of 50.7M at 32, none at 8 for 1.43x the time). */
int mdet_learned_set_fallback_margin(mdet_ctx *ctx, uint32_t margin_div);
/* The exact cover for later learned calls on ctx (enabled != 0; off in a new
 * context).  In the default form (radius2 == 0, n_probe > 0; n_probe then
 * only selects the form), the cluster pairs come from a bound instead of the
 * probes: with each cluster's TNF-space centre c and radius r (over its
 * members), a pair of contigs in clusters a and b is at TNF distance at least
 * min_{i in a} |x_i - c_b| - r_b and min_{j in b} |x_j - c_a| - r_a, and the
 * pair of clusters is evaluated unless one of these reaches the distance
 * beyond which no pair passes the BF16 prefilter (its radius, rounding
 * margins included).  Every pair the exhaustive prefilter would keep is then
 * evaluated, so the edge list is mdet_tnf_edges's, with no full-row
 * completion; stats->fallback_rows is 0.  The clusters are k-means clusters
 * (n_clusters; 0 = n/128 up to 2048 clusters, else n/84, at most 16384) of a
 * fixed 32-dimensional sign projection of the TNF rows: no network is used,
 * and mlp may be NULL.  The bound prunes well when clusters outnumber the
 * populations (genomes) of the input: measured at 200,000 contigs of 1,000
 * genomes 0.87% of the pairs evaluated (4.3 ms, 1.8x MDET_BF16_REFINE), at
 * 1,000,000 contigs of 5,000 genomes 0.20% (31 ms, 4.6x on the same GPU);
 * with fewer clusters than genomes most pairs are evaluated, never a wrong
 * one. */
int mdet_learned_set_exact_cover(mdet_ctx *ctx, int enabled);

/* ------------------------------------------------------------ autotuner -- */
/* No reference counterpart: the reference's only tuning is its fixed TILE
 * heuristic (cuda/Cuda2.cu:868-874) and the --ct/--cb/--cs launch flags
 * (cuda/Cuda.cu:1869-1871).
 * Launch shapes of the pair stage, one set per precision mode, held by the
 * context and used by every later edge-list call on it.  No shape changes
 * the edge list. */
typedef struct mdet_tune {
    uint32_t seg_cols;      /* MFMA Gram modes: prefilter item column span, a
                             * multiple of 256 in [256, 65536], or 0 (default):
                             * the power of two nearest n/50 in [512, 16384] */
    uint32_t persistent;    /* MFMA modes: 0 one prefilter block per item, 1
                             * (default) resident blocks take items from a
                             * counter */
    uint32_t refine_blocks; /* refinement blocks per CU, 1..64 (default 64;
                             * no more than fit are launched) */
    uint32_t item_order;    /* Gram modes with persistent blocks: 0 one item
                             * queue, row-block major; 1 (default) one queue
                             * per XCD (row blocks rb % 8), column-start major */
    double ms_prefilter;    /* autotuner: median stage times at the chosen */
    double ms_refine;       /* shape (0 when never tuned) */
} mdet_tune;
int mdet_tune_get(mdet_ctx *ctx, int precision, mdet_tune *out);
int mdet_tune_set(mdet_ctx *ctx, int precision, const mdet_tune *in);
/* Times the candidate shapes on this input (each the median of reps calls of
 * mdet_tnf_edges; reps 1..15) by the prefilter stage time: column spans
 * 512/1024/2048/4096, and longer ones up to the default where n makes that
 * longer, x {per-item blocks, persistent blocks with item order 0 or 1} (for
 * the Gram modes; EXACT_F32's shape is not tuned).  Keeps the fastest in ctx,
 * the default unless another is more than 2% faster, and returns it (out may be
 * NULL).  Small inputs (up to 6,144 contigs), which skip that stage, leave the
 * shape as it is (ms_prefilter 0).  refine_blocks is set to its default (every
 * value above what fits launches the same) and its stage timed there.  The last
 * call's edge list stays in ctx as after mdet_tnf_edges.  ~13 x reps + 1
 * edge-list calls, 19 x reps + 1 at 1,000,000 contigs. */
int mdet_tnf_autotune(mdet_ctx *ctx, const float *tnf_dev, const double *logsize_dev, uint32_t n, double cutoff,
                      uint32_t max_edges, int precision, uint32_t reps, mdet_tune *out);
/* The same for the learned mode (per-item or persistent prefilter blocks),
 * with mdet_tnf_edges_learned's arguments. */
int mdet_tnf_autotune_learned(mdet_ctx *ctx, mdet_mlp *mlp, const float *tnf_dev, const double *logsize_dev,
                              uint32_t n, double cutoff, uint32_t max_edges, float radius2, uint32_t n_clusters,
                              uint32_t n_probe, uint32_t reps, mdet_tune *out);

/*
 * Sampled row maxima for the automatic cutoff (pTNF = 0): for each sampled
 * position p < n_sample, max_out_dev[p] = 1 - 1/(1 + exp(m)) with m the
 * largest preProb between contig idx_dev[p] and every contig idx_dev[q],
 * q != p, q < n (and m >= DBL_MIN).  idx_dev is a permutation of 0..n-1 whose
 * first n_sample entries are the sample.  Replaces get_tnf_max_prob_sample
 * and launch_tnf_max_prob_sample_kernel_multi (cuda/Cuda2.cu:281-314,
 * 356-379); the maximum is exact (FP32 scan, FP64 re-evaluation of every
 * pair within the FP32 error band of the row maximum).
 */
int mdet_tnf_rowmax(mdet_ctx *ctx, const float *tnf_dev, const double *logsize_dev, uint32_t n,
                    const uint64_t *idx_dev, uint32_t n_sample, double *max_out_dev);

/* The FP32 form of the model the device evaluates: tensor Chebyshev
 * coefficients (4 x 8 x 7 floats: b1, c1, b2, c2; row p = degree in the
 * min-size variable) of the logistic polynomials of cal_tnf_dist
 * (cuda/Cuda2.cu:170-188, 747-771) on [log10 1500, log10 500000]^2 (domain2),
 * and sum |C| of each (abs_sum4).  Host-only; abs_sum4/domain2 may be NULL. */
int mdet_model_cheb(float *out, double *abs_sum4, double *domain2);
/* The monomial coefficient table `which` (0 b1, 1 c1, 2 b2, 3 c2) of the
 * logistic models as the library holds it (cuda/Cuda2.cu:170-188), with each
 * term's exponents (x = min, y = max log size) in exps_xy[2*t], [2*t+1];
 * *count receives the number of terms (17..19).  Host-only; coef and
 * exps_xy may be NULL. */
int mdet_model_coefs(int which, double *coef, int32_t *exps_xy, uint32_t cap, uint32_t *count);

/*
 * preProb of listed pairs (device arrays pi_dev[np], pj_dev[np]) in the
 * library's FP32 evaluator (pre32_dev, may be NULL) and its FP64 tie-breaker
 * (pre64_dev, may be NULL).  The device function cal_tnf_pre_dist_d
 * (cuda/Cuda2.cu:192-241) exposed for checking.  Every log size must lie in
 * [log10 1500, log10 500000] and every index below n; otherwise the call
 * returns MDET_E_RANGE (pairs with an index >= n get NaN, no row is read for
 * them).
 */
int mdet_tnf_preprob(mdet_ctx *ctx, const float *tnf_dev, const double *logsize_dev, uint32_t n,
                     const uint32_t *pi_dev, const uint32_t *pj_dev, uint64_t np, float *pre32_dev,
                     double *pre64_dev);

/*
 * FP64 similarity s = 1 - 1/(1 + exp(preProb)) of listed pairs (device arrays
 * pi_dev[np], pj_dev[np] -> s64_dev[np]), preProb from the FP64 tie-breaker:
 * the double the reference stores per edge in Graph::sTNF (get_tnf_graph2,
 * cuda/Cuda2.cu:257-258; gen_tnf_graph, cuda/Cuda2.cu:936-940).  The edge
 * list's own s_dev is FP32; the C++ drop-in calls this for the emitted edges.
 * An index >= n returns MDET_E_RANGE (that pair's output is NaN).
 */
int mdet_tnf_similarity64(mdet_ctx *ctx, const float *tnf_dev, const double *logsize_dev, uint32_t n,
                          const uint32_t *pi_dev, const uint32_t *pj_dev, uint64_t np, double *s64_dev);

/*
 * Binning consumer of the TNF graph with no abundance input (the edge score
 * is its similarity, sSCR = sTNF, cuda/Cuda2.cu:1969-1970): the edges ordered
 * by score, descending (orderhigh, cuda/Cuda2.cu:1981-1982; a stable device
 * sort here, equal scores keep their input order), then the sequential graph
 * traversal with label propagation at ten points of the share of contigs
 * connected, maxP/10 ... maxP, stopping at the first edge with score <= minS
 * (cuda/Cuda2.cu:1984-2062; label_propagation, cuda/Cuda2.cu:569-655).
 * Device edge arrays from_dev, to_dev (endpoints < n, from != to) and s_dev
 * (FP64 scores in [0, 1), e.g. from mdet_tnf_similarity64); host output
 * membership[n] = cluster label of each contig (a contig id, the reference's
 * mems); *rounds (may be null) = propagation points reached.  maxP and minS
 * as fractions in (0, 1) (the reference's percent options / 100).  The sort
 * runs on the device; the traversal, sequential by definition, on the host.
 * Errors: MDET_E_INVALID (null pointer, maxP/minS outside (0, 1)),
 * MDET_E_RANGE (endpoint >= n, a loop, a score outside [0, 1), more than
 * 2^31 - 1 edges).
 */
int mdet_bin_labels(mdet_ctx *ctx, const uint32_t *from_dev, const uint32_t *to_dev, const double *s_dev,
                    uint64_t n_edges, uint32_t n, double max_p, double min_s, uint64_t *membership,
                    uint32_t *rounds);

/*
 * The host half of mdet_bin_labels: the traversal over host edge arrays
 * already in traversal order (scores non-increasing; MDET_E_INVALID if a
 * score exceeds its predecessor).  Same outputs and errors.  Replaces the
 * loop at cuda/Cuda2.cu:1994-2062 given oSCR.
 */
int mdet_bin_traverse(const uint32_t *from, const uint32_t *to, const double *s, uint64_t n_edges, uint32_t n,
                      double max_p, double min_s, uint64_t *membership, uint32_t *rounds);

#ifdef __cplusplus
}
#endif

#endif /* MDET_TNF_H */
