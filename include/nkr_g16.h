/*
 * nkr_g16.h -- C ABI of the MI355X (gfx950) Groth16 prover backend for BN254.
 *
 * Every entry point returns 0 on success and a non-zero status on failure;
 * nkr_last_error() then returns a message (thread-local, valid until the next
 * call on the same thread).  Nothing aborts across this boundary.
 *
 * Data layouts are the reference's in-memory layouts (no conversion):
 *   Fr / Fq element   32 B: 4 little-endian u64 words of x*2^256 mod p
 *                     (libff Fp_model mont_repr, fp.hpp:42)
 *   G1 point          96 B: Jacobian X, Y, Z over Fq (libff alt_bn128_G1)
 *   G2 point         192 B: Jacobian X, Y, Z over Fq2 = (c0, c1)
 *   CSR matrix        u32 row_ptr[rows + 1], u32 col_idx[nnz], Fr values[nnz]
 *                     (protocols/groth16/common/include/r1cs/spmat.hpp:37-45)
 *   RawProof         576 B: ar, bs1, zk, qz (G1) then bs2 (G2)
 *                     (protocols/groth16/common/include/groth16/types.hpp:47-53)
 *   Proof            384 B: a (G1), b (G2), c (G1)  (types.hpp:55-59)
 * Output points are normalised: Z = 1, or (0, 1, 0) for the point at infinity,
 * exactly what libff's to_affine_coordinates() produces.
 *
 * Reference interfaces replaced (paths relative to the reference tree):
 *   nkr_g16_ctx_create   HipBackend::prepare
 *                        (protocols/groth16/backends/hip/src/backend.hip:270-296;
 *                         virtual Backend::prepare, common/include/groth16/backend.hpp:21)
 *   nkr_g16_prove        HipBackend::prove (backend.hip:298-335;
 *                         virtual Backend::prove, backend.hpp:23-27)
 *   nkr_g16_blind        blind_proof (protocols/groth16/common/src/protocol.cpp:85-94),
 *                        with r and s supplied by the caller
 *   nkr_fr_ntt           NTTContext::{ntt,intt,coset_ntt,coset_intt}
 *                        (operators/hip/include/ntt/ntt.hip:106-186) with libfqfft
 *                        basic_radix2_domain semantics (basic_radix2_domain.tcc:41-74)
 *   nkr_spmv             spMVMContext::spmvm (backends/hip/include/spmvm/spmvm.hip:53-71)
 *   nkr_g1_msm_*,        MSMContext::load_bases / MSMContext::msm
 *   nkr_g2_msm_*         (operators/hip/include/msm/msm.hip:61-158); result semantics of
 *                        libff multi_exp<BDLO12> as called by the CPU backend
 *                        (protocols/groth16/backends/cpu/src/backend.cpp:16-23)
 *   nkr_g16_quotient     the quotient stage of Backend::prove (backend.hip:313-321;
 *                        CPU backend.cpp:171-179)
 *
 * Handles are not thread-safe: calls on one handle must be serialised.
 * Device pointers appear only in the *_dev entry points, which exist so that
 * benchmarks can keep inputs resident in HBM.
 */
#ifndef NKR_G16_H
#define NKR_G16_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

const char *nkr_last_error(void);
/* Library version string. */
const char *nkr_version(void);
/* Number of visible GPUs. */
int nkr_device_count(int *count);

/* ---------------------------------------------------------------- Groth16 */
typedef struct {
    uint64_t rows;      /* constraints, a power of two >= 2 */
    uint64_t cols;      /* variables + 1 */
    uint64_t public_inputs;
    const uint32_t *a_row_ptr, *a_col_idx;
    const void *a_values;
    uint64_t a_nnz;
    const uint32_t *b_row_ptr, *b_col_idx;
    const void *b_values;
    uint64_t b_nnz;
    const uint32_t *c_row_ptr, *c_col_idx;
    const void *c_values;
    uint64_t c_nnz;
} nkr_g16_circuit;

typedef struct {
    const void *a_query;    /* cols G1 */
    const void *b_g1_query; /* cols G1 */
    const void *b_g2_query; /* cols G2 */
    const void *l_query;    /* cols G1 */
    const void *h_query;    /* rows G1 */
    const void *alpha_g1, *beta_g1, *beta_g2, *delta_g1, *delta_g2;
} nkr_g16_pk;

typedef struct nkr_g16_ctx nkr_g16_ctx;

/* Uploads the circuit, normalises and window-expands the proving key in HBM
 * and builds the NTT tables (the reference's prepare).  Host pointers. */
int nkr_g16_ctx_create(const nkr_g16_circuit *circuit, const nkr_g16_pk *pk, int device, nkr_g16_ctx **out);

/* Per-context tuning (0 in a field keeps the default).  The proof does not
 * depend on any of them, only the time does; nkr-zkp_amd/autotune.py picks
 * them per (domain size, witness density) by measurement.  No counterpart in
 * the reference (its window and stage choices are fixed,
 * operators/hip/include/msm/msm.hip:25-60).
 *   witness_window_bits  MSM window of the MSMs over all witness columns, 2..15
 *                          (bs1 and bs2 choose their own where few of the
 *                          columns occur in B)
 *   h_window_bits        MSM window of the H MSM, 2..16
 *   ntt_lds_log          10 or 11: 2^lds_log elements per transform tile
 *   ntt_radix_log        2 or 3: register radix of the transform rounds
 *   ntt_split_policy     1 + policy: 1 balanced passes, 2 full last pass
 *   msm_target_pieces_log  2^k accumulation threads per MSM launch, 12..24
 *                          (19: the library's choice, as nkr_msm_set_shape)
 *   witness_g1_piece_min   shortest run of entries of a thread in the witness
 *                          G1 MSMs, 1..64 */
typedef struct {
    uint32_t witness_window_bits, h_window_bits;
    uint32_t ntt_lds_log, ntt_radix_log, ntt_split_policy;
    uint32_t msm_target_pieces_log, witness_g1_piece_min;
} nkr_g16_tuning;
int nkr_g16_ctx_create_tuned(const nkr_g16_circuit *circuit, const nkr_g16_pk *pk, int device,
                             const nkr_g16_tuning *tuning, nkr_g16_ctx **out);
int nkr_g16_ctx_destroy(nkr_g16_ctx *ctx);
/* Device bytes held by the context. */
int nkr_g16_ctx_device_bytes(const nkr_g16_ctx *ctx, uint64_t *bytes);

/* Backend::prove: witness is cols Fr (z[0] = 1), raw_out receives 576 B. */
int nkr_g16_prove(nkr_g16_ctx *ctx, const void *witness, void *raw_out);
/* As nkr_g16_prove, also returning the intermediates (each rows Fr, natural
 * order) when the pointers are non-NULL: A*z, B*z, C*z and H. */
int nkr_g16_prove_ex(nkr_g16_ctx *ctx, const void *witness, void *raw_out, void *az, void *bz, void *cz, void *h);

/* As nkr_g16_prove with the witness already in device memory (cols Fr). */
int nkr_g16_prove_dev(nkr_g16_ctx *ctx, const void *witness_dev, void *raw_out);

/* prove followed by blind_proof with caller-supplied r, s (the reference's
 * groth16.prove.total scope, protocols/groth16/app/prove.cpp:79-88) in one
 * call: the r,s-only blinding terms are computed on the host while the GPU
 * works.  raw_out (576 B) and proof_out (384 B) are both written.  The
 * proving key given to nkr_g16_ctx_create must include alpha/beta/delta. */
int nkr_g16_prove_blind(nkr_g16_ctx *ctx, const void *witness, const void *r, const void *s, void *raw_out,
                        void *proof_out);
int nkr_g16_prove_blind_dev(nkr_g16_ctx *ctx, const void *witness_dev, const void *r, const void *s,
                            void *raw_out, void *proof_out);

/* Batched proving.  The reference proves one circuit per process and runs
 * independent proofs side by side as separate processes
 * (scripts/bench/runner.py:260-355); this entry point is a new caller of the
 * same contexts: count proofs (any mix of contexts created on the batch's
 * device, the same context any number of times) go through the GPU as one
 * launch sequence -- one SpMV launch, one launch per NTT pass per domain
 * size, shared MSM accumulation and reduction launches -- and each item
 * receives exactly what nkr_g16_prove_blind gives for it alone.  Items are
 * host memory: witness (cols Fr), r and s (Fr), raw_out (576 B), proof_out
 * (384 B).  A batch handle owns per-proof work buffers that grow to the
 * largest batch it has run; calls on one handle must be serialised, and no
 * context in a batch may be used by another thread during the call. */
typedef struct nkr_g16_batch nkr_g16_batch;
typedef struct {
    nkr_g16_ctx *ctx;
    const void *witness;
    const void *r, *s;
    void *raw_out, *proof_out;
} nkr_g16_batch_item;
int nkr_g16_batch_create(int device, nkr_g16_batch **out);
int nkr_g16_batch_prove(nkr_g16_batch *batch, const nkr_g16_batch_item *items, uint64_t count);
int nkr_g16_batch_destroy(nkr_g16_batch *batch);
/* Launch-sequence reuse (no counterpart in the reference, which launches
 * every kernel of every proof): a batch of the same contexts in the same
 * order as the handle's previous call, with no nkr_msm_set_shape that changed
 * anything in between, is captured into a HIP graph on its second occurrence and replayed while the composition repeats (the
 * size-class schedule of that composition); any other batch runs eagerly and
 * drops the graph.  Results are identical either way.  enabled = 0 turns the
 * capture off (and drops a graph); *active tells whether the handle holds a
 * graph now. */
int nkr_g16_batch_set_graphs(nkr_g16_batch *batch, int enabled);
int nkr_g16_batch_graph_active(const nkr_g16_batch *batch, int *active);

/* Serving: a request loop with continuous batching (no counterpart in the
 * reference, which serves nothing; its harness runs one prove per process,
 * scripts/bench/runner.py:260-355).  Contexts stay resident (keys and NTT
 * tables in HBM); submit() queues a proof and returns a ticket; `workers`
 * threads each own a batch (own streams), and a free worker takes every
 * pending request whose batch fits its share of the work-memory budget, up
 * to max_batch, so requests arriving while other batches are on the GPU are
 * admitted as workers and memory free up and run alongside them.  The budget
 * is clamped at creation to the device's free memory minus a reserve (the
 * larger of 1 GiB and 1/32 of the device) and split equally between the
 * workers.  A request alone needs nkr_g16_server_request_bytes of its context
 * (a batch at most about the sum: its MSMs share their launches), and one
 * larger than a worker's share is rejected by submit.  A worker releases its grow-only work buffers whenever keeping them
 * would exceed its share, so the work memory held by all workers stays within
 * the budget.  A request that cannot be proved (its context lacks the
 * blinding elements) fails alone: its wait() reports the error and the rest
 * of its batch completes; a batch that fails as a whole is retried request by
 * request.  wait() blocks until the ticket is done and gives its
 * submit-to-completion latency.  Results are exactly nkr_g16_prove_blind's.
 * The caller keeps witness, r, s and the outputs alive until wait() returns;
 * submit and wait may be called from any thread.
 * stats[4] = batches run, proofs done, largest batch, peak admitted bytes.
 * memory[4] = effective budget, one worker's share, work bytes the workers
 * hold now, most work bytes held at once. */
typedef struct nkr_g16_server nkr_g16_server;
int nkr_g16_server_create(int device, uint32_t workers, uint32_t max_batch, uint64_t work_budget_bytes,
                          nkr_g16_server **out);
int nkr_g16_server_submit(nkr_g16_server *server, nkr_g16_ctx *ctx, const void *witness, const void *r,
                          const void *s, void *raw_out, void *proof_out, uint64_t *ticket);
int nkr_g16_server_wait(nkr_g16_server *server, uint64_t ticket, double *latency_ms);
/* Warm-up before traffic (no counterpart in the reference): every worker
 * proves the `count` items once as one batch (outputs written to the items'
 * buffers), so that its work buffers are already sized for such requests
 * instead of growing on the first one, which would then pay the device
 * allocations.  Waits until no batch is in flight; requests submitted
 * meanwhile wait for it.  count <= max_batch and the items' batch must fit one
 * worker's share.  Not concurrently with another warm-up or
 * with nkr_g16_server_destroy. */
int nkr_g16_server_warm(nkr_g16_server *server, const nkr_g16_batch_item *items, uint64_t count);
int nkr_g16_server_request_bytes(const nkr_g16_ctx *ctx, uint64_t *bytes);
int nkr_g16_server_stats(const nkr_g16_server *server, uint64_t *stats);
int nkr_g16_server_memory(const nkr_g16_server *server, uint64_t *memory);
int nkr_g16_server_destroy(nkr_g16_server *server);

/* Stage timing with HIP events on the context's stream.  While enabled,
 * every prove adds its per-stage device time (ms) to running totals:
 *   0 SpMV, 1 NTT passes (6 transforms: 3 iFFT, 3 cosetFFT; the H query is
 *   prepared in the coset-evaluation basis, so no icosetFFT runs), 2 quotient
 *   pointwise, 3 MSM digit sort (2 schedules: witness and quotient),
 *   4 G1 MSM bucket accumulation (the k_accumulate launch of the G1 batch:
 *   ar, bs1, zk and H), 5 MSM folding, completion and bit planes (G1 and
 *   G2), 6 plane download + host finish, 7 G2 MSM bucket accumulation (the
 *   k_accumulate launch of bs2).  Stages on the two streams overlap, so the
 *   totals do not add up to the proof's latency.
 * counters[0] = proves timed, counters[1] = accumulation launches,
 * counters[2] = bucket entries (non-zero signed digits) of the witness
 * schedule, summed over proves (each is used by ar and zk, and by bs1 and bs2
 * unless they have a schedule of their own), counters[3] = bucket entries of
 * the H schedule (the fifth MSM). */
#define NKR_G16_STAGES 8
int nkr_g16_profile(nkr_g16_ctx *ctx, int enable);
int nkr_g16_profile_read(const nkr_g16_ctx *ctx, double *stage_ms, uint64_t *counters);
/* entries[0], [1] and [2]: the bucket entries, over the same proves, of the
 * schedules that ar and zk, bs1 and bs2, and H read.  bs1 and bs2 have one of
 * their own, over the variables that occur in B, where that leaves out at
 * least a quarter of the variables. */
int nkr_g16_profile_entries(const nkr_g16_ctx *ctx, uint64_t *entries);

/* check_witness (protocols/groth16/common/src/protocol.cpp:69-83): *ok = 1
 * when (A z) * (B z) = C z row by row.  Host arithmetic. */
int nkr_g16_check_witness(const nkr_g16_circuit *circuit, const void *witness, int *ok);

/* blind_proof with caller-supplied r, s (Fr, Montgomery).  Host arithmetic. */
int nkr_g16_blind(const nkr_g16_pk *pk, const void *raw, const void *r, const void *s, void *proof_out);

/* Output buffers of nkr_g16_setup, caller-allocated host memory: the
 * ProvingKey (types.hpp:30-38) with a_query, b_g1_query, l_query: cols G1;
 * b_g2_query: cols G2; h_query: rows G1; alpha/beta/delta points; and the
 * VerificationKey with ic: public_inputs + 1 G1. */
typedef struct {
    void *a_query, *b_g1_query, *b_g2_query, *l_query, *h_query;
    void *alpha_g1, *beta_g1, *beta_g2, *delta_g1, *delta_g2;
} nkr_g16_pk_out;

typedef struct {
    void *alpha_g1_beta_g2; /* GT, 384 B */
    void *gamma_g2, *delta_g2;
    void *ic;
} nkr_g16_vk_out;

/* Backend::setup (protocols/groth16/common/include/groth16/backend.hpp:20) as
 * CpuBackend::setup computes it (backends/cpu/src/backend.cpp:41-154) and
 * HipBackend::setup accelerates it (backends/hip/src/backend.hip:111-268),
 * with the trapdoors supplied by the caller instead of drawn inside:
 * trapdoors = 5 Fr (Montgomery) t, alpha, beta, gamma, delta.  Query
 * scalars, column evaluations and fixed-base multiplications run on the GPU;
 * alpha_g1_beta_g2 is the host pairing.  Points are written normalised. */
int nkr_g16_setup(const nkr_g16_circuit *circuit, const void *trapdoors, int device, const nkr_g16_pk_out *pk,
                  const nkr_g16_vk_out *vk);

/* VerificationKey (protocols/groth16/common/include/groth16/types.hpp:40-45):
 * alpha_g1_beta_g2 is a GT element (Fq12, 384 B: c0.c0.c0 .. c1.c2.c1, each
 * 32 B Montgomery Fq), gamma_g2 and delta_g2 are G2 (192 B), ic holds
 * ic_len G1 points (96 B each). */
typedef struct nkr_g16_vk {
    const void *alpha_g1_beta_g2;
    const void *gamma_g2;
    const void *delta_g2;
    const void *ic;
    uint64_t ic_len;
} nkr_g16_vk;

/* verify (protocols/groth16/common/src/protocol.cpp:96-108): *accepted = 1
 * when e(A, B) == alpha_g1_beta_g2 * e(IC, gamma) * e(C, delta) with
 * IC = ic[0] + sum_i x_i ic[i+1]; 0 when it fails, when ic_len != n_public + 1
 * (as the reference) or when a proof point is off its curve or B is outside
 * the order-r subgroup.  public_input: n_public Fr (Montgomery).  proof:
 * 384 B Proof.  Host arithmetic. */
int nkr_g16_verify(const nkr_g16_vk *vk, const void *public_input, uint64_t n_public, const void *proof,
                   int *accepted);

/* alt_bn128_reduced_pairing (libff alt_bn128_pairing.cpp:542-547): gt_out =
 * e(P, Q) for a G1 point (96 B) and a G2 point (192 B); the value of libff's
 * final exponentiation, f^(m (q^12 - 1)/r) with m = 2x(6x^2 + 3x + 1).
 * Host arithmetic. */
int nkr_bn254_pairing(const void *g1, const void *g2, void *gt_out);

/* prod_i e(P_i, Q_i) with one final exponentiation (k pairs, k may be 0). */
int nkr_bn254_pairing_product(const void *g1s, const void *g2s, uint64_t k, void *gt_out);

/* alt_bn128_ate_miller_loop (alt_bn128_pairing.cpp:368-420) and
 * alt_bn128_final_exponentiation (:226-237) separately.  The Miller value is
 * this library's (affine lines); only its final exponentiation is defined to
 * agree with the reference. */
int nkr_bn254_miller_loop(const void *g1, const void *g2, void *f_out);
int nkr_bn254_final_exponentiation(const void *f, void *gt_out);

/* Quotient stage alone: H from A*z, B*z, C*z (rows Fr each, host pointers). */
int nkr_g16_quotient(const void *az, const void *bz, const void *cz, uint64_t rows, void *h, int device);

/* ------------------------------------------------------ standalone operators */
/* kind: 0 FFT, 1 iFFT, 2 cosetFFT (g = 5), 3 icosetFFT.  n = 2^log_n elements. */
int nkr_fr_ntt(void *data, uint32_t log_n, int kind, int device);               /* host memory */
int nkr_fr_ntt_dev(void *data_dev, uint32_t log_n, int kind, void *stream);    /* device memory */

/* As nkr_fr_ntt_dev, allocating no device memory: for callers that cannot
 * allocate (code under HIP graph capture, tight serving loops, harnesses that
 * forbid hipMalloc).  No counterpart in the reference.  The tables live in
 * one fixed device array per GPU (32.2 MiB, held until the process ends), so log_n is limited to 1 .. 20; larger sizes fail
 * with an error.  The tables are rebuilt on `stream` by every call.  Every
 * call on one GPU shares that array: calls that overlap on one GPU (other
 * streams, other threads) race and must be serialised by the caller.
 * Results equal nkr_fr_ntt_dev's. */
int nkr_fr_ntt_dev_noalloc(void *data_dev, uint32_t log_n, int kind, void *stream);

/* NTT workgroup shape for contexts and domains created afterwards:
 * 2^lds_log elements per workgroup (10 or 11), 2^radix_log elements per
 * thread per register round (2 or 3), and how transforms larger than one
 * workgroup tile split their bits between passes (0: balanced; 1: the
 * unit-stride last pass takes a full tile and the strided passes at most
 * lds_log - 2 bits, so their loads are >= 128-byte contiguous runs).  A
 * tuning knob: results do not depend on it; the default is chosen by
 * measurement. */
int nkr_ntt_set_shape(uint32_t lds_log, uint32_t radix_log, uint32_t split_policy);

/* MSM tuning knobs for every MSM run afterwards: the accumulation splits the
 * sorted entries of a launch evenly over 2^target_pieces_log threads (10 ..
 * 22); at most complete_lanes_cap lane groups (1, 2, 4, 8 or 16) then sum one
 * bucket's partial sums.  Set while no proof runs.  Results do not depend on
 * either.  The defaults are (19, 16); 19 stands for the library's own choice
 * of threads by the number of entries, made by measurement. */
int nkr_msm_set_shape(uint32_t target_pieces_log, uint32_t complete_lanes_cap);

/* y = M * z for one CSR matrix (host memory). */
int nkr_spmv(uint64_t rows, uint64_t cols, const uint32_t *row_ptr, const uint32_t *col_idx, const void *values,
             uint64_t nnz, const void *z, void *y, int device);

/* A CSR matrix uploaded once, then y = M * z over device vectors: the
 * reference's spMVMContext (backends/hip/include/spmvm/spmvm.hip:24-72), whose
 * constructor uploads the matrices and whose spmvm multiplies device
 * vectors.  The host arrays are checked (offsets, columns) and copied at
 * create; run_dev is asynchronous on `stream` (NULL: the null stream) and
 * reads z_dev[cols], writes y_dev[rows]. */
typedef struct nkr_spmv_ctx nkr_spmv_ctx;
int nkr_spmv_create(uint64_t rows, uint64_t cols, const uint32_t *row_ptr, const uint32_t *col_idx,
                    const void *values, uint64_t nnz, int device, nkr_spmv_ctx **out);
int nkr_spmv_run_dev(nkr_spmv_ctx *ctx, const void *z_dev, void *y_dev, void *stream);
int nkr_spmv_destroy(nkr_spmv_ctx *ctx);

/* MSM with prepared bases (the reference's MSMContext: load_bases, then msm).
 * bases: n reference-layout points (any Z; infinity allowed).  c = 0 picks
 * the window width. */
typedef struct nkr_msm nkr_msm;
int nkr_g1_msm_create(const void *bases, uint64_t n, uint32_t c, int device, nkr_msm **out);
int nkr_g2_msm_create(const void *bases, uint64_t n, uint32_t c, int device, nkr_msm **out);
/* scalars: n Fr (host); out: one point (96 B for G1, 192 B for G2). */
int nkr_msm_run(nkr_msm *msm, const void *scalars, void *out);
/* scalars_dev: n Fr in device memory; stream may be NULL. */
int nkr_msm_run_dev(nkr_msm *msm, const void *scalars_dev, void *out, void *stream);
int nkr_msm_window_bits(const nkr_msm *msm, uint32_t *c);
int nkr_msm_destroy(nkr_msm *msm);

/* One-shot convenience: variable_base_msm(bases, scalars) semantics
 * (operators/include/nkr/operators/variable_base_msm.hpp:17-49). */
int nkr_g1_msm(const void *bases, const void *scalars, uint64_t n, void *out, int device);
int nkr_g2_msm(const void *bases, const void *scalars, uint64_t n, void *out, int device);

/* Fixed-base batch scalar multiplication out[i] = scalars[i] * base, the
 * building block of key generation (FixedBaseMsm,
 * operators/include/nkr/operators/fixed_base_msm.hpp:14-39).  base: one
 * host point (96 B / 192 B); outputs normalised points.  The _dev forms take
 * device scalars and a device output array; stream may be NULL. */
int nkr_g1_fixed_base_mul(const void *base, const void *scalars, uint64_t n, void *out, int device);
int nkr_g2_fixed_base_mul(const void *base, const void *scalars, uint64_t n, void *out, int device);
int nkr_g1_fixed_base_mul_dev(const void *base, const void *scalars_dev, uint64_t n, void *out_dev, void *stream);
int nkr_g2_fixed_base_mul_dev(const void *base, const void *scalars_dev, uint64_t n, void *out_dev, void *stream);

/* Batch field products on the device, for arithmetic parity checks:
 * op 0 Fr mul, 1 Fr add, 2 Fr sub, 3 Fq mul, 4 Fq add, 5 Fq sub, 6 Fq2 mul,
 * 7 Fq2 sqr (b ignored), 8 Fr inv (b ignored).  Host memory. */
int nkr_field_op(int op, const void *a, const void *b, void *out, uint64_t n, int device);

/* Device memory helpers so FFI callers can stage data without another runtime. */
int nkr_dev_alloc(uint64_t bytes, void **ptr);
int nkr_dev_free(void *ptr);
int nkr_memcpy_htod(void *dst_dev, const void *src, uint64_t bytes);
int nkr_memcpy_dtoh(void *dst, const void *src_dev, uint64_t bytes);
int nkr_device_synchronize(void);
/* PCI address of `device` ("dddd:bb:dd.f", NUL-terminated, at most len
 * bytes): lets a harness match the device to what a management library or
 * sysfs reports when it samples utilisation. */
int nkr_device_pci_bus_id(int device, char *buf, int len);
/* Plain streaming copy kernel (16-byte vectors): a known-traffic reference
 * for calibrating hardware byte counters.  bytes must be a multiple of 16. */
int nkr_dev_copy(void *dst_dev, const void *src_dev, uint64_t bytes, void *stream);
/* Integer-VALU calibration on `device` (no counterpart in the reference, whose
 * roofs are not measured): the issue rate of v_mad_u64_u32 over the whole
 * device, the 32x32+64-bit multiply-add every Montgomery product is built
 * from, and this library's Fr Montgomery products per second.  Takes a few
 * milliseconds. */
int nkr_valu_probe(int device, double *mad_per_s, double *fr_mul_per_s);

#ifdef __cplusplus
}
#endif

#endif
