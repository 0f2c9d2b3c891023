/*
 * tensororder_hip.h -- C ABI of the MI355X (gfx950) contraction executor.
 *
 * The reference executes a contraction plan through a Python "tensor library" plugin
 * (src/tensor_network/tensor_apis/base_api.py:8-28): per slice, a post-order walk that
 * calls tensordot on every join (src/tensor_network/tensor_network.pyx:142-156,
 * tensor_apis/numpy_apis.py:42-43), summing slice scalars in FP64 (base_api.py:17-28).
 * This library replaces that arithmetic.  The host compiles a plan into a list of launch
 * records whose descriptors live in device memory owned by the caller; every entry point
 * takes plain pointers and sizes, never throws, and returns a TO_* status code.
 *
 * Tensors are dense all-dimension-2 arrays in C order: a rank-r tensor is a vector of 2^r
 * entries and axis 0 is the most significant bit of the flat index.  A join contracts X
 * and Y over s shared bits:
 *     C[batch][(f << shf) | (y << shy)] =
 *         sum_k X[batch*xb + pdep(f, xf_pos) + pdep(k, xs_pos)]
 *             * Y[batch*yb + pdep(y, yf_pos) + pdep(k, ys_pos)]
 * where pdep(v, pos) places bit i of v at bit position pos[i].  A batch stride of 0
 * broadcasts an operand across the batch (slice-invariant tensors).  Free-bit positions
 * (xf_pos, yf_pos) must increase with the bit index.
 *
 * Entry types: TO_F64 computes in float64 throughout.  TO_F32S computes in float32 and
 * keeps, per tensor and batch item, a power-of-two exponent (to_scale_rec): true value =
 * stored value * 2^exp; consumers rescale each operand by 2^-e, e = frexp exponent of the
 * operand's max |entry|, so values never under- or overflow.  Slice results are summed in
 * float64 as (mantissa, int64 exponent) pairs in both modes.
 */
#ifndef TENSORORDER_HIP_H
#define TENSORORDER_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* status codes */
#define TO_OK 0
#define TO_ERR_OOM 1     /* caller should slice more: tensor_network.OutOfMemoryError */
#define TO_ERR_INVALID 2 /* malformed launch record or descriptor */
#define TO_ERR_HIP 3     /* HIP runtime error; see to_last_error() */

/* entry types */
#define TO_F64 0
#define TO_F32S 1

/* launch record op codes */
#define TO_OP_LEAF_GATHER 1  /* descs: to_leaf_desc[count] */
#define TO_OP_JOIN_STREAM 2  /* descs: to_join_desc[count]; variant = y values per thread (YC),
                                or TO_STREAM_VEC | YC for the 16-byte form: fx >= 10 (float) /
                                9 (double), the lowest 2 / 1 bits of X free, shy == 0,
                                shf == fy, YC == 2^fy, LDS 8*2^s (16-aligned) + YC*2^s entries;
                                or TO_STREAM_ROWS for the row form: shy == 0, shf == fy,
                                5 <= fy <= 10 (float) / 9 (double), fx >= 6, s <= 4, no LDS */
#define TO_STREAM_VEC 0x100
#define TO_STREAM_ROWS 0x200
#define TO_STREAM_ANY 0x400  /* one launch of streamed joins of mixed variants, each given by
                                its descriptor's kvar; lds = the largest any of them needs */
#define TO_STREAM_WAVE 0x800 /* one wave (64 lanes) per join, for small joins (s <= 6, ranks
                                of X, Y and C below 32): descriptor i is run by wave i % 4
                                of block i / 4 (grid >= count / 4, rounded up; block0 /
                                nblocks / kvar unread), no LDS */
#define TO_OP_JOIN_SPLITK 3  /* descs: to_join_desc[count]; partial sums (double) to d.partial */
#define TO_OP_JOIN_FINISH 4  /* descs: to_join_desc[count]; sums d.partial into C; variant 1:
                                one block per output (for nsplit >= 32); | TO_FINISH_NORM
                                (TO_F32S, fx == fy == 0): the result is stored as its mantissa,
                                its exponent added to the record's */
#define TO_FINISH_NORM 0x100
#define TO_OP_SCALE_CLEAR 5  /* aux0: to_scale_rec*, iaux0: record count */
#define TO_OP_ROOT_REDUCE 6  /* aux0: root values, aux1: to_scale_rec* (F32S) or 0,
                                aux2: to_accum*, aux3: wave params (int64[2]); variant 1: the
                                wave at params[0] == 0 starts the sum anew, and params[0] then
                                advances by iaux0, back to 0 after the last wave; iaux1: 0, or
                                the address of a to_accum in host memory that the device can
                                write, which gets a copy of the sum and then, in pad, the
                                number of sums written so far: a word for to_wait */
#define TO_OP_WAVE_ADVANCE 7 /* aux3: wave params; adds iaux0 to params[0] */
#define TO_OP_STEP_BEGIN 8   /* aux2: to_accum* (zeroed), aux3: wave params (params[0] = 0) */
#define TO_OP_PERMUTE 9      /* descs: to_perm_desc[count]; variant 1: 16-byte chunk kernel,
                                which needs nu == 13 (float) / 12 (double) and 16-byte
                                aligned buffers and strides; variant 3: the same with
                                nu == 14 / 13 (64 KB tiles); variant 0: nu <= 12 */
#define TO_OP_GEMM 10        /* descs: to_gemm_desc[count]; variant bit 0: 128-row output
                                tiles (mlog >= 7), 128 columns (nlog >= 7) or, with bit 1,
                                64 columns (nlog >= 6), instead of 64x64 (>= 6); bit 1: float
                                partial sums accumulated in double every 4 K-steps; bit 2
                                (with bit 0): the product is formed transposed, so a float
                                output with ldcn == 1 is written with 16-byte stores; bit 3
                                (with bit 0): 128x128 tiles (nlog >= 7) at one block per CU,
                                LDS double-buffered (variants 9, 11, 13, 15); bit 4 (float,
                                with bit 0, 128x128 tiles): the product on the bf16 matrix
                                cores, each operand split into three bf16 parts and six
                                partial products summed (with bit 3: variants 25, 27, 29,
                                31; with bit 1, klog >= 7) */
#define TO_OP_ROOT_STORE 11  /* descs: to_root_desc[count]: one instance's root -> its accumulator */
#define TO_OP_BATCH_BEGIN 12 /* aux2: to_accum[iaux0] zeroed; aux3: int64 start time (device clock) */
#define TO_OP_FOLD 14 /* descs: to_fold_desc[count]; variant TO_FOLD_ANY: one output per thread,
                         any bit layout; TO_FOLD_DOT: the same, 4 products per load;
                         TO_FOLD_VEC | y mode << 4 | nreg: the 16-byte form, TO_FOLD_REG | a << 4 |
                         b: a register tile, every descriptor of the launch with that y mode and
                         nreg, or those a and b */
#define TO_OP_FOLD_TREE 15 /* descs: to_tree_desc[count]; iaux0: waves per block (1 to 16, as many
                         as each program has streams); lds: the largest of their LDS needs */
#define TO_OP_FOLD_PAIR 17 /* descs: to_pair_desc[count], all with the same nk[0] >= nk[1]; variant:
                              nk[0] << 4 | nk[1], each at most 2, | TO_PAIR_ONE where no Y has
                              the lowest two o bits */
#define TO_PAIR_ONE 0x100
#define TO_OP_WAVE_BEGIN 16 /* TO_OP_LEAF_GATHER on the first iaux1 blocks of the grid and
                               TO_OP_SCALE_CLEAR (aux0, iaux0) on the others, in one launch:
                               descs: to_leaf_desc[count], whose records are not among those
                               cleared; aux3: wave params */
#define TO_OP_LEAF_BUILD 13  /* descs: to_leaf_build_desc[count]: leaf tables written from their
                                compact descriptions (OR / variable leaves) */

#define TO_MAX_BITS 32

/* One join of a launch group (a record in device memory). */
typedef struct to_join_desc {
    uint64_t x, y, c;          /* device pointers to X, Y, C (element type per entry type) */
    int64_t xb, yb, cb;        /* batch strides in elements (0 = broadcast) */
    uint64_t xs, ys, cs;       /* to_scale_rec* per batch item (TO_F32S), else 0 */
    int64_t xsb, ysb;          /* scale-record batch strides (0 or 1) */
    uint64_t partial;          /* split-K partial sums, double, nsplit per output
                                  (TO_OP_JOIN_SPLITK / _FINISH) */
    int32_t fx, fy, s;         /* X free bits, Y free bits, shared bits */
    int32_t shf, shy;          /* output bit offset of f and of y */
    int32_t nbatch;            /* batch items */
    int32_t block0, nblocks;   /* blocks of this join within its launch */
    int32_t nych;              /* y chunks (stream) */
    int32_t nsplit;            /* k splits (split-K) */
    int32_t lnych;             /* log2(nych) */
    int32_t stage;             /* stream, fx >= 8, bit 0: outputs staged through LDS (shy == 0,
                                  shf == fy, one y chunk; 256 * 2^fy entries after the Y
                                  slab); bit 1: X tile staged (all shared bits of X below
                                  bit 8 + s; 256 * 2^s entries after that) */
    int32_t kvar;              /* stream: this join's own variant (YC, TO_STREAM_VEC | YC or
                                  TO_STREAM_ROWS) when the launch variant is TO_STREAM_ANY */
    int8_t xf_pos[TO_MAX_BITS];
    int8_t xs_pos[TO_MAX_BITS];
    int8_t yf_pos[TO_MAX_BITS];
    int8_t ys_pos[TO_MAX_BITS];
} to_join_desc;

/* One leaf copied per batch item from its table of slice rows. */
typedef struct to_leaf_desc {
    uint64_t src;          /* table: rows x 2^rank entries */
    uint64_t dst;          /* nbatch x 2^rank entries */
    uint64_t coef;         /* int64 [ngroups]: row = sum_g coef[g] * bit_g(slice) */
    uint64_t rec;          /* to_scale_rec* per batch item (TO_F32S), else 0 */
    int64_t exp0;          /* exponent of every stored entry (TO_F32S) */
    int32_t rank, ngroups; /* ngroups = number of slice groups of the whole plan */
    int32_t nbatch;
    int32_t block0, nblocks;
    int32_t pad;
} to_leaf_desc;

/* One leaf table written on the device from its description
 * (src/tensor_network/tensor_network_constructions.py:44-159).  The table holds the 2^rank
 * entries of the leaf with its axes reordered (sliced axes first, as tensor.py:95-119
 * reorders them): table bit q (from the least significant) is bit pos[q] of the leaf's own
 * C-order index i.  With the bits of i as the axis values (axis a is bit rank-1-a):
 *   TO_LEAF_VAR: rank 0 -> val0; i == 0 -> val0; i == 2^rank - 1 -> val1; else 0;
 *   TO_LEAF_OR:  literal bits l = i ^ negmask (negmask: bits of negative literals);
 *                out_bit < 0: val1 if l != 0 else val0;
 *                else val1 if bit out_bit of l == (l without that bit != 0) else val0.
 * val0 / val1 are the values as stored (the weights in float64; their float32 encoding in
 * TO_F32S). */
#define TO_LEAF_VAR 0
#define TO_LEAF_OR 1
typedef struct to_leaf_build_desc {
    uint64_t dst;          /* 2^rank entries */
    double val0, val1;
    int64_t negmask;
    int32_t kind, rank, out_bit;
    int32_t block0, nblocks;
    int32_t pad;
    int8_t pos[TO_MAX_BITS];
} to_leaf_build_desc;
/* Per-tensor, per-batch-item scale (TO_F32S). */
typedef struct to_scale_rec {
    int64_t exp;      /* true value = stored value * 2^exp */
    uint32_t maxbits; /* float bits of max |stored entry| (atomicMax on the bits) */
    uint32_t pad;
} to_scale_rec;

/* Running FP64 sum of slice results: value = mant * 2^exp. */
typedef struct to_accum {
    double mant;
    int64_t exp;
    int64_t count; /* slice results accumulated */
    int64_t pad;
} to_accum;

/* A bit permutation of a batch of rank-r tensors: input bit p goes to output bit
 * out_pos(p).  The tile is the union of the lowest input and output bits (u: input
 * order, v: output order); the remaining bits enumerate tiles. */
typedef struct to_perm_desc {
    uint64_t in, out;
    int64_t inb, outb;   /* batch strides in elements */
    int32_t rank, nu, nrest, nbatch;
    int32_t block0, nblocks;
    int8_t u_in[16];     /* input bit of tile bit j (u order) */
    int8_t v_out[16];    /* output bit of tile bit j (v order) */
    int8_t v2u[16];      /* tile bit j of v order is tile bit v2u[j] of u order */
    int8_t rest_in[32];  /* input bit of rest bit j */
    int8_t rest_out[32]; /* output bit of rest bit j */
} to_perm_desc;

/* A batched dense product C[m][n] = sum_k A[m][k] * B[n][k]: A is 2^mlog x 2^klog and
 * B is 2^nlog x 2^klog, both row-major with k contiguous; C entry (m, n) is stored at
 * c + batch*cb + m*ldcm + n*ldcn.  Requires mlog, nlog >= 6 (mlog >= 7 and nlog >= 7, or
 * nlog >= 6 for the wide form, with 128-row tiles) and klog >= 4 (>= 5 for float with
 * 128-row tiles). */
typedef struct to_gemm_desc {
    uint64_t a, b, c;
    int64_t ab, bb, cb;        /* batch strides in elements (0 = broadcast) */
    int64_t ldcm, ldcn;
    uint64_t as, bs, cs;       /* to_scale_rec* of the operands and result (TO_F32S) */
    int64_t asb, bsb;          /* scale-record batch strides */
    int32_t mlog, nlog, klog;
    int32_t nbatch;
    int32_t block0, nblocks;
    int32_t lsplit;            /* 64x64 form (variants 0, 2) only: 0, or split K into 2^lsplit
                                  parts (K >> lsplit >= 16) whose double partial sums go to c
                                  as double[nbatch << (mlog + nlog)][2^lsplit], output o =
                                  (batch << (mlog + nlog)) | (m << nlog) | n, for a
                                  TO_OP_JOIN_FINISH launch (fx = mlog, fy = nlog, nsplit =
                                  2^lsplit) to add up into C */
    int32_t hlog;              /* batch items come in groups of 2^hlog that share one scale
                                  record (record batch >> hlog; 0: one record per item) */
} to_gemm_desc;

/* A folded join: C[o] = sum_k X[x(o, k)] * Y[y(o, k)], where every tensor is indexed by
 * *variables* (bits) and a variable may be in X, in Y or in both, summed (a k bit) or kept
 * (an o bit) either way.  Edges that COPY (variable) tensors force equal
 * (src/tensor_network/tensor_network.pyx:470-489) are one variable here, so the entries a
 * tensordot would store and multiply as structural zeros do not exist.  The offsets are sums
 * over the set bits of (o, k): entry i of bx / by / bc is what bit i adds to the X, Y and C
 * offset, in elements (0: the tensor does not have that variable; several positions at once
 * for a leaf that has it on several axes).  No two entries of one array overlap.  Bits are
 * listed by the role a kernel gives them:
 *   TO_FOLD_ANY: [0, 8) thread bits (lo of them o bits, then lk k bits, the rest 0);
 *     [8, 8 + ntile) o bits of the tile index; then nloop k bits walked by each thread and
 *     lsplit k bits across blocks.  lk > 0 only when ntile == 0 or lo == 8 - lk.
 *     With lsplit > 0 the double partial sums go to partial[(batch << (lo + ntile) | c) <<
 *     lsplit | sp], c the C offset, for a TO_OP_JOIN_FINISH launch (fx = lo + ntile).
 *   TO_FOLD_DOT: as TO_FOLD_ANY, with two more k bits, not listed, that add 1 and 2 to the
 *     offsets of X and of Y (X, Y and their batch strides aligned to 4 elements).
 *   TO_FOLD_REG: as TO_FOLD_ANY with lo == 8, lk == lsplit == 0; then nreg = a + b o bits, a
 *     that only X has and b that only Y has ((a, b) one of (1, 1), (2, 2), (2, 3), (2, 0)), all 2^nreg of whose outputs a thread holds at once.
 *   TO_FOLD_VEC: [0, 2) the o bits of 4 consecutive outputs, also the lowest 2 bits of X;
 *     [2, 10) o bits of the thread index; [10, 10 + ntile) tile; nloop k bits; nreg (<= 3) o
 *     bits that only Y has, all 2^nreg of whose outputs a thread holds at once.
 *     y mode: 0 Y has neither of the bits [0, 2); 1 both, as its lowest two; 2 any of them, in
 *     any place; 3 the first alone; 4 the second alone; 5 neither, and the first two of the
 *     nreg bits (nreg >= 2) are its lowest.  C, X (and Y in modes 1 and 5) and their batch
 *     strides aligned to 4 elements. */
#define TO_FOLD_ANY 0
#define TO_FOLD_VEC 0x100
#define TO_FOLD_REG 0x200
#define TO_FOLD_DOT 0x400
#define TO_FOLD_BITS 40
typedef struct to_fold_desc {
    uint64_t x, y, c;
    int64_t xb, yb, cb;        /* batch strides in elements (0 = broadcast) */
    uint64_t xs, ys, cs;       /* to_scale_rec* per batch item (TO_F32S), else 0 */
    int64_t xsb, ysb;          /* scale-record batch strides (0 or 1) */
    uint64_t partial;
    int32_t nbatch;
    int32_t block0, nblocks;
    int32_t lo, lk, ntile, nloop, lsplit, nreg;
    int32_t pad;
    uint32_t bx[TO_FOLD_BITS], by[TO_FOLD_BITS], bc[TO_FOLD_BITS];
} to_fold_desc;

/* The dot product of two folded joins that are not stored: C = sum_o (sum_i X0 Y0) (sum_j X1 Y1),
 * o over the variables of both joins' results, i and j over what each sums (nk[0], nk[1]
 * variables).  Entry b of bx[side] / by[side] is what bit b adds to that side's offsets, in
 * elements.  Bits: [0, 2) o bits that add 1 and 2 to both X; [2, 10) o bits of the thread
 * index; then nloop o bits walked by each thread, lsplit o bits across blocks, nreg o bits that
 * X0 lacks (its entries are loaded once for them), nk[0] bits i, nk[1] bits j.  X and its batch strides are aligned to 4
 * elements.  With lsplit > 0 the double partial sums go to
 * partial[batch << lsplit | sp] for a TO_OP_JOIN_FINISH launch, and rs[side], where not 0, gets
 * the exponent of its side (TO_F32S): the records that launch reads in place of the stored
 * results'.  The results' maxima are not known: the sum is stored as its mantissa, its exponent
 * added to the record's (with lsplit > 0 by TO_FINISH_NORM). */
typedef struct to_pair_desc {
    uint64_t x[2], y[2], c;
    int64_t xb[2], yb[2], cb;  /* batch strides in elements (0 = broadcast) */
    uint64_t xs[2], ys[2], cs; /* to_scale_rec* per batch item (TO_F32S), else 0; ys also 0 for a
                                  Y of ones */
    int64_t xsb[2], ysb[2];
    uint64_t rs[2], partial;
    int32_t nbatch;
    int32_t block0, nblocks;
    int32_t nloop, lsplit, nreg;
    int32_t nk[2];
    uint32_t bx[2][TO_FOLD_BITS], by[2][TO_FOLD_BITS];
} to_pair_desc;

/* A program of small folded joins that one block runs start to end for one batch item: a
 * connected part of the tree whose intermediate tensors fit LDS.  A join of a program is a
 * product of up to 4 tensors, summed over the k bits; one of 3 or 4 is stored scaled by the power
 * of two that brings its largest entry to [0.5, 1), which its record's exponent carries
 * (TO_F32S).  Each wave of the block walks its own stream of ntask words,
 * tasks[wave * ntask + i]: bits 0-15 the join, bits 16-22 its first
 * chunk of 64 outputs-times-shares and bits 23-26 log2 of the step to the next one, bit 30:
 * nothing to do, bit 31: all waves meet after this entry (in the same entries of every
 * stream).  A join is TO_TREE_WORDS words, ops[join * TO_TREE_WORDS + i]:
 *   0: lo | lk << 4 | nloop << 8 | nchunk << 12 (numbers of o bits and k bits on the lanes, of
 *      k bits walked, of o bits of the chunk index; 6 + nloop + nchunk at most 16),
 *      operands - 1 in bits 16-17, bits 20-24: operand 0-3, result lie in LDS, bits 25-29:
 *      their global scale record advances with the batch item; 3 or 4 operands only with
 *      nchunk == 0 and nloop <= 2
 *   1 + 2 j, 2 + 2 j: address of operand j (result: j = 4), low word first, or its element
 *      offset in the block's LDS tensors; 11 + j: its batch stride in elements (global);
 *      16 + j: its scale record: an LDS slot for an LDS tensor, else an index into recs
 *   32-47: what each bit adds to the result's offset, 64 + 16 j + i: to operand j's (as in
 *      to_fold_desc): 6 lane bits (lo o bits, lk k bits, the rest 0), nchunk, nloop
 *   128 + 64 j + l: the offset that the lane bits of lane l add to operand j's (result's).
 * LDS holds nslots 8-byte records, then (16-byte aligned) the tensors. */
#define TO_TREE_WORDS 448
#define TO_TREE_IDLE 0x40000000
#define TO_TREE_MEET 0x80000000
typedef struct to_tree_desc {
    uint64_t ops, tasks;       /* uint32 arrays in device memory */
    uint64_t recs;             /* to_scale_rec* of the program's global tensors (TO_F32S) */
    int32_t ntask, nslots;
    int32_t block0, nblocks;   /* one block per batch item */
} to_tree_desc;

/* The root scalar of one instance of a batch: stored into its accumulator as
 * (mantissa, exponent), with the device clock at that moment in accum.pad. */
typedef struct to_root_desc {
    uint64_t root; /* the rank-0 result */
    uint64_t rec;  /* its to_scale_rec (TO_F32S) or 0 */
    uint64_t acc;  /* to_accum* */
    int32_t block0, nblocks;
} to_root_desc;

/* One kernel launch. */
typedef struct to_launch {
    int32_t op;
    int32_t variant;
    int32_t count;  /* descriptors */
    int32_t grid;   /* blocks (256 threads each) */
    int32_t lds;    /* dynamic LDS bytes */
    int32_t flags;  /* TO_LAUNCH_* (graph capture only; to_run runs records in order) */
    uint64_t descs; /* device pointer to the descriptor array */
    uint64_t aux0, aux1, aux2, aux3; /* per op; for the descriptor-table ops (LEAF_GATHER,
                                        JOIN_STREAM, JOIN_SPLITK, JOIN_FINISH, PERMUTE, GEMM,
                                        FOLD, FOLD_TREE, LEAF_BUILD) aux1 is 0 or a device int32[grid] map of
                                        each block to its descriptor (the last one whose
                                        block0 is at or below the block), read instead of a
                                        binary search over block0 (TO_STREAM_WAVE launches
                                        ignore it: block and wave fix the descriptor) */
    int64_t iaux0, iaux1;
} to_launch;

/* to_launch.flags, read by to_graph_create: the record runs on a second captured stream
 * (SIDE), and/or the side stream is joined into the main one and forked from it again
 * before the record (JOIN), so SIDE records between two JOINs run beside the main ones. */
#define TO_LAUNCH_SIDE 0x1
#define TO_LAUNCH_JOIN 0x2

/* Library ABI version (bumped when a struct layout changes). */
int to_version(void);

/* Size in bytes of each record type, for host-side layout checks. */
int to_struct_sizes(int64_t* join_desc, int64_t* leaf_desc, int64_t* scale_rec,
                     int64_t* accum, int64_t* launch, int64_t* perm_desc, int64_t* gemm_desc,
                     int64_t* root_desc, int64_t* leaf_build_desc);

/* Size in bytes of to_fold_desc and to_tree_desc, for the same check. */
int to_fold_desc_size(void);
int to_tree_desc_size(void);
int to_pair_desc_size(void);

/* Last error message of the calling thread ("" when none). */
const char* to_last_error(void);

/* Number of visible HIP devices. */
int to_device_count(int* count);

/* Select the device for subsequent calls on this thread. */
int to_set_device(int device);

/* Launch the records in order on `stream` (hipStream_t, 0 = default stream).
 * Replaces the per-node tensordot calls of one post-order walk
 * (src/tensor_network/tensor_network.pyx:142-156) for a whole batch of slices. */
int to_run(const to_launch* launches, int count, int entry_type, void* stream);

/* As to_run, recording a HIP event before each record and after the last on `stream`;
 * waits for completion and stores each record's device time in ms[i] (count floats). */
int to_run_timed(const to_launch* launches, int count, int entry_type, void* stream, float* ms);

/* Capture the records into a HIP graph once; replay it with to_graph_launch.  Records
 * flagged TO_LAUNCH_SIDE are captured on a second stream (created and destroyed here,
 * default priority) between TO_LAUNCH_JOIN points; the graph ends joined. */
int to_graph_create(const to_launch* launches, int count, int entry_type, void* stream,
                    void** graph_exec);
int to_graph_launch(void* graph_exec, void* stream);
int to_graph_destroy(void* graph_exec);

/* Reorder the axes of a rank-r all-dimension-2 tensor: out axis j = in axis perm[j],
 * as numpy.transpose (used by tensor_apis/jax_apis.py:83-88, 146-162 and by
 * tensor.py:112-117).  Element size 4 or 8 bytes. */
int to_permute(const void* in, void* out, int rank, const int32_t* perm, int elem_bytes,
               int64_t batch, void* stream);

/* numpy.tensordot(a, b, (axes_a, axes_b)) of two all-dimension-2 tensors on the device:
 * the per-join primitive of the reference's post-order walk
 * (src/tensor_network/tensor_network.pyx:152-154 -> tensor_apis/numpy_apis.py:42-43).
 * c receives 2^(rank_a + rank_b - 2 nshared) entries in numpy's axis order (a's unshared
 * axes in order, then b's); ranks <= 30, output rank <= 30; c must not overlap a or b.
 * TO_F64: float64 tensors, the records are ignored.  TO_F32S: float32 tensors with one
 * to_scale_rec each (a_rec, b_rec read; c_rec written).  One streamed join, or, for many
 * shared axes and few outputs, split-K partial sums in double in `workspace` (8-byte
 * aligned; to_tensordot_workspace gives the bytes, 0 when none are needed) and a
 * fixed-order finishing sum.  Asynchronous on `stream`. */
int to_tensordot_workspace(int rank_a, int rank_b, const int32_t* axes_a, const int32_t* axes_b,
                           int nshared, int entry_type, int64_t* bytes);
int to_tensordot(const void* a, const void* b, void* c, int rank_a, int rank_b,
                 const int32_t* axes_a, const int32_t* axes_b, int nshared, int entry_type,
                 const void* a_rec, const void* b_rec, void* c_rec, void* workspace,
                 int64_t workspace_bytes, void* stream);
/* to_tensordot without the workspace arguments, for callers that cannot allocate device
 * memory (code under HIP graph capture, tight serving loops, harnesses that forbid
 * hipMalloc); it has no counterpart in the reference.  It allocates nothing: the split-K
 * partial sums go to a file-scope device array of 8 MiB (1M doubles) that each GPU holds
 * until the process ends; a call needing more (to_tensordot_workspace > 8 MiB) returns
 * TO_ERR_INVALID.  Every call on one GPU shares that GPU's array: calls that overlap on
 * one GPU (other streams, other threads) race and must be serialised by the caller. */
int to_tensordot_noalloc(const void* a, const void* b, void* c, int rank_a, int rank_b,
                         const int32_t* axes_a, const int32_t* axes_b, int nshared, int entry_type,
                         const void* a_rec, const void* b_rec, void* c_rec, void* stream);
/* Copy `bytes` (a multiple of 4) of host memory at `src` to 4-byte aligned device memory at
 * `dst`, in stream order: the data travel in kernel arguments, up to 3 KB a launch, so the host
 * memory may be reused as soon as the call returns and nothing waits.  For descriptors and
 * other small records; a copy engine is faster above some 16 KB. */
int to_upload(void* dst, const void* src, int64_t bytes, void* stream);

/* Frequency of the device clock stamped by TO_OP_ROOT_STORE / TO_OP_BATCH_BEGIN, in kHz. */
int to_wall_clock_khz(int* khz);

/* Block until all work on `stream` is done. */
int to_synchronize(void* stream);

/* Store `value` in the host word *word (host memory that the device writes) once the work now
 * on `stream` is done; to_wait spins on such a word for up to 2 ms, then blocks as
 * to_synchronize does, and returns when *word >= value or the stream is idle.  The work of a
 * stream is then seen to end without the stream's own completion marker. */
int to_signal(int64_t* word, int64_t value, void* stream);
int to_wait(const int64_t* word, int64_t value, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* TENSORORDER_HIP_H */
