// Folded joins (to_fold_desc): part of tensororder_hip.hip, inside its anonymous namespace.
//
// A join over variables: edges forced equal by COPY tensors are one index bit, which may be
// in both operands and in the result at once, so no structural zero is stored, moved or
// multiplied.  On the 70-variable 4096-slice formula that is 2^26 instead of 2^34 products
// and 2^25 instead of 2^27 entries per slice (the plan the learned model picks), so nearly
// every join reads a large tensor once, multiplies it by a small one and writes it once:
// bound by HBM, not by the matrix cores.

// Offsets of a deposit: bit i of v adds row entry first + i (held by lane first + i).  The
// entries of one row never overlap, so sums are ors.
__device__ __forceinline__ uint32_t fold_dep(uint32_t v, uint32_t row, int first, int n) {
    uint32_t r = 0;
    for (int i = 0; i < n; ++i) r |= (0u - ((v >> i) & 1u)) & (uint32_t)__builtin_amdgcn_readlane((int)row, first + i);
    return r;
}

struct FoldRows {
    uint32_t x, y, c;
};

// lane i < TO_FOLD_BITS holds the bit entries i (one load per lane and tensor)
__device__ __forceinline__ FoldRows fold_rows(const to_fold_desc* __restrict__ d) {
    const int lane = threadIdx.x & 63;
    const int i = lane < TO_FOLD_BITS ? lane : TO_FOLD_BITS - 1;
    return FoldRows{d->bx[i], d->by[i], d->bc[i]};
}

// Walk 2^nloop shared indices (bit entries from lane `first` of row.x and lane ylanes + first
// of row.y) in Gray-code order, so each step of KU indices changes one bit
// above them: f(dx, dy) gets the KU x / y offsets of a step (inside it the low bits follow
// Gray order too, so the walk is a bijection).
template <int KU, typename F>
__device__ __forceinline__ void fold_walk(uint32_t xk, uint32_t yk, const FoldRows& row, int first, int ylanes,
                                          int nloop, F f) {
    constexpr int LKU = KU == 4 ? 2 : (KU == 2 ? 1 : 0);
    uint32_t dx[KU], dy[KU];
    dx[0] = dy[0] = 0;
    if constexpr (KU >= 2) {
        dx[1] = (uint32_t)__builtin_amdgcn_readlane((int)row.x, first);
        dy[1] = (uint32_t)__builtin_amdgcn_readlane((int)row.y, ylanes + first);
    }
    if constexpr (KU == 4) {
        const uint32_t bx = (uint32_t)__builtin_amdgcn_readlane((int)row.x, first + 1);
        const uint32_t by = (uint32_t)__builtin_amdgcn_readlane((int)row.y, ylanes + first + 1);
        dx[2] = dx[1] | bx;
        dx[3] = bx;
        dy[2] = dy[1] | by;
        dy[3] = by;
    }
    const uint32_t steps = 1u << (nloop - LKU);
    for (uint32_t k = 1;; ++k) {
        uint32_t ox[KU], oy[KU];
#pragma unroll
        for (int j = 0; j < KU; ++j) {
            ox[j] = xk ^ dx[j];
            oy[j] = yk ^ dy[j];
        }
        f(ox, oy);
        if (k == steps) break;
        const int b = first + LKU + __builtin_ctz(k);
        xk ^= (uint32_t)__builtin_amdgcn_readlane((int)row.x, b);
        yk ^= (uint32_t)__builtin_amdgcn_readlane((int)row.y, ylanes + b);
    }
}

// Scale of a batch item's result: the operands' power-of-two factors (applied to the sums,
// which are in double, so exactly) and the exponent they carry.
struct FoldScale {
    double f;
    int64_t e;
};

template <bool SCALED>
__device__ __forceinline__ FoldScale fold_scale(const to_fold_desc* __restrict__ d, int64_t batch) {
    if (!SCALED) return FoldScale{1.0, 0};
    const OpScale a = op_scale(d->xs, d->xsb, batch), b = op_scale(d->ys, d->ysb, batch);
    return FoldScale{(double)a.f * (double)b.f, a.e + b.e};
}

// Largest of the wave's words, the same in every lane: row shifts and row broadcasts (VALU only),
// where shuffles would go through LDS six times
__device__ __forceinline__ uint32_t fold_wave_umax(uint32_t m) {
    auto step = [&](auto ctrl) {
        const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, decltype(ctrl)::value, 0xf, 0xf, true);
        m = o > m ? o : m;
    };
    step(std::integral_constant<int, 0x111>{});  // row_shr:1, 2, 4, 8
    step(std::integral_constant<int, 0x112>{});
    step(std::integral_constant<int, 0x114>{});
    step(std::integral_constant<int, 0x118>{});
    step(std::integral_constant<int, 0x142>{});  // row_bcast:15, 31
    step(std::integral_constant<int, 0x143>{});
    return (uint32_t)__builtin_amdgcn_readlane((int)m, 63);
}

// ... of its non-negative floats, which compare as their bits
__device__ __forceinline__ float fold_wave_max(float v) { return __uint_as_float(fold_wave_umax(__float_as_uint(v))); }

// Sum over thread bits [lo, lo + lk) of a 256-thread block: shuffles inside a wave, LDS
// across waves, both in a fixed order.  The sums are valid where those bits are zero.
__device__ __forceinline__ double fold_reduce(double v, int lo, int lk, double* red) {
    const int tid = threadIdx.x;
    const int hi = lo + lk;
    for (int b = lo; b < hi && b < 6; ++b) v += __shfl_xor(v, 1 << b, 64);
    if (hi > 6) {
        __syncthreads();
        red[tid] = v;
        __syncthreads();
        const int w0 = lo > 6 ? lo : 6;
        double s = 0.0;
        for (int j = 0; j < (1 << (hi - w0)); ++j) s += red[(tid & ~(((1 << (hi - w0)) - 1) << w0)) | (j << w0)];
        v = s;
    }
    return v;
}

// General form: one output per thread, or one share of an output's shared range (lk thread
// bits), any bit layout.  Products of floats are exact in the double sums, which are rounded
// once, when stored.
// DOT: every shared index is four consecutive ones of X and of Y (16 or 32 bytes per load):
// 4096 dot products of 2^20 floats in 5.6 ms (6.1 TB/s), 15 with 4-byte loads.
template <typename T, bool SCALED, bool DOT>
__device__ __forceinline__ void fold_any_body(const to_fold_desc* __restrict__ d, const int local, double* red) {
    const int tid = threadIdx.x;
    const FoldRows row = fold_rows(d);
    const int lo = d->lo, lk = d->lk, ntile = d->ntile, nloop = d->nloop, lsplit = d->lsplit;
    const int nthr = lo + lk;
    const TO_GLOBAL T* __restrict__ X = gptr<const T>(d->x);
    const TO_GLOBAL T* __restrict__ Y = gptr<const T>(d->y);
    TO_GLOBAL T* __restrict__ C = gptr<T>(d->c);
    const int kb = 8 + ntile;
    const uint32_t xl = fold_dep(tid, row.x, 0, nthr), yl = fold_dep(tid, row.y, 0, nthr);
    const uint32_t cl = fold_dep(tid, row.c, 0, lo);
    const bool active = tid < (1 << nthr);
    const bool writer = tid < (1 << lo);
    const int64_t n = (int64_t)d->nbatch << (ntile + lsplit);
    const int64_t t0 = n * local / d->nblocks, t1 = n * (local + 1) / d->nblocks;
    int64_t cur = -1;
    FoldScale sc{1.0, 0};
    float mrun = 0.0f;
    for (int64_t t = t0; t < t1; ++t) {
        const uint32_t sp = (uint32_t)t & ((1u << lsplit) - 1);
        const uint32_t tile = (uint32_t)(t >> lsplit) & ((1u << ntile) - 1);
        const int64_t batch = t >> (lsplit + ntile);
        if (SCALED && batch != cur) {
            if (cur >= 0 && lsplit == 0) {
                const float w = fold_wave_max(mrun);
                if ((tid & 63) == 0) note_max(d->cs, cur, w);
                mrun = 0.0f;
            }
            sc = fold_scale<SCALED>(d, batch);
            cur = batch;
        }
        const uint32_t xt = fold_dep(tile, row.x, 8, ntile) | fold_dep(sp, row.x, kb + nloop, lsplit);
        const uint32_t yt = fold_dep(tile, row.y, 8, ntile) | fold_dep(sp, row.y, kb + nloop, lsplit);
        const uint32_t co = fold_dep(tile, row.c, 8, ntile) | cl;
        double acc = 0.0, part[4] = {0.0, 0.0, 0.0, 0.0};
        if (active) {
            const TO_GLOBAL T* Xp = X + batch * d->xb + xl;
            const TO_GLOBAL T* Yp = Y + batch * d->yb + yl;
            auto walk = [&](auto ku) {
                constexpr int KU = decltype(ku)::value;
                fold_walk<KU>(xt, yt, row, kb, 0, nloop, [&](const uint32_t* ox, const uint32_t* oy) {
                    if constexpr (DOT) {
                        typedef T V4 __attribute__((ext_vector_type(4)));
                        V4 xv[KU], yv[KU];
#pragma unroll
                        for (int j = 0; j < KU; ++j) {
                            xv[j] = *reinterpret_cast<const TO_GLOBAL V4*>(Xp + ox[j]);
                            yv[j] = *reinterpret_cast<const TO_GLOBAL V4*>(Yp + oy[j]);
                        }
#pragma unroll
                        for (int j = 0; j < KU; ++j)
#pragma unroll
                            for (int v = 0; v < 4; ++v) part[v] = fma((double)xv[j][v], (double)yv[j][v], part[v]);
                    } else {
                        T xv[KU], yv[KU];
#pragma unroll
                        for (int j = 0; j < KU; ++j) {
                            xv[j] = Xp[ox[j]];
                            yv[j] = Yp[oy[j]];
                        }
#pragma unroll
                        for (int j = 0; j < KU; ++j) acc = fma((double)xv[j], (double)yv[j], acc);
                    }
                });
            };
            if (nloop >= 2) walk(std::integral_constant<int, 4>{});
            else if (nloop == 1) walk(std::integral_constant<int, 2>{});
            else walk(std::integral_constant<int, 1>{});
        }
        if (DOT) acc = (part[0] + part[1]) + (part[2] + part[3]);
        if (lk > 0) acc = fold_reduce(acc, lo, lk, red);
        if (writer) {
            if (lsplit > 0) {
                gptr<double>(d->partial)[((((uint64_t)batch << (lo + ntile)) | co) << lsplit) | sp] = SCALED ? acc * sc.f : acc;
            } else {
                const T v = (T)(SCALED ? acc * sc.f : acc);
                C[batch * d->cb + co] = v;
                if (SCALED) {
                    mrun = fmaxf(mrun, (float)absval(v));
                    if (tid == 0 && tile == 0) note_exp(d->cs, batch, sc.e);
                }
            }
        }
    }
    if (SCALED && cur >= 0 && lsplit == 0) {
        const float w = fold_wave_max(mrun);
        if ((tid & 63) == 0) note_max(d->cs, cur, w);
    }
}

template <typename T, bool SCALED, bool DOT>
__global__ __launch_bounds__(kBlock) void k_fold_any(const to_fold_desc* __restrict__ descs, int ndesc, const int32_t* __restrict__ bmap) {
    __shared__ double red[kBlock];
    const to_fold_desc* d = descs + find_desc(descs, ndesc, blockIdx.x, bmap);
    fold_any_body<T, SCALED, DOT>(d, blockIdx.x - d->block0, red);
}

// Register tile: a thread owns the 2^A by 2^B outputs of A variables only X has and B only Y
// has, and loads 2^A + 2^B entries for their products; the lanes run along the lowest other
// variables of the result.  For the joins of two mid-sized tensors each of which has one of the
// result's two lowest variables alone, so that neither streams in the 16-byte form, where the
// one-output form loads two entries a product.  Scaled floats, one-output form / tile: 4096 slices
// of 2^8 by 2^6 over 2 to 2^12 95 / 19 us; 64 of 2^16 by 2^13 over 2^2 to 2^20 631 / 84; 1024 of
// 2^14 by 2^11 over 2^3 to 2^16 544 / 112; 256 of 2^16 by 2^14 over 2^8 to 2^13 181 / 73.
template <typename T, bool SCALED, int A, int B>
__global__ __launch_bounds__(kBlock) void k_fold_reg(const to_fold_desc* __restrict__ descs, int ndesc, const int32_t* __restrict__ bmap) {
    constexpr int NX = 1 << A, NY = 1 << B;
    const to_fold_desc* d = descs + find_desc(descs, ndesc, blockIdx.x, bmap);
    const int local = blockIdx.x - d->block0;
    const int tid = threadIdx.x;
    const FoldRows row = fold_rows(d);
    const int ntile = d->ntile, nloop = d->nloop;
    const int kb = 8 + ntile, rb = kb + nloop;
    const TO_GLOBAL T* __restrict__ X = gptr<const T>(d->x);
    const TO_GLOBAL T* __restrict__ Y = gptr<const T>(d->y);
    TO_GLOBAL T* __restrict__ C = gptr<T>(d->c);
    const uint32_t xl = fold_dep(tid, row.x, 0, 8), yl = fold_dep(tid, row.y, 0, 8), cl = fold_dep(tid, row.c, 0, 8);
    uint32_t rx[NX], ry[NY], cx[NX], cy[NY];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
        rx[i] = fold_dep(i, row.x, rb, A);
        cx[i] = fold_dep(i, row.c, rb, A);
    }
#pragma unroll
    for (int j = 0; j < NY; ++j) {
        ry[j] = fold_dep(j, row.y, rb + A, B);
        cy[j] = fold_dep(j, row.c, rb + A, B);
    }
    const int64_t n = (int64_t)d->nbatch << ntile;
    const int64_t t0 = n * local / d->nblocks, t1 = n * (local + 1) / d->nblocks;
    int64_t cur = -1;
    FoldScale sc{1.0, 0};
    float mrun = 0.0f;
    for (int64_t t = t0; t < t1; ++t) {
        const uint32_t tile = (uint32_t)t & ((1u << ntile) - 1);
        const int64_t batch = t >> ntile;
        if (SCALED && batch != cur) {
            if (cur >= 0) {
                const float w = fold_wave_max(mrun);
                if ((tid & 63) == 0) note_max(d->cs, cur, w);
                mrun = 0.0f;
            }
            sc = fold_scale<SCALED>(d, batch);
            cur = batch;
        }
        const TO_GLOBAL T* Xp = X + batch * d->xb + xl;
        const TO_GLOBAL T* Yp = Y + batch * d->yb + yl;
        const uint32_t xt = fold_dep(tile, row.x, 8, ntile), yt = fold_dep(tile, row.y, 8, ntile);
        TO_GLOBAL T* Cp = C + batch * d->cb + (fold_dep(tile, row.c, 8, ntile) | cl);
        double acc[NX][NY];
#pragma unroll
        for (int i = 0; i < NX; ++i)
#pragma unroll
            for (int j = 0; j < NY; ++j) acc[i][j] = 0.0;
        auto walk = [&](auto ku) {
            constexpr int KU = decltype(ku)::value;
            fold_walk<KU>(xt, yt, row, kb, 0, nloop, [&](const uint32_t* ox, const uint32_t* oy) {
                T xv[KU][NX], yv[KU][NY];
#pragma unroll
                for (int k = 0; k < KU; ++k) {
#pragma unroll
                    for (int i = 0; i < NX; ++i) xv[k][i] = Xp[ox[k] | rx[i]];
#pragma unroll
                    for (int j = 0; j < NY; ++j) yv[k][j] = Yp[oy[k] | ry[j]];
                }
#pragma unroll
                for (int k = 0; k < KU; ++k)
#pragma unroll
                    for (int i = 0; i < NX; ++i)
#pragma unroll
                        for (int j = 0; j < NY; ++j) acc[i][j] = fma((double)xv[k][i], (double)yv[k][j], acc[i][j]);
            });
        };
        if (nloop >= 1) walk(std::integral_constant<int, 2>{});
        else walk(std::integral_constant<int, 1>{});
#pragma unroll
        for (int i = 0; i < NX; ++i)
#pragma unroll
            for (int j = 0; j < NY; ++j) {
                const T v = (T)(SCALED ? acc[i][j] * sc.f : acc[i][j]);
                Cp[cx[i] | cy[j]] = v;
                if (SCALED) mrun = fmaxf(mrun, (float)absval(v));
            }
        if (SCALED && tid == 0 && tile == 0) note_exp(d->cs, batch, sc.e);
    }
    if (SCALED && cur >= 0) {
        const float w = fold_wave_max(mrun);
        if ((tid & 63) == 0) note_max(d->cs, cur, w);
    }
}

// 16-byte form for the large joins: a thread owns 4 consecutive outputs times the 2^RY
// outputs of the register bits (variables only Y has), so an X entry is loaded once for all
// of them, 16 bytes at a time; Y is read through L1, with as few loads as the places of the
// outputs' two lowest variables and of the register variables in it allow (YM).  Bound by the
// HBM bytes of X and C where few indices are summed: 2^19 by 2^15 over 2 to 2^20, 4096 slices
// (26 GB), 5.3-5.7 ms, the rate of a copy.  2^16 by 2^16 over 2^3 to 2^20 (19 GB) takes 5.7 ms: its
// stores alone take 3.0, the loads and double products alone 2.7, and the address units are
// busy for 84 % of the time.  Tried there: loads one step ahead of the products and the stores
// (6.7 ms, more registers), nontemporal stores (5.7), half the register outputs (6.8), blocks
// of one XCD on neighbouring tiles (5.8), 4 and 16 times the blocks (5.8, 5.9).
template <typename T, bool SCALED, int RY, int YM>
__global__ __launch_bounds__(kBlock) void k_fold_vec(const to_fold_desc* __restrict__ descs, int ndesc, const int32_t* __restrict__ bmap) {
    constexpr int R = 1 << RY;
    constexpr int KMAX = RY >= 2 ? 2 : 4;  // shared indices in flight
    typedef T V4 __attribute__((ext_vector_type(4)));
    const to_fold_desc* d = descs + find_desc(descs, ndesc, blockIdx.x, bmap);
    const int local = blockIdx.x - d->block0;
    const int tid = threadIdx.x;
    const FoldRows row = fold_rows(d);
    const int ntile = d->ntile, nloop = d->nloop;
    const int kb = 10 + ntile, rb = kb + nloop;
    const TO_GLOBAL T* __restrict__ X = gptr<const T>(d->x);
    const TO_GLOBAL T* __restrict__ Y = gptr<const T>(d->y);
    TO_GLOBAL T* __restrict__ C = gptr<T>(d->c);
    const uint32_t xl = fold_dep(tid, row.x, 2, 8), yl = fold_dep(tid, row.y, 2, 8), cl = fold_dep(tid, row.c, 2, 8);
    uint32_t ry[R], rc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        ry[r] = fold_dep(r, row.y, rb, RY);
        rc[r] = fold_dep(r, row.c, rb, RY);
    }
    const uint32_t y1 = (uint32_t)__builtin_amdgcn_readlane((int)row.y, 0);
    const uint32_t y2 = (uint32_t)__builtin_amdgcn_readlane((int)row.y, 1);
    const int64_t n = (int64_t)d->nbatch << ntile;
    const int64_t t0 = n * local / d->nblocks, t1 = n * (local + 1) / d->nblocks;
    int64_t cur = -1;
    FoldScale sc{1.0, 0};
    float mrun = 0.0f;
    for (int64_t t = t0; t < t1; ++t) {
        const uint32_t tile = (uint32_t)t & ((1u << ntile) - 1);
        const int64_t batch = t >> ntile;
        if (SCALED && batch != cur) {
            if (cur >= 0) {
                const float w = fold_wave_max(mrun);
                if ((tid & 63) == 0) note_max(d->cs, cur, w);
                mrun = 0.0f;
            }
            sc = fold_scale<SCALED>(d, batch);
            cur = batch;
        }
        const TO_GLOBAL T* Xp = X + batch * d->xb + xl;
        const TO_GLOBAL T* Yp = Y + batch * d->yb + yl;
        const uint32_t xt = fold_dep(tile, row.x, 10, ntile), yt = fold_dep(tile, row.y, 10, ntile);
        TO_GLOBAL T* Cp = C + batch * d->cb + (fold_dep(tile, row.c, 10, ntile) | cl);
        double acc[R][4];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[r][v] = 0.0;
        auto walk = [&](auto ku) {
            constexpr int KU = decltype(ku)::value;
            fold_walk<KU>(xt, yt, row, kb, 0, nloop, [&](const uint32_t* ox, const uint32_t* oy) {
                V4 xv[KU];
#pragma unroll
                for (int j = 0; j < KU; ++j) xv[j] = *reinterpret_cast<const TO_GLOBAL V4*>(Xp + ox[j]);
                if constexpr (YM == 5) {  // four register outputs' entries lie together
                    V4 yv[KU][R / 4];
#pragma unroll
                    for (int j = 0; j < KU; ++j)
#pragma unroll
                        for (int r = 0; r < R / 4; ++r)
                            yv[j][r] = *reinterpret_cast<const TO_GLOBAL V4*>(Yp + (oy[j] | ry[4 * r]));
#pragma unroll
                    for (int j = 0; j < KU; ++j)
#pragma unroll
                        for (int r = 0; r < R; ++r)
#pragma unroll
                            for (int v = 0; v < 4; ++v)
                                acc[r][v] = fma((double)xv[j][v], (double)yv[j][r / 4][r & 3], acc[r][v]);
                    return;
                }
#pragma unroll
                for (int j = 0; j < KU; ++j) {
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const TO_GLOBAL T* p = Yp + (oy[j] | ry[r]);
                        if constexpr (YM == 0) {
                            const double y = (double)*p;
#pragma unroll
                            for (int v = 0; v < 4; ++v) acc[r][v] = fma((double)xv[j][v], y, acc[r][v]);
                        } else if constexpr (YM == 1) {
                            const V4 y = *reinterpret_cast<const TO_GLOBAL V4*>(p);
#pragma unroll
                            for (int v = 0; v < 4; ++v) acc[r][v] = fma((double)xv[j][v], (double)y[v], acc[r][v]);
                        } else if constexpr (YM == 2) {
                            const T y[4] = {p[0], p[y1], p[y2], p[y1 | y2]};
#pragma unroll
                            for (int v = 0; v < 4; ++v) acc[r][v] = fma((double)xv[j][v], (double)y[v], acc[r][v]);
                        } else {  // Y has one of the outputs' two lowest variables
                            const double a = (double)p[0], b = (double)p[YM == 3 ? y1 : y2];
#pragma unroll
                            for (int v = 0; v < 4; ++v)
                                acc[r][v] = fma((double)xv[j][v], (YM == 3 ? v & 1 : v >> 1) ? b : a, acc[r][v]);
                        }
                    }
                }
            });
        };
        if (KMAX == 4 && nloop >= 2) walk(std::integral_constant<int, KMAX>{});
        else if (nloop >= 1) walk(std::integral_constant<int, 2>{});
        else walk(std::integral_constant<int, 1>{});
#pragma unroll
        for (int r = 0; r < R; ++r) {
            V4 o;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                o[v] = (T)(SCALED ? acc[r][v] * sc.f : acc[r][v]);
                if (SCALED) mrun = fmaxf(mrun, (float)absval(o[v]));
            }
            *reinterpret_cast<TO_GLOBAL V4*>(Cp + rc[r]) = o;
        }
        if (SCALED && tid == 0 && tile == 0) note_exp(d->cs, batch, sc.e);
    }
    if (SCALED && cur >= 0) {
        const float w = fold_wave_max(mrun);
        if ((tid & 63) == 0) note_max(d->cs, cur, w);
    }
}

// The dot product of two joins' results (to_pair_desc) that are never stored: a thread takes 4
// consecutive entries of both results at a time, sums their products with the small operands in
// registers and multiplies.  X0's entries serve all the variables only Y0 has.  Bound by the HBM
// bytes of X0 and X1: 4096 slices of two 2^20-entry operands in 6.9 ms (5 TB/s), where the two
// joins and the dot product took 7.4, 7.3 and 5.6.
template <typename T, bool SCALED, int SA, int SB, bool ONE>
__global__ __launch_bounds__(kBlock) void k_fold_pair(const to_pair_desc* __restrict__ descs, int ndesc, const int32_t* __restrict__ bmap) {
    constexpr int NA = 1 << SA, NB = 1 << SB;
    typedef T V4 __attribute__((ext_vector_type(4)));
    __shared__ double red[kBlock];
    const to_pair_desc* d = descs + find_desc(descs, ndesc, blockIdx.x, bmap);
    const int local = blockIdx.x - d->block0;
    const int tid = threadIdx.x;
    const int bit = (tid & 63) < TO_FOLD_BITS ? tid & 63 : TO_FOLD_BITS - 1;
    const uint32_t rxa = d->bx[0][bit], rya = d->by[0][bit], rxb = d->bx[1][bit], ryb = d->by[1][bit];
    auto entry = [](uint32_t row, int b) { return (uint32_t)__builtin_amdgcn_readlane((int)row, b); };
    const int nloop = d->nloop, lsplit = d->lsplit, nreg = d->nreg;
    const int rb = 10 + nloop + lsplit, ka = rb + nreg, kb = ka + SA;
    uint32_t kxa[NA], kya[NA], kxb[NB], kyb[NB];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        kxa[i] = fold_dep(i, rxa, ka, SA);
        kya[i] = fold_dep(i, rya, ka, SA);
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        kxb[j] = fold_dep(j, rxb, kb, SB);
        kyb[j] = fold_dep(j, ryb, kb, SB);
    }
    const uint32_t ya1 = entry(rya, 0), ya2 = entry(rya, 1), yb1 = entry(ryb, 0), yb2 = entry(ryb, 1);
    auto load_x = [](const TO_GLOBAL T* p) { return *reinterpret_cast<const TO_GLOBAL V4*>(p); };
    // (the number of loads is the launch's, not the descriptor's: a branch around each would make
    // it wait for the one before, 12.8 instead of 6.9 ms below)
    constexpr int NY = ONE ? 1 : 4;
    auto load_y = [](T* y, const TO_GLOBAL T* p, uint32_t y1, uint32_t y2) {
        y[0] = p[0];
        if (!ONE) {
            y[1] = p[y1];
            y[2] = p[y2];
            y[3] = p[y1 | y2];
        }
    };
    const int64_t n = (int64_t)d->nbatch << lsplit;
    const int64_t t0 = n * local / d->nblocks, t1 = n * (local + 1) / d->nblocks;
    for (int64_t t = t0; t < t1; ++t) {
        const uint32_t sp = (uint32_t)t & ((1u << lsplit) - 1);
        const int64_t batch = t >> lsplit;
        auto start = [&](uint64_t p, int64_t stride, uint32_t row) {
            return gptr<const T>(p) + batch * stride + (fold_dep(tid, row, 2, 8) | fold_dep(sp, row, 10 + nloop, lsplit));
        };
        const TO_GLOBAL T* Xa = start(d->x[0], d->xb[0], rxa);
        const TO_GLOBAL T* Ya = start(d->y[0], d->yb[0], rya);
        const TO_GLOBAL T* Xb = start(d->x[1], d->xb[1], rxb);
        const TO_GLOBAL T* Yb = start(d->y[1], d->yb[1], ryb);
        double part[4] = {0.0, 0.0, 0.0, 0.0};
        // two nested Gray walks; the inner one goes on from the offsets it last ended with (an
        // exclusive or with a constant: still every value once)
        uint32_t xa = 0, ya = 0, xb = 0, yb = 0;
        for (uint32_t k = 1;; ++k) {
            V4 xv[NA];
#pragma unroll
            for (int i = 0; i < NA; ++i) xv[i] = load_x(Xa + (xa | kxa[i]));
            for (uint32_t r = 1;; ++r) {
                V4 xw[NB];
                T yv[NA][NY], yw[NB][NY];
#pragma unroll
                for (int j = 0; j < NB; ++j) xw[j] = load_x(Xb + (xb | kxb[j]));
#pragma unroll
                for (int j = 0; j < NB; ++j) load_y(yw[j], Yb + (yb | kyb[j]), yb1, yb2);
#pragma unroll
                for (int i = 0; i < NA; ++i) load_y(yv[i], Ya + (ya | kya[i]), ya1, ya2);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    double a = 0.0, b = 0.0;
#pragma unroll
                    for (int i = 0; i < NA; ++i) a = fma((double)xv[i][v], (double)yv[i][v % NY], a);
#pragma unroll
                    for (int j = 0; j < NB; ++j) b = fma((double)xw[j][v], (double)yw[j][v % NY], b);
                    part[v] = fma(a, b, part[v]);
                }
                if (r == 1u << nreg) break;
                const int f = rb + __builtin_ctz(r);
                ya ^= entry(rya, f);
                xb ^= entry(rxb, f);
                yb ^= entry(ryb, f);
            }
            if (k == 1u << nloop) break;
            const int f = 10 + __builtin_ctz(k);
            xa ^= entry(rxa, f);
            ya ^= entry(rya, f);
            xb ^= entry(rxb, f);
            yb ^= entry(ryb, f);
        }
        const double sum = fold_reduce((part[0] + part[1]) + (part[2] + part[3]), 0, 8, red);
        if (tid == 0) {
            FoldScale s{1.0, 0};
            if (SCALED) {
                int64_t e[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const OpScale x = op_scale(d->xs[k], d->xsb[k], batch);
                    s.f *= (double)x.f;
                    e[k] = x.e;
                    if (d->ys[k]) {
                        const OpScale y = op_scale(d->ys[k], d->ysb[k], batch);
                        s.f *= (double)y.f;
                        e[k] += y.e;
                    }
                    if (lsplit > 0 && sp == 0 && d->rs[k]) note_exp(d->rs[k], batch, e[k]);
                }
                s.e = e[0] + e[1];
            }
            if (lsplit > 0) {
                gptr<double>(d->partial)[(uint64_t)batch << lsplit | sp] = SCALED ? sum * s.f : sum;
            } else {
                const T v = (T)norm_sum<SCALED>(SCALED ? sum * s.f : sum, s.e);
                gptr<T>(d->c)[batch * d->cb] = v;
                if (SCALED) {
                    note_max(d->cs, batch, (float)absval(v));
                    note_exp(d->cs, batch, s.e);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------------
// Programs of small joins, one block per batch item (to_tree_desc): the intermediate tensors
// stay in LDS and the levels meet at block barriers, where a launch per level costs 3-5 us.
// Bound by the latency of a level: a wave issues one instruction per 4-5 cycles, so what counts
// is how few a join takes.  Its whole description, the offset of every lane included, is
// fetched while the wave works on the join before it, and the joins that need no more than one
// round of four products per lane (nearly all) run straight through: 0.7 us per level in
// float64, 1.1 us scaled (a chain of 64 joins; 1.2 and 1.6 us at 2^10 outputs), against 3-5 us
// for a launch; a product of 3 or 4 tensors, scaled by its own maximum, 0.07 us more (2 x 2
// matrices in a chain: 1.35 -> 1.43 us a level).  The n = 90 vertex cover's 224 joins are 10 levels of one block, 32 us where
// their launches took 450.  Tried: deposits computed per join instead of fetched lane offsets
// (twice the time of a level), one generic-pointer loop for every sum (long sums 1.6x), the
// maximum by LDS atomics of all lanes (+2 us per level of 64 outputs).

constexpr int kTreeMaxLds = 128 * 1024;

struct TreeRec {
    int32_t exp;
    uint32_t maxbits;
};

struct TreeWords {
    uint32_t head, bits, off[5];  // words 0-63, 64-127, and this lane's offsets (result: 4)
};

__device__ __forceinline__ TreeWords tree_words(const TO_GLOBAL uint32_t* ops, uint32_t task) {
    const TO_GLOBAL uint32_t* p = ops + (task & 0xffff) * TO_TREE_WORDS;
    return TreeWords{p[0], p[64], {p[128], p[192], p[256], p[320], p[384]}};
}

// power of two that brings a tensor of this maximum to at most 1 (any nearby one would do)
__device__ __forceinline__ int tree_exp(uint32_t maxbits) {
    return maxbits ? (int)(maxbits >> 23) - 126 : 0;
}

template <typename T, bool SCALED>
__global__ __launch_bounds__(1024) void k_fold_tree(const to_tree_desc* __restrict__ descs, int ndesc,
                                                    const int32_t* __restrict__ bmap) {
    extern __shared__ __align__(16) unsigned char smem[];
    const to_tree_desc* d = descs + find_desc(descs, ndesc, blockIdx.x, bmap);
    const int64_t batch = blockIdx.x - d->block0;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ntask = d->ntask, nslots = d->nslots;
    TreeRec* recs = reinterpret_cast<TreeRec*>(smem);
    T* data = reinterpret_cast<T*>(smem + ((nslots * sizeof(TreeRec) + 15) & ~(size_t)15));
    const TO_GLOBAL uint32_t* tasks = gptr<const uint32_t>(d->tasks) + (int64_t)wave * ntask;
    const TO_GLOBAL uint32_t* ops = gptr<const uint32_t>(d->ops) + lane;
    const uint64_t grecs = d->recs;
    uint32_t task = tasks[0];
    TreeWords w = tree_words(ops, task);
    if (SCALED) {
        for (int i = threadIdx.x; i < nslots; i += blockDim.x) recs[i] = TreeRec{0, 0u};
        __syncthreads();
    }
    for (int i = 0; i < ntask; ++i) {
        const uint32_t next = tasks[i + 1 < ntask ? i + 1 : i];
        const TreeWords wn = tree_words(ops, next);
        if (!(task & TO_TREE_IDLE)) {
            auto word = [&](int j) { return (uint32_t)__builtin_amdgcn_readlane((int)w.head, j); };
            auto wide = [&](int j) { return (uint64_t)word(j) | (uint64_t)word(j + 1) << 32; };
            const uint32_t h = word(0);
            const int lo = h & 15, lk = (h >> 4) & 15, nloop = (h >> 8) & 15, nchunk = (h >> 12) & 15;
            const int nops = ((h >> 16) & 3) + 1;
            const bool active = lane < (1 << (lo + lk)), writer = lane < (1 << lo);
            const bool cl = (h >> 24) & 1;
            const uint32_t slot = word(20);
            const int kb = 6 + nchunk;
            double f = 1.0;
            int64_t e = 0;
            if (SCALED) {
                int x = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (j < nops) {
                        const uint32_t s = word(16 + j);
                        if ((h >> (20 + j)) & 1) {
                            const TreeRec r = recs[s];
                            x += tree_exp(r.maxbits);
                            e += r.exp;
                        } else {
                            const TO_GLOBAL to_scale_rec* r =
                                gptr<const to_scale_rec>(grecs) + ((int64_t)s + (((h >> (25 + j)) & 1) ? batch : 0));
                            x += tree_exp(r->maxbits);
                            e += r->exp;
                        }
                    }
                }
                if (nops <= 2) {
                    e += x;
                    f = __longlong_as_double((long long)(1023 - x) << 52);
                }
            }
            // entry b of operand j's bits (the result: j = 4)
            auto entry = [&](int j, int b) {
                return (uint32_t)__builtin_amdgcn_readlane(j < 4 ? (int)w.bits : (int)w.head, (j < 4 ? 16 * j : 32) + b);
            };
            const uint32_t first = (task >> 16) & 127;
            const int lstep = (task >> 23) & 15;
            float mrun = 0.0f;
            auto finish = [&](double acc, uint32_t co) {
                for (int b = lo; b < lo + lk; ++b) acc += __shfl_xor(acc, 1 << b, 64);
                if (SCALED && nops > 2) {
                    // A product of 3 or 4 tensors may lie far below the product of their maxima, so
                    // it is scaled by its own largest entry (to [0.5, 1); all entries are in this
                    // wave, and double holds any product of four floats), whose high word gives
                    // an upper bound for the record.  One reduction, as the others need after
                    // their store.
                    const uint32_t top = fold_wave_umax((uint32_t)((unsigned long long)__double_as_longlong(acc) >> 32) & 0x7fffffffu);
                    const int x = top >= 0x00100000u && top < 0x7ff00000u ? (int)(top >> 20) - 1022 : 0;
                    f = __longlong_as_double((long long)(1023 - x) << 52);
                    e += x;
                    mrun = top ? (float)(__longlong_as_double((long long)((unsigned long long)top << 32 | 0xffffffffu)) * f) : 0.0f;
                }
                const T v = (T)(SCALED ? acc * f : acc);
                if (writer) {
                    if (cl) data[word(9) + co] = v;
                    else gptr<T>(wide(9))[batch * (int64_t)word(15) + co] = v;
                    if (SCALED && nops <= 2) mrun = fmaxf(mrun, (float)absval(v));
                }
            };
            if (nchunk == 0 && nloop <= 2) {
                // one round: up to 4 operands through generic pointers (LDS or global), the up
                // to 4 shared indices at once
                T v[4][4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (j < nops) {
                        const T* q = (((h >> (20 + j)) & 1)
                                          ? data + word(1 + 2 * j)
                                          : reinterpret_cast<const T*>(wide(1 + 2 * j)) + batch * (int64_t)word(11 + j)) +
                                     w.off[j];
                        const uint32_t b0 = entry(j, 6), b1 = entry(j, 7);
                        if (active) {
                            v[j][0] = q[0];
                            if (nloop >= 1) v[j][1] = q[b0];
                            if (nloop >= 2) {
                                v[j][2] = q[b1];
                                v[j][3] = q[b0 | b1];
                            }
                        }
                    }
                }
                double acc = 0.0;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (u < (1 << nloop)) {
                        double t = (double)v[0][u];
#pragma unroll
                        for (int j = 1; j < 4; ++j)
                            if (j < nops) t *= (double)v[j][u];
                        acc += t;
                    }
                }
                finish(active ? acc : 0.0, w.off[4]);
            } else {
                // The task's chunks, each a walk of the shared range four indices at a time.  Both
                // go in Gray order, so a step changes one bit of the offsets (entries do not
                // overlap: xor).
                uint32_t xo = w.off[0], yo = w.off[1], co = w.off[4];
                for (int b = 0; b < lstep; ++b)
                    if ((first >> b) & 1) {
                        xo |= entry(0, 6 + b);
                        yo |= entry(1, 6 + b);
                        co |= entry(4, 6 + b);
                    }
                const uint32_t chunks = 1u << (nchunk - lstep);
                auto run = [&](auto X, auto Y) {
                    for (uint32_t c = 1;; ++c) {
                        double acc = 0.0;
                        auto walk = [&](auto ku) {
                            constexpr int KU = decltype(ku)::value;
                            fold_walk<KU>(xo, yo, FoldRows{w.bits, w.bits, 0u}, kb, 16, nloop,
                                          [&](const uint32_t* ox, const uint32_t* oy) {
                                if (active) {
                                    T xv[KU], yv[KU];
#pragma unroll
                                    for (int j = 0; j < KU; ++j) {
                                        xv[j] = X[ox[j]];
                                        yv[j] = Y[oy[j]];
                                    }
#pragma unroll
                                    for (int j = 0; j < KU; ++j) acc = fma((double)xv[j], (double)yv[j], acc);
                                }
                            });
                        };
                        if (nloop >= 2) walk(std::integral_constant<int, 4>{});
                        else if (nloop == 1) walk(std::integral_constant<int, 2>{});
                        else walk(std::integral_constant<int, 1>{});
                        finish(acc, co);
                        if (c == chunks) break;
                        const int b = 6 + lstep + __builtin_ctz(c);
                        xo ^= entry(0, b);
                        yo ^= entry(1, b);
                        co ^= entry(4, b);
                    }
                };
                const T* Xl = data + word(1);
                const T* Yl = data + word(3);
                const TO_GLOBAL T* Xg = gptr<const T>(wide(1)) + batch * (int64_t)word(11);
                const TO_GLOBAL T* Yg = gptr<const T>(wide(3)) + batch * (int64_t)word(12);
                const bool xl = (h >> 20) & 1, yl = (h >> 21) & 1;
                if (xl && yl) run(Xl, Yl);
                else if (xl) run(Xl, Yg);
                else if (yl) run(Xg, Yl);
                else run(Xg, Yg);
            }
            if (SCALED) {
                const float m = nops > 2 ? mrun : fold_wave_max(mrun);
                if (cl) {
                    if (lane == 0) {
                        atomicMax(&recs[slot].maxbits, __float_as_uint(m));
                        if (first == 0) recs[slot].exp = (int32_t)e;
                    }
                } else {
                    const int64_t r = (int64_t)slot + (((h >> 29) & 1) ? batch : 0);
                    if (lane == 0) {
                        note_max(grecs, r, m);
                        if (first == 0) note_exp(grecs, r, e);
                    }
                }
            }
        }
        if (task & TO_TREE_MEET) __syncthreads();
        task = next;
        w = wn;
    }
}
