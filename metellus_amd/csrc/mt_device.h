// mt_device.h -- hand-written gfx950 (CDNA4) device library.
//
// Prepended to every kernel the fragment compiler generates, then compiled
// by hiprtc.  Generated code composes these pieces; the fused elementwise
// expressions arrive as lambdas (prologue transforms, epilogues, merges).
//
//   * mt_dims                 dims passed by value in the kernel arguments
//   * mt_ld4 / mt_st4         128-bit global loads / stores (_nt: nontemporal;
//                             mt_st4_wt: device scope, written through L2)
//   * mt_div_fast             division feeding a matmul (refined reciprocal
//                             times x, within 2 ulp; IEEE division at the edges)
//   * mt_wave_*               wave64 butterfly reductions (fixed order)
//   * mt_tile_colvec / rowvec / scalar
//                             cooperative ROWS x COLS tile fetch: global ->
//                             registers (transform applied to in-bounds
//                             elements, 0 outside), then registers -> LDS;
//                             fetch_raw + commit_xf apply the transform at
//                             commit time instead, so the global loads stay
//                             in flight across the MFMAs of the current chunk
//   * mt_tile_*_g             the same loaders with fetch_gather/commit_apply:
//                             a prologue's full-size operands are loaded with
//                             the tile, the chain is applied at commit
//   * MT_GLOBAL               global address space qualifier (pointer tables
//                             of batched kernels hold global pointers, which
//                             keeps their loads global_load, not flat_load)
//   * mt_tile_dma / mt_swz    direct-to-LDS tile loads (global_load_lds_dwordx4,
//                             no registers, no LDS stores) into dense tiles
//                             whose 16-byte slots are XOR-swizzled per row
//   * mt_mfma_tile            one LDS k-chunk for a wave's WM x WN grid of 32x32
//                             blocks: fp32 operands split into three bf16 parts
//                             in registers (mt_split), six bf16 MFMAs per step
//   * mt_own / mt_cut         what of the operands' low bits the split cut off,
//                             noticed by each wave or by some for the others
//   * mt_mfma_retry / mt_mfma_exact
//                             the fp32 MFMAs a wave falls back to when its
//                             results are not finite or too small for the
//                             split, or the bits cut off could matter
//   * mt_mfma_tile_f32        the same chunk on fp32 MFMAs (hand-composed kernels)
//   * mt_rw_*                 row-owning waves for matmuls 128 columns wide
//                             (split MFMAs, A in registers, B's parts in LDS)
//   * mt_sn_*                 skinny matmuls (few rows): operands straight from
//                             global memory into fp32 MFMAs, k split over waves
//                             and workgroups
//   * mt_acc_row              row of accumulator register v in a 32x32 block
//   * mt_stream_k / mt_sk_*   stream-K schedule of a persistent matmul and the
//                             workspace flags that hand split tiles' partial
//                             sums to the workgroup finishing them
//   * mt_wave_row_reduce / mt_rr_*
//                             row reductions of a matmul's output tile in its
//                             epilogue (lane exchanges, then per-tile values
//                             combined by the last workgroup of a row block)
//
// All indices are unsigned 32-bit except global offsets (size_t).

typedef float mt_f32x4 __attribute__((ext_vector_type(4)));
typedef float mt_f32x2 __attribute__((ext_vector_type(2)));
typedef float mt_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned mt_u32x4 __attribute__((ext_vector_type(4)));

struct mt_dims {
    unsigned int v[16];
};

#define MT_INLINE __device__ __forceinline__
#define MT_GLOBAL __attribute__((address_space(1)))

#ifndef INFINITY
#define INFINITY __builtin_inff()
#endif
#ifndef NAN
#define NAN __builtin_nanf("")
#endif

MT_INLINE mt_f32x4 mt_ld4(const float* p) { return *reinterpret_cast<const mt_f32x4*>(p); }
// 128-bit load from any element address: the hardware asks for 4-byte
// alignment only (every extra cache line touched costs a cycle or so).
typedef float mt_f32x4u __attribute__((ext_vector_type(4), aligned(4)));
MT_INLINE mt_f32x4 mt_ld4u(const float* p) { return *reinterpret_cast<const mt_f32x4u*>(p); }
MT_INLINE mt_f32x4 mt_ld4u_nt(const float* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const mt_f32x4u*>(p));
}
MT_INLINE void mt_st4(float* p, mt_f32x4 v) { *reinterpret_cast<mt_f32x4*>(p) = v; }
// Streaming variants: nontemporal hint (data used once; do not keep in cache).
MT_INLINE mt_f32x4 mt_ld4_nt(const float* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const mt_f32x4*>(p));
}
MT_INLINE void mt_st4_nt(float* p, mt_f32x4 v) { __builtin_nontemporal_store(v, reinterpret_cast<mt_f32x4*>(p)); }
// 128-bit global store at device scope (sc1): it writes through the XCD's L2
// instead of leaving a dirty line there, which suits outputs written once by
// streaming kernels.  p must point to global memory (never LDS).  A 128-bit
// store reads its data registers after it issues; the compiler cannot see
// this store, so it is followed by two wait states (see mt_buffer_store4).
MT_INLINE void mt_st4_wt(float* p, mt_f32x4 v) {
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(p), "v"(v) : "memory");
}

// x / y where the quotient enters a matmul.  r is the hardware reciprocal
// refined by one Newton step, r + r * (1 - y * r); it depends on y only, so
// the compiler computes it once per distinct divisor (a row or column
// broadcast operand gives one per loaded vector), and each element costs:
//   * 1 <= |y| < 2^125: the product x * r -- within 2 ulp of the IEEE
//     quotient; |x * r| <= |x|, so nothing overflows, and zero, infinite
//     and NaN numerators give what the division gives;
//   * 2^-125 < |y| < 1: the product plus one residual (Markstein) correction
//     q + r * (x - q * y) -- within 1 ulp;
//   * anything else (zero, subnormal, huge or non-finite divisors, quotients
//     of 2^125 and beyond on the second path): the IEEE division.
// Measured on the C5 P.V kernel (one division per A element): 296 us with
// the correction on every element, 276 us with the product alone.
// The two pieces that depend on y alone: the refined reciprocal, and whether
// x * r is the whole quotient (mt_div_plain).  A loader whose divisors are
// all plain computes x * mt_div_rcp(y) directly (commit_apply_fast).
MT_INLINE float mt_div_rcp(float y) {
    const float r = __builtin_amdgcn_rcpf(y);
    return __builtin_fmaf(__builtin_fmaf(-y, r, 1.0f), r, r);
}
MT_INLINE bool mt_div_plain(float y) {
    const float ay = __builtin_fabsf(y);
    return ay >= 1.0f && ay < 0x1.0p+125f;
}
MT_INLINE float mt_div_fast(float x, float y) {
    const float ay = __builtin_fabsf(y);
    const float r = mt_div_rcp(y);
    const float q = x * r;
    if (__builtin_expect(mt_div_plain(y), 1)) return q;
    const float v = __builtin_fmaf(__builtin_fmaf(-q, y, x), r, q);
    const bool ok = ay > 0x1.0p-125f && ay < 1.0f && __builtin_fabsf(v) < 0x1.0p+125f;
    // The IEEE division stays on its (rarely taken) branch: the empty asm
    // statement emits nothing but cannot be speculated, so the compiler does
    // not compute the division for every lane and select.
    if (__builtin_expect(!ok, 0)) {
        float xs = x;
        asm volatile("" : "+v"(xs));
        return xs / y;
    }
    return v;
}

MT_INLINE unsigned mt_lane() { return threadIdx.x & 63u; }
// Wave index as a scalar (wave-uniform) value.
MT_INLINE unsigned mt_wave() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// ---------------------------------------------------------------------------
// wave64 reductions.  Butterfly over xor offsets 32, 16, 8, 4, 2, 1: after
// step `off`, lane l holds v_l (op) v_{l^off}.  Every lane ends with the same
// value; the pairing tree is fixed, so results are reproducible (and the CPU
// oracle replays the same tree).
// ---------------------------------------------------------------------------

MT_INLINE float mt_shfl_xor(float v, int off) { return __shfl_xor(v, off, 64); }

MT_INLINE float mt_wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = v + mt_shfl_xor(v, off);
    return v;
}
MT_INLINE float mt_wave_product(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = v * mt_shfl_xor(v, off);
    return v;
}
MT_INLINE float mt_wave_max(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, mt_shfl_xor(v, off));
    return v;
}
MT_INLINE float mt_wave_min(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fminf(v, mt_shfl_xor(v, off));
    return v;
}

// ---------------------------------------------------------------------------
// Cooperative tile loaders.  A loader owns the registers for its share of one
// ROWS x COLS tile (NT lanes).  fetch<CHECK>() issues the global loads for the
// tile at (row0, col0) of a strided matrix (element (r, c) at
// src[r*rs + c*cs]); F(raw, row, col) transforms each in-bounds element
// (elementwise prologue); elements outside (rlim, clim) are 0 (identity of
// the matmul / sum consumer).  commit<LD>() writes the registers into an LDS
// tile with row pitch LD floats.  Splitting the two lets the mainloop keep
// the next tile's loads in flight while the MFMAs run.
// ---------------------------------------------------------------------------

struct mt_identity {
    MT_INLINE float operator()(float v, unsigned, unsigned) const { return v; }
};

// Partial fetches.  Every fetch takes an optional (q, Q): it then issues only
// the loads of part q of Q, slot i of n belonging to part (i * Q) / n, so Q
// calls with q = 0 .. Q-1 issue every load exactly once (the default 0, 1 is
// the whole tile).  The mainloop spreads a chunk's loads over the MFMA
// sequence this way instead of issuing them in one burst: a burst of vector
// memory instructions holds each wave in load issue while the address units
// work through it, and its MFMAs wait behind them.
__host__ __device__ __forceinline__ constexpr bool mt_in_part(int i, int n, int q, int Q) {
    return Q <= 1 || (i * Q) / n == q;
}

// Four consecutive elements from p, of which the first `left` (at least one)
// are inside the matrix: one 128-bit load at any element address, or element by
// element at its edge (0 outside).
template <bool NT = false>
MT_INLINE mt_f32x4 mt_ld_slot(const float* p, unsigned left) {
    if (left >= 4u) return NT ? mt_ld4u_nt(p) : mt_ld4u(p);
    mt_f32x4 x = {p[0], 0.f, 0.f, 0.f};
    if (left > 1u) x.y = p[1];
    if (left > 2u) x.z = p[2];
    return x;
}
// The first `left` of four consecutive elements to p (any element address).  WT:
// the single ones at device scope too, as the next row's begin in the same line: kept
// in the L2 of one XCD while another writes the rest through, such a line cost an
// 8000 x 2001 transpose 51 us instead of 38.
template <bool WT = false>
MT_INLINE void mt_st_slot(float* p, mt_f32x4 v, unsigned left) {
    if (left >= 4u) {
        if (WT)
            mt_st4_wt(p, v);
        else
            *reinterpret_cast<mt_f32x4u*>(p) = v;
        return;
    }
    if constexpr (WT) {
        __hip_atomic_store(p, v.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (left > 1u) __hip_atomic_store(p + 1, v.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (left > 2u) __hip_atomic_store(p + 2, v.z, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    p[0] = v.x;
    if (left > 1u) p[1] = v.y;
    if (left > 2u) p[2] = v.z;
}
// The slot's elements outside the matrix are 0 again after a transform.
MT_INLINE void mt_clear_slot(mt_f32x4& x, unsigned left) {
    if (left < 2u) x.y = 0.f;
    if (left < 3u) x.z = 0.f;
    if (left < 4u) x.w = 0.f;
}

// Vectorised along columns: cs == 1, COLS % 4 == 0, any row stride and (CHECK)
// limits.
template <int ROWS, int COLS, int NT>
struct mt_tile_colvec {
    static constexpr int CV = COLS / 4;
    static constexpr int TOTAL = ROWS * CV;
    static constexpr int PER = (TOTAL + NT - 1) / NT;
    mt_f32x4 v[PER];

    template <bool CHECK, typename F>
    MT_INLINE void fetch(const float* __restrict__ src, unsigned rs, unsigned row0, unsigned col0,
                         unsigned rlim, unsigned clim, unsigned tid, F f, int q = 0, int Q = 1) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (!mt_in_part(i, PER, q, Q)) continue;
            const unsigned idx = tid + i * NT;
            const unsigned r = idx / CV, c = (idx % CV) * 4u;
            const unsigned gr = row0 + r, gc = col0 + c;
            mt_f32x4 x = {0.f, 0.f, 0.f, 0.f};
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < rlim && gc < clim))) {
                const unsigned left = CHECK ? clim - gc : 4u;
                x = mt_ld_slot(src + (size_t)gr * rs + gc, left);
                x.x = f(x.x, gr, gc);
                if (left > 1u) x.y = f(x.y, gr, gc + 1u);
                if (left > 2u) x.z = f(x.z, gr, gc + 2u);
                if (left > 3u) x.w = f(x.w, gr, gc + 3u);
            }
            v[i] = x;
        }
    }

    // Any row stride, limits and base alignment: a slot is one 128-bit load
    // (at any element address) when its 4 columns are in bounds, otherwise
    // element by element (out-of-bounds elements are 0, and f is applied to
    // in-bounds elements only).  Same register layout as fetch().
    template <typename F>
    MT_INLINE void fetch_safe(const float* __restrict__ src, unsigned rs, unsigned row0, unsigned col0,
                              unsigned rlim, unsigned clim, unsigned tid, F f, int q = 0, int Q = 1) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (!mt_in_part(i, PER, q, Q)) continue;
            const unsigned idx = tid + i * NT;
            const unsigned r = idx / CV, c = (idx % CV) * 4u;
            const unsigned gr = row0 + r, gc = col0 + c;
            mt_f32x4 x = {0.f, 0.f, 0.f, 0.f};
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && gr < rlim && gc < clim) {
                const float* p = src + (size_t)gr * rs + gc;
                if (gc + 3u < clim) {
                    x = mt_ld4u(p);
                    x.x = f(x.x, gr, gc);
                    x.y = f(x.y, gr, gc + 1u);
                    x.z = f(x.z, gr, gc + 2u);
                    x.w = f(x.w, gr, gc + 3u);
                } else {
                    x.x = f(p[0], gr, gc);
                    if (gc + 1u < clim) x.y = f(p[1], gr, gc + 1u);
                    if (gc + 2u < clim) x.z = f(p[2], gr, gc + 2u);
                    if (gc + 3u < clim) x.w = f(p[3], gr, gc + 3u);
                }
            }
            v[i] = x;
        }
    }

    // 128-bit LDS stores when the row pitch keeps them 16-byte aligned.
    template <int LD>
    MT_INLINE void commit(float* lds, unsigned tid) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const unsigned idx = tid + i * NT;
            if (TOTAL % NT == 0 || idx < (unsigned)TOTAL) {
                const unsigned r = idx / CV, c = (idx % CV) * 4u;
                if constexpr (LD % 4 == 0) {
                    mt_st4(lds + r * LD + c, v[i]);
                } else {
                    float* d = lds + r * LD + c;
                    d[0] = v[i].x, d[1] = v[i].y, d[2] = v[i].z, d[3] = v[i].w;
                }
            }
        }
    }

    // Deferred transform: fetch_raw keeps the loaded values untouched (0
    // outside the bounds) and remembers the tile origin; commit_xf applies f
    // to the in-bounds elements on the way to LDS.
    unsigned r0, c0, rl, cl;

    template <bool CHECK>
    MT_INLINE void fetch_raw(const float* __restrict__ src, unsigned rs, unsigned row0, unsigned col0,
                             unsigned rlim, unsigned clim, unsigned tid, int q = 0, int Q = 1) {
        r0 = row0, c0 = col0, rl = rlim, cl = clim;
        fetch<CHECK>(src, rs, row0, col0, rlim, clim, tid, mt_identity{}, q, Q);
    }

    template <int LD, bool CHECK, typename F>
    MT_INLINE void commit_xf(float* lds, unsigned tid, F f) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const unsigned idx = tid + i * NT;
            const unsigned r = idx / CV, c = (idx % CV) * 4u;
            const unsigned gr = r0 + r, gc = c0 + c;
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < rl && gc < cl))) {
                const unsigned left = CHECK ? cl - gc : 4u;
                v[i].x = f(v[i].x, gr, gc);
                if (left > 1u) v[i].y = f(v[i].y, gr, gc + 1u);
                if (left > 2u) v[i].z = f(v[i].z, gr, gc + 2u);
                if (left > 3u) v[i].w = f(v[i].w, gr, gc + 3u);
            }
        }
        commit<LD>(lds, tid);
    }
};

// Vectorised along rows: rs == 1, ROWS % 4 == 0, any column stride and (CHECK)
// limits.
template <int ROWS, int COLS, int NT>
struct mt_tile_rowvec {
    static constexpr int RV = ROWS / 4;
    static constexpr int TOTAL = RV * COLS;
    static constexpr int PER = (TOTAL + NT - 1) / NT;
    // Tall tiles (an A operand) give each lane KB neighbouring columns of its
    // four rows, which leave as one store per row; eight lanes read a 128-byte
    // line and the next eight the next KB columns.  Single stores met in a bank
    // eight at a time: 1024 x 2048 x 4096 with X^T 182 -> 152 us on MI355X.
    static constexpr int KB = RV % 8 != 0 || ROWS <= COLS || TOTAL % NT != 0 ? 1
                              : PER % 4 == 0 && COLS % 4 == 0                ? 4
                              : PER % 2 == 0 && COLS % 2 == 0                ? 2
                                                                             : 1;
    mt_f32x4 v[PER];

    // The tile's column (in c) and first row of slot i.
    static MT_INLINE unsigned slot(unsigned tid, int i, unsigned& c) {
        if constexpr (KB == 1) {
            const unsigned idx = tid + i * NT;
            c = idx / RV;
            return (idx % RV) * 4u;
        } else {
            constexpr unsigned KQ = COLS / KB;
            const unsigned b = tid + (i / KB) * NT;
            c = (b / 8u) % KQ * KB + (unsigned)(i % KB);
            return (b / (8u * KQ) * 8u + b % 8u) * 4u;
        }
    }

    template <bool CHECK, typename F>
    MT_INLINE void fetch(const float* __restrict__ src, unsigned cs, unsigned row0, unsigned col0,
                         unsigned rlim, unsigned clim, unsigned tid, F f, int q = 0, int Q = 1) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (!mt_in_part(i, PER, q, Q)) continue;
            const unsigned idx = tid + i * NT;
            unsigned c;
            const unsigned r = slot(tid, i, c);
            const unsigned gr = row0 + r, gc = col0 + c;
            mt_f32x4 x = {0.f, 0.f, 0.f, 0.f};
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < rlim && gc < clim))) {
                const unsigned left = CHECK ? rlim - gr : 4u;
                x = mt_ld_slot(src + gr + (size_t)gc * cs, left);
                x.x = f(x.x, gr, gc);
                if (left > 1u) x.y = f(x.y, gr + 1u, gc);
                if (left > 2u) x.z = f(x.z, gr + 2u, gc);
                if (left > 3u) x.w = f(x.w, gr + 3u, gc);
            }
            v[i] = x;
        }
    }

    template <int LD>
    MT_INLINE void commit(float* lds, unsigned tid) const {
        if constexpr (KB > 1 && LD % KB == 0) {
#pragma unroll
            for (int i = 0; i < PER; i += KB) {
                unsigned c;
                float* at = lds + slot(tid, i, c) * LD;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if constexpr (KB == 4) {
                        *reinterpret_cast<mt_f32x4*>(at + j * LD + c) =
                            mt_f32x4{v[i][j], v[i + 1][j], v[i + 2][j], v[i + 3][j]};
                    } else {
                        *reinterpret_cast<mt_f32x2*>(at + j * LD + c) = mt_f32x2{v[i][j], v[i + 1][j]};
                    }
                }
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const unsigned idx = tid + i * NT;
            if (TOTAL % NT == 0 || idx < (unsigned)TOTAL) {
                unsigned c;
                const unsigned r = slot(tid, i, c);
                lds[(r + 0u) * LD + c] = v[i].x;
                lds[(r + 1u) * LD + c] = v[i].y;
                lds[(r + 2u) * LD + c] = v[i].z;
                lds[(r + 3u) * LD + c] = v[i].w;
            }
        }
    }

    unsigned r0, c0, rl, cl;

    template <bool CHECK>
    MT_INLINE void fetch_raw(const float* __restrict__ src, unsigned cs, unsigned row0, unsigned col0,
                             unsigned rlim, unsigned clim, unsigned tid, int q = 0, int Q = 1) {
        r0 = row0, c0 = col0, rl = rlim, cl = clim;
        fetch<CHECK>(src, cs, row0, col0, rlim, clim, tid, mt_identity{}, q, Q);
    }

    template <int LD, bool CHECK, typename F>
    MT_INLINE void commit_xf(float* lds, unsigned tid, F f) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const unsigned idx = tid + i * NT;
            unsigned c;
            const unsigned r = slot(tid, i, c);
            const unsigned gr = r0 + r, gc = c0 + c;
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < rl && gc < cl))) {
                const unsigned left = CHECK ? rl - gr : 4u;
                v[i].x = f(v[i].x, gr, gc);
                if (left > 1u) v[i].y = f(v[i].y, gr + 1u, gc);
                if (left > 2u) v[i].z = f(v[i].z, gr + 2u, gc);
                if (left > 3u) v[i].w = f(v[i].w, gr + 3u, gc);
            }
        }
        commit<LD>(lds, tid);
    }
};

// Any strides: one element per load.
template <int ROWS, int COLS, int NT>
struct mt_tile_scalar {
    static constexpr int TOTAL = ROWS * COLS;
    static constexpr int PER = (TOTAL + NT - 1) / NT;
    float v[PER];

    template <bool CHECK, typename F>
    MT_INLINE void fetch(const float* __restrict__ src, unsigned rs, unsigned cs, unsigned row0,
                         unsigned col0, unsigned rlim, unsigned clim, unsigned tid, F f, int q = 0, int Q = 1) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (!mt_in_part(i, PER, q, Q)) continue;
            const unsigned idx = tid + i * NT;
            const unsigned r = idx / COLS, c = idx % COLS;
            const unsigned gr = row0 + r, gc = col0 + c;
            float x = 0.f;
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < rlim && gc < clim))) {
                x = f(src[(size_t)gr * rs + (size_t)gc * cs], gr, gc);
            }
            v[i] = x;
        }
    }

    template <int LD>
    MT_INLINE void commit(float* lds, unsigned tid) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const unsigned idx = tid + i * NT;
            if (TOTAL % NT == 0 || idx < (unsigned)TOTAL) {
                const unsigned r = idx / COLS, c = idx % COLS;
                lds[r * LD + c] = v[i];
            }
        }
    }

    unsigned r0, c0, rl, cl;

    template <bool CHECK>
    MT_INLINE void fetch_raw(const float* __restrict__ src, unsigned rs, unsigned cs, unsigned row0,
                             unsigned col0, unsigned rlim, unsigned clim, unsigned tid, int q = 0, int Q = 1) {
        r0 = row0, c0 = col0, rl = rlim, cl = clim;
        fetch<CHECK>(src, rs, cs, row0, col0, rlim, clim, tid, mt_identity{}, q, Q);
    }

    template <int LD, bool CHECK, typename F>
    MT_INLINE void commit_xf(float* lds, unsigned tid, F f) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const unsigned idx = tid + i * NT;
            const unsigned r = idx / COLS, c = idx % COLS;
            const unsigned gr = r0 + r, gc = c0 + c;
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < rl && gc < cl))) {
                v[i] = f(v[i], gr, gc);
            }
        }
        commit<LD>(lds, tid);
    }
};

// ---------------------------------------------------------------------------
// Gather / apply loaders: a prologue that reads E full-size operands loads
// them together with the tile (fetch_gather: g(row, col) -> mt_vals<E> per
// element) and applies the chain when the tile is committed to LDS
// (commit_apply: a(raw, extras) per in-bounds element), so neither the tile
// nor its operands are waited for before the current chunk's MFMAs.  Out of
// bounds elements stay 0 and are not transformed.  SLOT = true (vectorised
// loaders): the operands are constant along the vector axis (a column
// broadcast for mt_tile_colvec_g, a row broadcast for mt_tile_rowvec_g), so
// they are gathered once per 128-bit slot and the 4 elements share them --
// one value, so work that depends only on it (a divisor's reciprocal) is
// done once per slot.
// ---------------------------------------------------------------------------

template <int E>
struct mt_vals {
    float v[E];
};

template <int ROWS, int COLS, int NT, int E, bool SLOT = false>
struct mt_tile_colvec_g : mt_tile_colvec<ROWS, COLS, NT> {
    using Base = mt_tile_colvec<ROWS, COLS, NT>;
    using Base::CV;
    using Base::PER;
    using Base::TOTAL;
    static constexpr int NG = SLOT ? 1 : 4;  // gathers per slot
    mt_vals<E> ex[PER][NG];

    template <bool CHECK, typename G>
    MT_INLINE void fetch_gather(const float* __restrict__ src, unsigned rs, unsigned row0, unsigned col0,
                                unsigned rlim, unsigned clim, unsigned tid, G g, int q = 0, int Q = 1) {
        this->r0 = row0, this->c0 = col0, this->rl = rlim, this->cl = clim;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (!mt_in_part(i, PER, q, Q)) continue;
            const unsigned idx = tid + i * NT;
            const unsigned r = idx / CV, c = (idx % CV) * 4u;
            const unsigned gr = row0 + r, gc = col0 + c;
            mt_f32x4 x = {0.f, 0.f, 0.f, 0.f};
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < rlim && gc < clim))) {
                const unsigned left = CHECK ? clim - gc : 4u;
                x = mt_ld_slot(src + (size_t)gr * rs + gc, left);
#pragma unroll
                for (int j = 0; j < NG; ++j)
                    if (j == 0 || (unsigned)j < left) ex[i][j] = g(gr, gc + (unsigned)j);
            }
            this->v[i] = x;
        }
    }

    // SLOT gathers are constant along the loaded rows' k axis, so the next
    // chunk of the same tile needs the same operands: fetch_keep loads the
    // tile alone and keeps ex (and the work derived from it, such as a
    // divisor's reciprocal, stays loop-invariant for the compiler).
    template <bool CHECK>
    MT_INLINE void fetch_keep(const float* __restrict__ src, unsigned rs, unsigned row0, unsigned col0,
                              unsigned rlim, unsigned clim, unsigned tid, int q = 0, int Q = 1) {
        static_assert(SLOT, "only per-slot gathers are invariant along k");
        this->r0 = row0, this->c0 = col0, this->rl = rlim, this->cl = clim;
        Base::template fetch<CHECK>(src, rs, row0, col0, rlim, clim, tid, mt_identity{}, q, Q);
    }

    // True in every lane when P(e) holds for the gathered operands of every
    // in-bounds slot of every lane of the wave (one wave-uniform test).
    template <bool CHECK, typename P>
    MT_INLINE bool all_plain(unsigned tid, P p) const {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const unsigned idx = tid + i * NT;
            const unsigned r = idx / CV, c = (idx % CV) * 4u;
            const unsigned gr = this->r0 + r, gc = this->c0 + c;
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < this->rl && gc < this->cl))) {
#pragma unroll
                for (int j = 0; j < NG; ++j)
                    if (j == 0 || !CHECK || (unsigned)j < this->cl - gc) ok = ok && p(ex[i][j]);
            }
        }
        return __builtin_amdgcn_ballot_w64(!ok) == 0ull;
    }

    // commit_apply with Q -- the chain with its divisions reduced to
    // x * mt_div_rcp(y), exact when P holds -- when all_plain, without a
    // branch per element; A otherwise.
    template <int LD, bool CHECK, typename A, typename Q, typename P>
    MT_INLINE void commit_apply_fast(float* lds, unsigned tid, A a, Q q, P p) {
        if (__builtin_expect(all_plain<CHECK>(tid, p), 1)) {
            commit_apply<LD, CHECK>(lds, tid, q);
        } else {
            commit_apply<LD, CHECK>(lds, tid, a);
        }
    }

    template <int LD, bool CHECK, typename A>
    MT_INLINE void commit_apply(float* lds, unsigned tid, A a) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const unsigned idx = tid + i * NT;
            const unsigned r = idx / CV, c = (idx % CV) * 4u;
            const unsigned gr = this->r0 + r, gc = this->c0 + c;
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < this->rl && gc < this->cl))) {
                this->v[i].x = a(this->v[i].x, ex[i][0]);
                this->v[i].y = a(this->v[i].y, ex[i][1 % NG]);
                this->v[i].z = a(this->v[i].z, ex[i][2 % NG]);
                this->v[i].w = a(this->v[i].w, ex[i][3 % NG]);
                if (CHECK) mt_clear_slot(this->v[i], this->cl - gc);
            }
        }
        Base::template commit<LD>(lds, tid);
    }
};

template <int ROWS, int COLS, int NT, int E, bool SLOT = false>
struct mt_tile_rowvec_g : mt_tile_rowvec<ROWS, COLS, NT> {
    using Base = mt_tile_rowvec<ROWS, COLS, NT>;
    using Base::RV;
    using Base::PER;
    using Base::TOTAL;
    static constexpr int NG = SLOT ? 1 : 4;  // gathers per slot
    mt_vals<E> ex[PER][NG];

    template <bool CHECK, typename G>
    MT_INLINE void fetch_gather(const float* __restrict__ src, unsigned cs, unsigned row0, unsigned col0,
                                unsigned rlim, unsigned clim, unsigned tid, G g, int q = 0, int Q = 1) {
        this->r0 = row0, this->c0 = col0, this->rl = rlim, this->cl = clim;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (!mt_in_part(i, PER, q, Q)) continue;
            const unsigned idx = tid + i * NT;
            unsigned c;
            const unsigned r = Base::slot(tid, i, c);
            const unsigned gr = row0 + r, gc = col0 + c;
            mt_f32x4 x = {0.f, 0.f, 0.f, 0.f};
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < rlim && gc < clim))) {
                const unsigned left = CHECK ? rlim - gr : 4u;
                x = mt_ld_slot(src + gr + (size_t)gc * cs, left);
#pragma unroll
                for (int j = 0; j < NG; ++j)
                    if (j == 0 || (unsigned)j < left) ex[i][j] = g(gr + (unsigned)j, gc);
            }
            this->v[i] = x;
        }
    }

    template <bool CHECK>
    MT_INLINE void fetch_keep(const float* __restrict__ src, unsigned cs, unsigned row0, unsigned col0,
                              unsigned rlim, unsigned clim, unsigned tid, int q = 0, int Q = 1) {
        static_assert(SLOT, "only per-slot gathers are invariant along k");
        this->r0 = row0, this->c0 = col0, this->rl = rlim, this->cl = clim;
        Base::template fetch<CHECK>(src, cs, row0, col0, rlim, clim, tid, mt_identity{}, q, Q);
    }

    // True in every lane when P(e) holds for the gathered operands of every
    // in-bounds slot of every lane of the wave (one wave-uniform test).
    template <bool CHECK, typename P>
    MT_INLINE bool all_plain(unsigned tid, P p) const {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const unsigned idx = tid + i * NT;
            unsigned c;
            const unsigned r = Base::slot(tid, i, c);
            const unsigned gr = this->r0 + r, gc = this->c0 + c;
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < this->rl && gc < this->cl))) {
#pragma unroll
                for (int j = 0; j < NG; ++j)
                    if (j == 0 || !CHECK || (unsigned)j < this->rl - gr) ok = ok && p(ex[i][j]);
            }
        }
        return __builtin_amdgcn_ballot_w64(!ok) == 0ull;
    }

    // commit_apply with Q -- the chain with its divisions reduced to
    // x * mt_div_rcp(y), exact when P holds -- when all_plain, without a
    // branch per element; A otherwise.
    template <int LD, bool CHECK, typename A, typename Q, typename P>
    MT_INLINE void commit_apply_fast(float* lds, unsigned tid, A a, Q q, P p) {
        if (__builtin_expect(all_plain<CHECK>(tid, p), 1)) {
            commit_apply<LD, CHECK>(lds, tid, q);
        } else {
            commit_apply<LD, CHECK>(lds, tid, a);
        }
    }

    template <int LD, bool CHECK, typename A>
    MT_INLINE void commit_apply(float* lds, unsigned tid, A a) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const unsigned idx = tid + i * NT;
            unsigned c;
            const unsigned r = Base::slot(tid, i, c);
            const unsigned gr = this->r0 + r, gc = this->c0 + c;
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < this->rl && gc < this->cl))) {
                this->v[i].x = a(this->v[i].x, ex[i][0]);
                this->v[i].y = a(this->v[i].y, ex[i][1 % NG]);
                this->v[i].z = a(this->v[i].z, ex[i][2 % NG]);
                this->v[i].w = a(this->v[i].w, ex[i][3 % NG]);
                if (CHECK) mt_clear_slot(this->v[i], this->rl - gr);
            }
        }
        Base::template commit<LD>(lds, tid);
    }
};

template <int ROWS, int COLS, int NT, int E>
struct mt_tile_scalar_g : mt_tile_scalar<ROWS, COLS, NT> {
    using Base = mt_tile_scalar<ROWS, COLS, NT>;
    using Base::PER;
    using Base::TOTAL;
    mt_vals<E> ex[PER];

    template <bool CHECK, typename G>
    MT_INLINE void fetch_gather(const float* __restrict__ src, unsigned rs, unsigned cs, unsigned row0,
                                unsigned col0, unsigned rlim, unsigned clim, unsigned tid, G g, int q = 0,
                                int Q = 1) {
        this->r0 = row0, this->c0 = col0, this->rl = rlim, this->cl = clim;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (!mt_in_part(i, PER, q, Q)) continue;
            const unsigned idx = tid + i * NT;
            const unsigned r = idx / COLS, c = idx % COLS;
            const unsigned gr = row0 + r, gc = col0 + c;
            float x = 0.f;
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < rlim && gc < clim))) {
                x = src[(size_t)gr * rs + (size_t)gc * cs];
                ex[i] = g(gr, gc);
            }
            this->v[i] = x;
        }
    }

    template <int LD, bool CHECK, typename A>
    MT_INLINE void commit_apply(float* lds, unsigned tid, A a) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const unsigned idx = tid + i * NT;
            const unsigned r = idx / COLS, c = idx % COLS;
            const unsigned gr = this->r0 + r, gc = this->c0 + c;
            if ((TOTAL % NT == 0 || idx < (unsigned)TOTAL) && (!CHECK || (gr < this->rl && gc < this->cl))) {
                this->v[i] = a(this->v[i], ex[i]);
            }
        }
        Base::template commit<LD>(lds, tid);
    }
};

// Integer helpers callable from host code too (the CPU tests check them).
#define MT_HD __host__ __device__ __forceinline__

// ---------------------------------------------------------------------------
// Direct-to-LDS tile loads (gfx950 global_load_lds_dwordx4).  One such load
// moves 16 bytes per lane from global memory straight into LDS at
// M0 + 16 * lane, so a wave writes 1 KiB of contiguous LDS per instruction
// and no registers or LDS-store instructions are spent on the tile.  Tiles
// are therefore dense; operand tiles the MFMAs read row-wise with 128-bit
// reads permute the 16-byte slots of each row by mt_swz (an XOR of the
// slot index), which keeps those reads free of bank conflicts.
//
// The loads are issued from inline asm: the compiler then does not see an
// LDS write it would wait for before every later LDS read (it cannot tell
// the stage being filled from the one being read).  The mainloop waits for
// them itself (s_waitcnt) before the barrier that publishes the chunk.
// ---------------------------------------------------------------------------

// Physical slot permutation of row r of a dense LDS tile with S 16-byte slots
// per row (slot p holds logical slot p ^ mt_swz<S>(r)).  It depends on
// r mod 16 only, and makes the slots read by 8 consecutive rows, and by the
// even and the odd rows among 16 consecutive ones, pairwise distinct -- a
// 128-bit read of one slot per row by consecutive lanes then meets no bank
// conflict whether the LDS serves 128 or 256 bytes per cycle.
template <int S>
MT_HD unsigned mt_swz(unsigned r) {
    static_assert(S == 4 || S == 8, "swizzle defined for 16- and 32-float rows");
    if constexpr (S == 8) return ((r >> 1) ^ ((r & 1u) << 2)) & 7u;
    return ((r >> 1) ^ (r >> 2)) & 3u;
}

MT_INLINE unsigned mt_lds_addr(const float* p) {
    return (unsigned)(unsigned long long)(const __attribute__((address_space(3))) float*)p;
}

// 16 bytes from sbase + voff to LDS byte address lds_byte + 16 * lane:
// sbase is a wave-uniform address held in scalar registers, voff this lane's
// 32-bit byte offset from it, lds_byte wave uniform.  One wait state
// separates the M0 write from the load reading it.
MT_INLINE void mt_dma16(unsigned long long sbase, unsigned voff, unsigned lds_byte) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(voff), "s"(sbase), "s"(lds_byte)
                 : "memory", "m0");
}

// A wave-uniform address as a scalar value (both halves read from the first
// lane; the compiler folds this when the address is already scalar).
MT_INLINE unsigned long long mt_uniform_addr(const float* p) {
    const unsigned long long a = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

// Where a direct-to-LDS load puts its data: lane `lane` of wave-load `inst`
// writes physical slot 64 inst + lane of a dense tile with S slots per row,
// i.e. row r, physical slot p; it loads the row's logical slot p (SWZ: p ^
// mt_swz<S>(r)), so logical slot L of row r sits at physical L ^ mt_swz<S>(r).
template <int S, bool SWZ>
MT_HD void mt_dma_slot(unsigned inst, unsigned lane, unsigned& r, unsigned& logical) {
    const unsigned slot = inst * 64u + lane;
    r = slot / S;
    logical = slot % S;
    if constexpr (SWZ) logical ^= mt_swz<S>(r);
}

// ROWS x COLS tile of a row-major source (row stride rs floats, a multiple of
// 4; 16-byte aligned base) at (row0, col0), every element in bounds, into a
// dense LDS tile; SWZ permutes each row's slots by mt_swz.  Wave w issues
// wave-loads w PERW .. w PERW + PERW - 1, each 1 KiB of contiguous LDS.
//
// The loader is built once per kernel with the source's row stride: each
// lane's byte offsets from the tile origin do not change from chunk to
// chunk, so they are computed there, and a fetch adds only the tile
// origin -- a scalar address -- through the load's scalar-base form.  The
// offsets are 32-bit: ((ROWS - 1) rs + COLS) * 4 must stay below 2^32 (the
// assembler checks).  Recomputing the full per-lane addresses in every
// chunk cost ~900 cycles of VALU work per 32-wide chunk on a 256x256 tile
// (4096^3 GEMM, measured in shader cycles per workgroup: 2.26 -> 2.19 M).
template <int ROWS, int COLS, int NT, bool SWZ>
struct mt_tile_dma {
    static constexpr int S = COLS / 4;
    static constexpr int INSTR = ROWS * S / 64;
    static constexpr int PERW = INSTR / (NT / 64);
    static_assert(COLS % 4 == 0 && (ROWS * S) % 64 == 0 && INSTR % (NT / 64) == 0,
                  "the tile must split into whole 1 KiB wave loads, the same number per wave");
    unsigned off[PERW];  // this lane's byte offset of each of the wave's loads
    unsigned lds_off;    // byte offset of the wave's first load in the tile (uniform)

    MT_INLINE mt_tile_dma(unsigned rs, unsigned tid) {
        const unsigned lane = tid & 63u;
        const unsigned wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        lds_off = wave * PERW * 1024u;
#pragma unroll
        for (int q = 0; q < PERW; ++q) {
            unsigned r, logical;
            mt_dma_slot<S, SWZ>(wave * PERW + q, lane, r, logical);
            off[q] = (r * rs + 4u * logical) * 4u;
        }
    }

    // rs: the row stride the loader was built with.
    MT_INLINE void fetch(const float* __restrict__ src, unsigned rs, unsigned row0, unsigned col0, float* lds,
                         int part = 0, int parts = 1) const {
        const unsigned long long origin = mt_uniform_addr(src + (size_t)row0 * rs + col0);
        const unsigned base = __builtin_amdgcn_readfirstlane(mt_lds_addr(lds)) + lds_off;
#pragma unroll
        for (int q = 0; q < PERW; ++q) {
            if (!mt_in_part(q, PERW, part, parts)) continue;
            mt_dma16(origin, off[q], base + (unsigned)q * 1024u);
        }
    }
};

// ---------------------------------------------------------------------------
// fp32 MFMA over one LDS k-chunk.
//
// v_mfma_f32_32x32x2f32 computes D[32x32] += A[32x2] * B[2x32]; lane l supplies
// A[l%32][l/32] and B[l/32][l%32].  The two k slots of one instruction are
// taken from the two halves of the chunk: lane half h = l/32 feeds chunk
// column k = h*TK/2 + s at step s.  Both operands use the same mapping, so
// every product A[i][k]*B[k][j] of the chunk is accumulated exactly once, and
// consecutive steps s read consecutive A elements (128-bit LDS reads).
//
// As points at the wave's first A row in an LDS tile [rows][LDA] (row-major,
// m x k); Bs at the wave's first column in an LDS tile [TK][LDB] (k x n).
// acc[i][j] is the 32x32 block at rows 32*i, cols 32*j of the wave tile.
//
// Layouts: A rows of LDA floats, or (ASWZ) a dense [rows][TK] tile written by
// direct-to-LDS loads whose 16-byte slots are permuted by mt_swz; B either
// [TK][LDB] (k-major), or (BNM) n-major [cols][TK] swizzled like A and read
// 128 bits at a time.  Every layout feeds the MFMAs the same values in the
// same order, so results are identical across layouts.
// ---------------------------------------------------------------------------

template <int WM, int WN, int TK, int LDA, int LDB, bool ASWZ = false, bool BNM = false>
MT_INLINE void mt_mfma_tile_f32(const float* __restrict__ As, const float* __restrict__ Bs,
                                mt_f32x16 (&acc)[WM][WN], unsigned lane) {
    static_assert(TK % 8 == 0, "TK must be a multiple of 8");
    static_assert(LDA % 4 == 0, "LDA must keep 16-byte alignment");
    static_assert(!ASWZ || LDA == TK, "a swizzled A tile is dense");
    static_assert(!BNM || LDB == TK, "an n-major B tile is dense");
    constexpr int HALF = TK / 2;
    const unsigned li = lane & 31u;
    const unsigned lh = lane >> 5;
    // Swizzled tiles: the wave's first row is a multiple of 16, so row
    // 32 i + li of the wave permutes its slots by mt_swz(li).
    unsigned m = 0u;
    if constexpr (ASWZ || BNM) m = mt_swz<TK / 4>(li);
    const float* a_base = ASWZ ? As + li * TK : As + li * LDA + lh * HALF;
    const float* b_base = BNM ? Bs + li * TK : Bs + (lh * HALF) * LDB + li;
    // Raise this wave's issue priority while it feeds the matrix core, so a
    // wave still holding MFMAs is preferred over one writing the next chunk
    // to LDS or waiting at the barrier (measured +2.6-3.6 % on 4096^3 and
    // C4 GEMMs).  The priority of instruction issue inside a SIMD only.
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s0 = 0; s0 < HALF; s0 += 4) {
        const unsigned slot = (lh * HALF + (unsigned)s0) / 4u;  // swizzled tiles: logical 16-byte slot
        mt_f32x4 a[WM];
#pragma unroll
        for (int i = 0; i < WM; ++i)
            a[i] = ASWZ ? mt_ld4(a_base + i * 32 * TK + 4u * (slot ^ m)) : mt_ld4(a_base + i * 32 * LDA + s0);
        mt_f32x4 bv[BNM ? WN : 1];
        if constexpr (BNM) {
#pragma unroll
            for (int j = 0; j < WN; ++j) bv[j] = mt_ld4(b_base + j * 32 * TK + 4u * (slot ^ m));
        }
#pragma unroll
        for (int ss = 0; ss < 4; ++ss) {
            float b[WN];
#pragma unroll
            for (int j = 0; j < WN; ++j) b[j] = BNM ? bv[j][ss] : b_base[(s0 + ss) * LDB + j * 32];
#pragma unroll
            for (int i = 0; i < WM; ++i) {
#pragma unroll
                for (int j = 0; j < WN; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][ss], b[j], acc[i][j], 0, 0, 0);
                }
            }
        }
    }
    __builtin_amdgcn_s_setprio(0);
}

// ---------------------------------------------------------------------------
// fp32 products on the bf16 matrix cores.  A float is the sum of three bf16
// numbers: x1 = x rounded to bf16, x2 = x - x1 rounded to bf16, x3 = the rest.
// 24 = 8 + 8 + 8 significant bits, so the sum is exact, and each remainder is
// an exact fp32 subtraction.  Of the nine partial products of x y the six of
// at least 2^-16 |x y| are accumulated, smallest first,
//     x3 y1 + x2 y2 + x1 y3 + x2 y1 + x1 y2 + x1 y1,
// by v_mfma_f32_32x32x16_bf16 into the fp32 accumulator; x2 y3, x3 y2 and
// x3 y3 are below the last bit of the fp32 product.  Rounding x1 (instead of
// cutting it off) gives x2 a sign of its own: the MFMA drops what lies far
// below the accumulator's last bit, and with x2 y2 always of the product's
// sign that added up (all-positive operands, K = 4096: 3.4e-6 instead of 5.9e-7).
// (Three-part bf16 products: G. Henry, P. Tang, A. Heinecke, "Leveraging the
// bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations",
// ARITH 2019.)
//
// Why: the fp32 MFMA does 64 multiply-adds per cycle and SIMD, the bf16 one
// 1024, so six of them have 2.7 times its rate.  Measured on MI355X, 4096^3:
// 1018 us (135 TFLOP/s) with fp32 MFMAs, 741 us (185 TFLOP/s) this way; the
// matrix cores are then busy 63 % of the cycles and the clock has fallen from
// 2.05 to 1.68 GHz (a plain bf16 GEMM of 8192^3 reaches 1.22 PFLOP/s on the
// same GPU, six times 203 TFLOP/s: power, not the split, is the next limit).
// Error against 64 bits, relative 2-norm, fp32 MFMA -> split, N(0, 1) operands:
// K = 64: 1.44e-7 -> 1.09e-7; 512: 4.1e-7 -> 3.4e-7; 1024: 5.8e-7 -> 4.9e-7;
// 4096: 1.15e-6 -> 1.00e-6; 11008: 1.88e-6 -> 1.69e-6; all positive, 64:
// 1.17e-7 -> 0.86e-7; 1024: 4.7e-7 -> 3.3e-7; 4096: 9.4e-7 -> 5.9e-7; 11008:
// 1.52e-6 -> 0.96e-6 (fewer roundings of the accumulator: six per 16 k's, not
// eight).
//
// The splits are made in registers from fp32 LDS tiles, so every loader and
// prologue stays as it is.  A wave splits the WM + WN fragments it multiplies,
// 5.5 VALU operations per element against 6 WM WN MFMAs of 32 cycles: square
// wave tiles split the least per MFMA.  Each lane half supplies 8 consecutive
// k's of an MFMA's 16 (the chunk's two halves, as in mt_mfma_tile_f32).
//
// What a split cannot do: an infinite x, or one that rounds to an infinite x1
// (from 0x1.ffp+127), leaves a NaN or an infinity of the wrong sign as its
// remainder, which makes every sum it enters a NaN; mt_mfma_retry finds those by
// their results.  And an x below 2^-110 may have bits below 2^-133, bf16's
// smallest number (the MFMAs keep subnormals): the third part cuts them off, an
// error of up to 2^-133 times whatever the other operand is.  Results do not show
// that, so a split says whether it cut anything off (mt_lost): half a VALU operation
// per element, in every wave or in one of each row and column of waves (mt_own,
// mt_cut).  Measured on MI355X without and with it: 4096^3 661 -> 671 us, 4096 x
// 4096 x 11008 1850 -> 1932, 1531 x 1000 x 3001 96 -> 102, C4 MLP 5.86 -> 5.99 ms.
// Dearer were a running minimum and maximum of the operands held by every wave
// (4096^3 737 us where the look in every wave took 712), or taken by every lane of
// its share of the LDS tile (742), or a look at every fourth chunk branched to inside
// the asm of the split (691, but 2252 instead of 2103 for 4096 x 4096 x 8191).
// ---------------------------------------------------------------------------

typedef __bf16 mt_bf16x8 __attribute__((ext_vector_type(8)));

// Eight floats as three vectors of eight bf16.
struct mt_split8 {
    mt_u32x4 p1, p2, p3;
};

MT_INLINE unsigned mt_cvt_pk_bf16(float lo, float hi) {  // round to nearest even
    unsigned r;
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(lo), "v"(hi));
    return r;
}
MT_INLINE unsigned mt_pack_hi16(float lo, float hi) {  // upper halves of two floats
    return __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, hi), __builtin_bit_cast(unsigned, lo), 0x07060302u);
}
MT_INLINE float mt_keep_hi16(unsigned x) { return __builtin_bit_cast(float, x & 0xffff0000u); }

// Lanes whose splits of A's and of B's elements cut off nonzero bits.
struct mt_lost {
    unsigned long long a, b;
};

// A wave's note of what its own splits lost.
struct mt_own {
    static constexpr bool LOOK = true;
    mt_lost& lost;

    MT_INLINE mt_lost& open(mt_lost&) const { return lost; }
    MT_INLINE void tell(const mt_lost&) const {}
};

// Or the workgroup's: words in LDS, one for the waves that split the same rows of A
// and one for those that split the same columns of B, zeroed before the k loop and
// read after it.  One wave of each row and column of waves looks, the same one
// through the loop.
template <bool WAVE_LOOKS>
struct mt_cut {
    static constexpr bool LOOK = WAVE_LOOKS;
    unsigned* a;
    unsigned* b;

    MT_INLINE mt_lost& open(mt_lost& chunk) const { return chunk; }
    MT_INLINE void tell(const mt_lost& lost) const {
        if constexpr (LOOK) {
            if (__builtin_expect(lost.a != 0ull, 0)) *a = 1u;
            if (__builtin_expect(lost.b != 0ull, 0)) *b = 1u;
        }
    }
    MT_INLINE mt_lost told() const {
        return {(unsigned)__builtin_amdgcn_readfirstlane(*a), (unsigned)__builtin_amdgcn_readfirstlane(*b)};
    }
};

template <bool LOOK>
MT_INLINE mt_split8 mt_split(mt_f32x4 u, mt_f32x4 v, unsigned long long& lost) {
    mt_split8 o;
    unsigned low = 0u;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float x0 = q < 2 ? u[2 * q] : v[2 * q - 4], x1 = q < 2 ? u[2 * q + 1] : v[2 * q - 3];
        const unsigned h = mt_cvt_pk_bf16(x0, x1);
        o.p1[q] = h;
        const float r0 = x0 - __builtin_bit_cast(float, h << 16), r1 = x1 - mt_keep_hi16(h);
        const unsigned m = mt_cvt_pk_bf16(r0, r1);
        o.p2[q] = m;
        const float z0 = r0 - __builtin_bit_cast(float, m << 16), z1 = r1 - mt_keep_hi16(m);
        o.p3[q] = mt_pack_hi16(z0, z1);
        if constexpr (LOOK) low |= __builtin_bit_cast(unsigned, z0) | __builtin_bit_cast(unsigned, z1);
    }
    if constexpr (LOOK) lost |= __ballot((low & 0xffffu) != 0u);
    return o;
}

MT_INLINE mt_f32x16 mt_mfma_bf16(mt_u32x4 a, mt_u32x4 b, mt_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mt_bf16x8, a), __builtin_bit_cast(mt_bf16x8, b),
                                                   c, 0, 0, 0);
}

// The six partial products of one 32x32 block and 16 k's, smallest first.
MT_INLINE mt_f32x16 mt_mfma_parts(const mt_split8& a, const mt_split8& b, mt_f32x16 c) {
    c = mt_mfma_bf16(a.p3, b.p1, c);
    c = mt_mfma_bf16(a.p2, b.p2, c);
    c = mt_mfma_bf16(a.p1, b.p3, c);
    c = mt_mfma_bf16(a.p2, b.p1, c);
    c = mt_mfma_bf16(a.p1, b.p2, c);
    return mt_mfma_bf16(a.p1, b.p1, c);
}

// One row block of a step of 16 k's: a0, a1 the lane's 8 consecutive k's of A,
// b[j] column block j's parts.  Product by product over the column blocks, so
// an MFMA does not wait for the one before it (C4 X @ W1: 1840 us; block by
// block 1924 us).
template <int WN, bool LOOK>
MT_INLINE void mt_mfma_split(mt_f32x4 a0, mt_f32x4 a1, const mt_split8 (&b)[WN], unsigned long long& lost,
                             mt_f32x16 (&acc)[WN]) {
    const mt_split8 a = mt_split<LOOK>(a0, a1, lost);
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[j] = mt_mfma_bf16(a.p3, b[j].p1, acc[j]);
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[j] = mt_mfma_bf16(a.p2, b[j].p2, acc[j]);
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[j] = mt_mfma_bf16(a.p1, b[j].p3, acc[j]);
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[j] = mt_mfma_bf16(a.p2, b[j].p1, acc[j]);
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[j] = mt_mfma_bf16(a.p1, b[j].p2, acc[j]);
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[j] = mt_mfma_bf16(a.p1, b[j].p1, acc[j]);
}

// hook(q) runs before the LDS reads of each group of 8 k's, q = 0 .. TK/8 - 1:
// the mainloop issues its next chunk's loads there, spread over the MFMAs.
struct mt_no_hook {
    MT_INLINE void operator()(int) const {}
};

// The chunk in the layouts of mt_mfma_tile_f32.
template <int WM, int WN, int TK, int LDA, int LDB, bool ASWZ = false, bool BNM = false, typename N,
          typename H = mt_no_hook>
MT_INLINE void mt_mfma_tile(const float* __restrict__ As, const float* __restrict__ Bs, N notes,
                            mt_f32x16 (&acc)[WM][WN], unsigned lane, H hook = H{}) {
    constexpr bool LOOK = N::LOOK;
    mt_lost chunk = {};
    mt_lost& lost = notes.open(chunk);
    static_assert(TK % 16 == 0, "TK must be a multiple of 16");
    static_assert(LDA % 4 == 0, "LDA must keep 16-byte alignment");
    static_assert(!ASWZ || LDA == TK, "a swizzled A tile is dense");
    static_assert(!BNM || LDB == TK, "an n-major B tile is dense");
    constexpr int HALF = TK / 2;
    const unsigned li = lane & 31u;
    const unsigned lh = lane >> 5;
    unsigned m = 0u;
    if constexpr (ASWZ || BNM) m = mt_swz<TK / 4>(li);
    const float* a_base = ASWZ ? As + li * TK : As + li * LDA + lh * HALF;
    const float* b_base = BNM ? Bs + li * TK : Bs + (lh * HALF) * LDB + li;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s0 = 0; s0 < HALF; s0 += 8) {
        // swizzled tiles: logical 16-byte slots of the lane's two quads
        const unsigned slot0 = (lh * HALF + (unsigned)s0) / 4u, slot1 = slot0 + 1u;
        mt_split8 b[WN];
        hook(s0 / 4);
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            if constexpr (BNM) {
                const float* row = b_base + j * 32 * TK;
                b[j] = mt_split<LOOK>(mt_ld4(row + 4u * (slot0 ^ m)), mt_ld4(row + 4u * (slot1 ^ m)), lost.b);
            } else {
                mt_f32x4 q[2];
#pragma unroll
                for (int ss = 0; ss < 8; ++ss) q[ss / 4][ss % 4] = b_base[(s0 + ss) * LDB + j * 32];
                b[j] = mt_split<LOOK>(q[0], q[1], lost.b);
            }
        }
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            if (i == WM / 2) hook(s0 / 4 + 1);
            const float* row = a_base + i * 32 * LDA;
            const mt_f32x4 a0 = ASWZ ? mt_ld4(row + 4u * (slot0 ^ m)) : mt_ld4(row + s0);
            const mt_f32x4 a1 = ASWZ ? mt_ld4(row + 4u * (slot1 ^ m)) : mt_ld4(row + s0 + 4);
            mt_mfma_split<WN, LOOK>(a0, a1, b, lost.a, acc[i]);
        }
    }
    notes.tell(lost);
    __builtin_amdgcn_s_setprio(0);
}

// A long mainloop's chunk (MatmulMainloopFragment.held).  What one chunk leaves
// to the next is empty: fp32 MFMAs gained 1 % from a group of operands carried
// over the barrier, but the split's parts take the registers it was held in
// (4096^3 with the group carried: 739 us on 8 waves and 1494 us, spilled, on 16;
// without: 731 and 750 us).
template <int WM, int WN>
struct mt_mfma_group {};

template <int WM, int WN>
MT_INLINE void mt_mfma_group_run(const mt_mfma_group<WM, WN>&, mt_f32x16 (&)[WM][WN]) {}

template <int WM, int WN, int TK, int LDA, int LDB, bool ASWZ = false, bool BNM = false, typename N>
MT_INLINE void mt_mfma_tile_held(const float* __restrict__ As, const float* __restrict__ Bs, N notes,
                                 mt_f32x16 (&acc)[WM][WN], unsigned lane, mt_mfma_group<WM, WN>&, bool) {
    mt_mfma_tile<WM, WN, TK, LDA, LDB, ASWZ, BNM>(As, Bs, notes, acc, lane);
}

// Row (within a 32x32 output block) of accumulator register v held by `lane`;
// the column is lane % 32.
MT_INLINE unsigned mt_acc_row(int v, unsigned lane) {
    return 8u * (unsigned)(v >> 2) + 4u * (lane >> 5) + (unsigned)(v & 3);
}

// The lane, as a value the compiler computes nothing from ahead of its use: what a
// rare path needs of it must not take registers from the k loop before.
MT_INLINE unsigned mt_late(unsigned lane) {
    asm volatile("" : "+v"(lane));
    return lane;
}

// Largest magnitude of lines [l0, l1), elements [e0, e1) each, of a matrix whose
// lines are contiguous and `pitch` apart: the whole wave, 4 lines of 64 elements a
// load.
MT_INLINE float mt_largest(const float* __restrict__ src, size_t pitch, unsigned l0, unsigned l1, unsigned e0,
                           unsigned e1, unsigned lane) {
    constexpr unsigned UNROLL = 8u;
    float top = 0.0f;
    lane = mt_late(lane);
    for (unsigned e = e0 + 4u * (lane & 15u); e < e1; e += 64u)
        for (unsigned l = l0 + (lane >> 4); l < l1; l += 4u * UNROLL) {
            mt_f32x4 x[UNROLL];
#pragma unroll
            for (unsigned u = 0; u < UNROLL; ++u)
                x[u] = l + 4u * u < l1 ? mt_ld_slot(src + (l + 4u * u) * pitch + e, e1 - e) : mt_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (unsigned u = 0; u < UNROLL; ++u)
#pragma unroll
                for (int q = 0; q < 4; ++q) top = __builtin_fmaxf(top, __builtin_fabsf(x[u][q]));
        }
    return mt_wave_max(top);
}

// Whether the wave's accumulators may differ from the fp32 products' sums for
// want of range: a value that is not finite (every sum an infinite or NaN operand
// enters is a NaN here, where fp32 may give an infinity; and a part of a product
// may pass the largest float where the product does not, as x1 is rounded up); a
// nonzero one below 2^-96, whose smaller partial products may be subnormal; and,
// where an operand's splits cut bits off, one these could matter to: K of them are
// below K 2^-133 times the other operand's largest magnitude, which ta() and tb()
// look up.  So the weights of a softmax may underflow beside ordinary ones.  Rows
// and columns from `rows` and `cols` on are outside the matrix.  Wave uniform.
template <int WM, int WN, typename TA, typename TB>
MT_INLINE bool mt_mfma_retry(const mt_f32x16 (&acc)[WM][WN], const mt_lost& lost, unsigned K, unsigned rows,
                             unsigned cols, unsigned lane, TA ta, TB tb) {
    bool odd = false;
    if (__builtin_expect((lost.a | lost.b) != 0ull, 0)) {
        const float top = __builtin_fmaxf(lost.b != 0ull ? ta() : 0.0f, lost.a != 0ull ? tb() : 0.0f);
        const float least = 0x1.0p-107f * (float)K * top;  // 2^25 times what both may have lost
        lane = mt_late(lane);
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int j = 0; j < WN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    float x = acc[i][j][v];
                    // else |x| is computed ahead for this and the check below: 29 spills
                    // a tile (4096 x 4096 x 11008: 1993 us with them, 1932 without)
                    asm volatile("" : "+v"(x));
                    odd |= !(__builtin_fabsf(x) >= least) && 32u * (unsigned)i + mt_acc_row(v, lane) < rows &&
                           32u * (unsigned)j + (lane & 31u) < cols;
                }
    }
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float x = __builtin_fabsf(acc[i][j][v]);
                odd |= !(x >= 0x1.0p-96f && x <= 0x1.fffffep+127f) && x != 0.0f;
            }
    return __builtin_expect(__ballot(odd) != 0ull, 0);
}

// The wave's blocks at (m0, n0) over k in [kb, ke) again, with fp32 MFMAs on
// operands read from global memory: fa(row, k) and fb(col, k) give four k's from k
// on with their prologue applied, 0 outside the matrix and from ke on.  Each wave
// decides and works alone: no LDS, no barrier.  A lane half takes 8 k's of 16, so a
// row of an operand is two 128-bit loads where it lies along k.  Measured on MI355X
// with an infinity in every wave of 4096^3: 4270 -> 2550 us, one infinity in
// all 1430 -> 1120 us (a k at a time before, 8 in flight).
template <int WM, int WN, typename FA, typename FB>
MT_INLINE void mt_mfma_exact(FA fa, FB fb, unsigned m0, unsigned n0, unsigned kb, unsigned ke, unsigned lane,
                             mt_f32x16 (&acc)[WM][WN]) {
    lane = mt_late(lane);
    const unsigned li = lane & 31u, lh = lane >> 5;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) acc[i][j] = mt_f32x16{};
    for (unsigned k = kb; k < ke; k += 16u) {
        mt_f32x4 a[2][WM], b[2][WN];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const unsigned kk = k + 8u * lh + 4u * (unsigned)q;
#pragma unroll
            for (int i = 0; i < WM; ++i) a[q][i] = fa(m0 + 32u * (unsigned)i + li, kk);
#pragma unroll
            for (int j = 0; j < WN; ++j) b[q][j] = fb(n0 + 32u * (unsigned)j + li, kk);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < WM; ++i)
#pragma unroll
                    for (int j = 0; j < WN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q][i][s], b[q][j][s], acc[i][j], 0, 0, 0);
    }
}

// Four k's of an operand from k on: element (line, k) at src[line * ls + k * ks],
// 0 for lines from `lines` and k's from ke on; f(raw, k) applies its prologue.
template <bool ALONG_K, typename F>
MT_INLINE mt_f32x4 mt_exact_quad(const float* __restrict__ src, size_t ls, size_t ks, unsigned line, unsigned k,
                                 unsigned lines, unsigned ke, F f) {
    mt_f32x4 x = {0.f, 0.f, 0.f, 0.f};
    if (line < lines && k < ke) {
        const float* p = src + line * ls + k * ks;
        if constexpr (ALONG_K) {
            x = mt_ld_slot(p, ke - k);
        } else {
#pragma unroll
            for (unsigned s = 0; s < 4u; ++s)
                if (k + s < ke) x[s] = p[s * ks];
        }
#pragma unroll
        for (unsigned s = 0; s < 4u; ++s)
            if (k + s < ke) x[s] = f(x[s], k + s);
    }
    return x;
}

// ---------------------------------------------------------------------------
// Row-owning waves for matmuls 128 columns wide, on the split products above.
// A workgroup of 16 waves makes a 256 x 128 tile; waves 2w and 2w + 1 own rows
// 32 w .. 32 w + 31, one column half each (two 32x32 blocks).  A goes from
// global memory straight into the registers of the wave that splits it (a
// prologue applied there).  B is split once per workgroup, not once per wave:
// each lane loads 8 k's of one column, splits them and writes the three parts
// to LDS as 16-byte units, which the MFMAs read as they are.
//   k: step s of a 64-wide chunk takes k's 16 s .. 16 s + 15, lane half h the 8
//      from 16 s + 8 h (k group 2 s + h);
//   LDS stage: unit (group g, column n) of part 1 at 128 g + n of `hi`, part 2
//      1024 units on, part 3 at 128 g + n of `lo`: lanes read and write
//      consecutive units, so no bank conflicts.
// Why: with 16 rows to a wave (fp32 MFMAs) every wave read all of B; LDS reads
// were a quarter of the MFMA time and would be all of it at the split's rate.
// Two waves sharing rows read half of B each and load A twice, the second time
// from the caches.
// ---------------------------------------------------------------------------

// This lane's share of a B chunk: column tid % 128, k group tid / 128.
struct mt_rw_stage {
    float v[8];

    MT_INLINE void fetch(const float* __restrict__ src, unsigned ldb, unsigned k0, unsigned tid) {
        const float* p = src + (size_t)(k0 + 8u * (tid >> 7)) * ldb + (tid & 127u);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = p[(size_t)e * ldb];
    }
    MT_INLINE void commit(float* hi, float* lo, unsigned tid, mt_cut<true> cut) const {
        mt_lost lost = {};
        const mt_split8 x = mt_split<true>(mt_f32x4{v[0], v[1], v[2], v[3]}, mt_f32x4{v[4], v[5], v[6], v[7]}, lost.b);
        reinterpret_cast<mt_u32x4*>(hi)[tid] = x.p1;
        reinterpret_cast<mt_u32x4*>(hi)[1024u + tid] = x.p2;
        reinterpret_cast<mt_u32x4*>(lo)[tid] = x.p3;
        cut.tell(lost);
    }
};

// This lane's A values of step s of the chunk at k0: arow points at its row's
// column 8 (lane / 32).
MT_INLINE void mt_rw_load(mt_f32x4 (&a)[2], const float* __restrict__ arow, unsigned k0, int s) {
    a[0] = mt_ld4(arow + k0 + 16u * (unsigned)s);
    a[1] = mt_ld4(arow + k0 + 16u * (unsigned)s + 4u);
}

// One 64-wide chunk: a holds its raw A values (pa applies the prologue) and,
// step by step, receives those of the chunk at k_next (`more`): a step's loads
// have the rest of this chunk and the steps before theirs in the next to land.
template <bool LOOK, typename P>
MT_INLINE void mt_rw_chunk(mt_f32x4 (&a)[4][2], const float* __restrict__ arow, unsigned k_next, bool more,
                           const float* __restrict__ hi, const float* __restrict__ lo, unsigned n0, P pa, unsigned lane,
                           mt_cut<LOOK> cut, mt_f32x16 (&acc)[1][2]) {
    mt_lost lost = {};
    const mt_u32x4* __restrict__ h4 = reinterpret_cast<const mt_u32x4*>(hi) + n0 + (lane & 31u);
    const mt_u32x4* __restrict__ l4 = reinterpret_cast<const mt_u32x4*>(lo) + n0 + (lane & 31u);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const unsigned g = 128u * (2u * (unsigned)s + (lane >> 5));
        mt_f32x4 x[2];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e / 4][e % 4] = pa(a[s][e / 4][e % 4]);
        if (more) mt_rw_load(a[s], arow, k_next, s);
        const mt_split8 xa = mt_split<LOOK>(x[0], x[1], lost.a);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const mt_split8 b = {h4[g + 32u * j], h4[1024u + g + 32u * j], l4[g + 32u * j]};
            acc[0][j] = mt_mfma_parts(xa, b, acc[0][j]);
        }
    }
    cut.tell(lost);
    __builtin_amdgcn_s_setprio(0);
}

// ---------------------------------------------------------------------------
// Skinny matmuls: few output tiles, so what counts is how fast B streams in
// (decoding: a few rows against whole weights) or how short the chain of
// dependent loads is (small matrices).  A workgroup makes a 16 MB x 64 tile;
// its waves split the tile's k's, and workgroups may split them further.  Both
// operands go from global memory straight into the registers of
// v_mfma_f32_16x16x4f32 (D[16x16] += A[16x4] * B[4x16]; lane l supplies
// A[l%16][l/16], B[l/16][l%16] and holds D[4 (l/16) + i][l%16]): nothing is
// shared between waves, so there is no LDS stage and no barrier in the k loop,
// and each wave keeps its own loads in flight.
//   k: a group of 16 k's is 4 steps; lane quarter g = l/16 takes k's
//      4 g .. 4 g + 3 of it, one per step, so an A row is one 128-bit load;
//   n: B read along n (row-major): the load of step s holds row k + 4 g + s,
//      columns 4 c .. 4 c + 3, c = l%16 -- column block j is columns 4 c + j,
//      and 16 lanes read 256 contiguous bytes; B read along k (a transposed
//      view): load j holds column 16 j + c, the quarter's 4 k's.
// The waves' sums meet in LDS and are added in wave order; workgroups that
// split a tile add theirs through the workspace in split order (the last to
// arrive does, mt_sn_arrive), so results do not depend on timing.
// ---------------------------------------------------------------------------

// One group's B values at k (k < ke; rows from ke on are 0): b[s][j] (along n)
// or b[j][s] (along k) for step s, column block j.
template <bool ALONG_K, bool NT>
MT_INLINE void mt_sn_load_b(mt_f32x4 (&b)[4], const float* __restrict__ src, unsigned pitch, unsigned k, unsigned ke,
                            unsigned n0, unsigned N, unsigned lane) {
    const unsigned c = lane & 15u, kg = k + 4u * (lane >> 4);
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        const unsigned major = ALONG_K ? n0 + 16u * (unsigned)x + c : kg + (unsigned)x;
        const unsigned minor = ALONG_K ? kg : n0 + 4u * c;
        const unsigned major_end = ALONG_K ? N : ke, minor_end = ALONG_K ? ke : N;
        mt_f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (major < major_end) {
            const float* p = src + (size_t)major * pitch + minor;
            if (minor + 4u <= minor_end) {
                v = NT ? mt_ld4u_nt(p) : mt_ld4u(p);
            } else {
                if (minor < minor_end) v.x = p[0];
                if (minor + 1u < minor_end) v.y = p[1];
                if (minor + 2u < minor_end) v.z = p[2];
            }
        }
        b[x] = v;
    }
}

// One group's A values: row block m, this lane's 4 k's, its prologue applied:
// fv(row, k) gives four k's at once (QUADS), fa(row, k) one.
template <int MB, bool QUADS, typename FV, typename FA>
MT_INLINE void mt_sn_load_a(mt_f32x4 (&a)[MB], FV fv, FA fa, unsigned k, unsigned ke, unsigned m0, unsigned M,
                            unsigned lane) {
    const unsigned kg = k + 4u * (lane >> 4);
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        const unsigned row = m0 + 16u * (unsigned)m + (lane & 15u);
        mt_f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (row < M) {
            if (QUADS && kg + 4u <= ke) {
                v = fv(row, kg);
            } else {
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    if (kg + (unsigned)s < ke) v[s] = fa(row, kg + (unsigned)s);
            }
        }
        a[m] = v;
    }
}

// The wave's groups [g0, g1) of 16 k's each (K in all), UNROLL of them loaded
// before any is multiplied.  Two keep the registers low enough for the other
// waves to hide the loads (8 rows, 4096 x 11008: 39.8 us with 2, 42.7 with 4,
// 47.8 with 8).
template <int MB, bool QUADS_A, bool B_ALONG_K, bool NT_B, typename FV, typename FA>
MT_INLINE void mt_sn_mainloop(FV fv, FA fa, const float* __restrict__ B, unsigned ldb, unsigned g0, unsigned g1,
                              unsigned K, unsigned m0, unsigned M, unsigned n0, unsigned N, unsigned lane,
                              mt_f32x4 (&acc)[MB][4]) {
    constexpr int UNROLL = 2;
    for (unsigned g = g0; g < g1; g += UNROLL) {
        mt_f32x4 a[UNROLL][MB], b[UNROLL][4];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            if (g + (unsigned)u >= g1) {  // wave uniform
#pragma unroll
                for (int m = 0; m < MB; ++m) a[u][m] = mt_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int x = 0; x < 4; ++x) b[u][x] = mt_f32x4{0.f, 0.f, 0.f, 0.f};
                continue;
            }
            mt_sn_load_b<B_ALONG_K, NT_B>(b[u], B, ldb, 16u * (g + (unsigned)u), K, n0, N, lane);
            mt_sn_load_a<MB, QUADS_A>(a[u], fv, fa, 16u * (g + (unsigned)u), K, m0, M, lane);
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int m = 0; m < MB; ++m)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][m][s], B_ALONG_K ? b[u][j][s] : b[u][s][j],
                                                                        acc[m][j], 0, 0, 0);
    }
}

// Partial sums handed between workgroups of one launch: device-scope stores
// and loads (through the XCD's L2, which is not coherent with the others')
// instead of the fences of mt_rr_publish -- an agent-scope release writes back
// the whole L2 and an acquire invalidates it, per workgroup.
MT_INLINE void mt_sn_put(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
MT_INLINE float mt_sn_get(const float* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The same 128 bits at a time, at byte offset `at` of a part of `bytes` bytes
// (16: the device-scope policy of buffer instructions).
struct mt_sn_part {
    __amdgpu_buffer_rsrc_t r;
    MT_INLINE mt_sn_part(float* base, unsigned bytes) {
        r = __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00020000);
    }
    MT_INLINE void put(unsigned at, mt_f32x4 v) const {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(mt_u32x4, v), r, at, 0, 16);
    }
    MT_INLINE mt_f32x4 get(unsigned at) const {
        return __builtin_bit_cast(mt_f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 16));
    }
};
// Count this workgroup in, its device-scope stores complete; true in the last of
// `parts` workgroups, which resets the counter for the next launch.
MT_INLINE bool mt_sn_arrive(unsigned* counter, unsigned parts, unsigned* flag_lds) {
    __builtin_amdgcn_s_waitcnt(0);  // every lane's stores have reached memory
    __syncthreads();
    if (threadIdx.x == 0u) {
        const unsigned old = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = old + 1u == parts;
        if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag_lds = last ? 1u : 0u;
    }
    __syncthreads();
    return *flag_lds != 0u;
}

// Element e = 64 row + col of a wave's tile in its LDS slab: register
// (m, j, i) of lane l at 64 (16 m + 4 j + i) + l.
template <bool B_ALONG_K>
MT_INLINE unsigned mt_sn_slot(unsigned e) {
    const unsigned row = e >> 6, col = e & 63u;
    const unsigned j = B_ALONG_K ? col >> 4 : col & 3u, c = B_ALONG_K ? col & 15u : col >> 2;
    return 64u * (16u * (row >> 4) + 4u * j + (row & 3u)) + 16u * ((row >> 2) & 3u) + c;
}

// ---------------------------------------------------------------------------
// K-resident row waves for matmuls with a short K (64 or 128) whose B is read
// along K (n-major: B[k][n] at n * ldb + k, such as the transposed view K^T
// of attention scores).  Each of a workgroup's 16 waves owns 16 rows of a
// 256-row block and keeps those rows' whole K in registers (K/4 floats per
// lane, loaded once).  B streams through LDS in 128-column chunks, n-major
// [128][K], two stages; each chunk is a finished 256 x 128 output tile, 8
// column blocks of v_mfma_f32_16x16x4f32 per wave, stored with 128-bit
// stores issued between the MFMAs of the next column half.
//   k: lane group g = l/16 takes k = g K/4 + s at step s < K/4, so its A
//      values are K/4 consecutive floats of its row (128-bit loads), and its
//      B values of 4 consecutive steps are one 128-bit LDS read, logical
//      16-byte slot g K/16 + t (t = s/4) of the B row;
//   n: column block j puts lane column c = l%16 at output column
//      64 (j/4) + 4c + j%4, so blocks 4h .. 4h + 3 give a lane 4 consecutive
//      output columns of each of its rows (a 128-bit store; 256 contiguous
//      bytes per 16 lanes);
//   LDS: B row n (K/4 slots) holds logical slot L at physical slot
//      L ^ mt_kr_swz(n).  gfx950 serves a ds_read_b128 in 4 passes of 16
//      lanes, each pass two 8-lane groups k and k ^ 3 of one half-wave
//      (lanes 0-7 with 24-31, 8-15 with 16-23, ...), from 64 4-byte banks
//      (byte address mod 256) -- measured with rocprof's LDS bank-conflict
//      counter on fixed lane/address patterns.  Lane (g, c) reads row
//      64 (j/4) + 4c + j%4 at logical slot g K/16 + t, and a pass holds
//      lanes c < 8 of one g with lanes c >= 8 of g ^ 1.  So mt_kr_swz(n) is
//      c mod 8 for K = 128 (bit 3 of the slot then follows g) and c for
//      K = 64 (bit 3 follows c): the 16 lanes of every pass hit 16
//      distinct 16-byte bank groups.
// ---------------------------------------------------------------------------

template <int K>
MT_HD unsigned mt_kr_swz(unsigned n) {
    static_assert(K == 64 || K == 128, "K-resident rows hold K = 64 or 128");
    return (n >> 2) & (K == 128 ? 7u : 15u);
}

// Where wave-load `inst`, lane `lane` of the B loader puts its 16 bytes: row r
// of the [128][K] chunk, physical slot p = (64 inst + lane) mod K/4; it loads
// the row's logical slot p ^ mt_kr_swz(r).
template <int K>
MT_HD void mt_kr_slot(unsigned inst, unsigned lane, unsigned& r, unsigned& logical) {
    constexpr unsigned S = K / 4;
    const unsigned slot = inst * 64u + lane;
    r = slot / S;
    logical = (slot % S) ^ mt_kr_swz<K>(r);
}

// 128 n-major B rows of K floats (row stride ldb floats, a multiple of 4)
// into a dense swizzled LDS chunk [128][K] by direct-to-LDS loads; each
// lane's byte offsets from the chunk origin are computed once.
template <int K, int NT>
struct mt_kr_dma {
    static constexpr int S = K / 4;
    static constexpr int INSTR = 128 * S / 64;
    static constexpr int PERW = INSTR / (NT / 64);
    static_assert(INSTR % (NT / 64) == 0, "the chunk must split into the same number of wave loads per wave");
    unsigned off[PERW];
    unsigned lds_off;

    MT_INLINE mt_kr_dma(unsigned ldb, unsigned tid) {
        const unsigned lane = tid & 63u;
        const unsigned wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        lds_off = wave * PERW * 1024u;
#pragma unroll
        for (int q = 0; q < PERW; ++q) {
            unsigned r, logical;
            mt_kr_slot<K>(wave * PERW + q, lane, r, logical);
            off[q] = (r * ldb + 4u * logical) * 4u;
        }
    }

    // B rows n0 .. n0 + 127 of src (B[k][n] = src[n * ldb + k]).
    MT_INLINE void fetch(const float* __restrict__ src, unsigned ldb, unsigned n0, float* lds) const {
        const unsigned long long origin = mt_uniform_addr(src + (size_t)n0 * ldb);
        const unsigned base = __builtin_amdgcn_readfirstlane(mt_lds_addr(lds)) + lds_off;
#pragma unroll
        for (int q = 0; q < PERW; ++q) mt_dma16(origin, off[q], base + (unsigned)q * 1024u);
    }
};

// The B values of one group: quad t (4 steps), column half h (blocks
// 4h .. 4h + 3): rows 64h + 4c + jj of the chunk, logical slot g K/16 + t.
struct mt_kr_group {
    mt_f32x4 b[4];
};

template <int K>
MT_INLINE mt_f32x4 mt_kr_b(const float* __restrict__ bl, unsigned phys_slot, int h, int jj) {
    return mt_ld4(bl + (unsigned)(64 * h + jj) * K + 4u * phys_slot);
}

struct mt_kr_no_hook {
    MT_INLINE void operator()(int) const {}
};

// One 128-column chunk from the B stage at Bs and this lane's K/4 A values
// (already transformed by any prologue), column half by column half: groups
// q = 0 .. K/8 - 1 are quad t = q mod K/16 of half h = q / (K/16), 16 MFMAs
// each, steps 0 .. 3 in turn over the half's 4 blocks.  The group's B
// values sit in one set of 16 registers: block jj's value for the next
// group is read right after its step-3 MFMA (the order pinned with
// sched_barrier; measured on C5 S, as fast as two register sets, which
// cost 15 more VGPRs).  hook(q) runs after
// group q's MFMAs are issued -- the kernel stores one row of the other
// half's finished accumulators there, so the stores go out between MFMAs.
// The k order per output element is fixed: quads t = 0 .. K/16 - 1, steps
// 0 .. 3 within each.
template <int K, typename H = mt_kr_no_hook>
MT_INLINE void mt_kr_chunk(const mt_f32x4 (&a)[K / 16], const float* __restrict__ Bs, unsigned lane,
                           mt_f32x4 (&acc)[8], H hook = H{}) {
    constexpr int T = K / 16;
    const unsigned c = lane & 15u;
    const unsigned g = lane >> 4;
    const float* __restrict__ bl = Bs + 4u * c * (unsigned)K;
    const unsigned sw = mt_kr_swz<K>(4u * c);  // the same for every row this lane reads
    __builtin_amdgcn_s_setprio(1);
    mt_kr_group f;
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) f.b[jj] = mt_kr_b<K>(bl, (g * (unsigned)T) ^ sw, 0, jj);
#pragma unroll
    for (int q = 0; q < 2 * T; ++q) {
        const int h = q / T, t = q % T;
        const int hn = (q + 1) / T, tn = (q + 1) % T;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ss = 0; ss < 3; ++ss)
#pragma unroll
            for (int jj = 0; jj < 4; ++jj)
                acc[4 * h + jj] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][ss], f.b[jj][ss], acc[4 * h + jj], 0, 0, 0);
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            acc[4 * h + jj] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][3], f.b[jj][3], acc[4 * h + jj], 0, 0, 0);
            if (q + 1 < 2 * T) f.b[jj] = mt_kr_b<K>(bl, (g * (unsigned)T + (unsigned)tn) ^ sw, hn, jj);
        }
        __builtin_amdgcn_sched_barrier(0);
        hook(q);
    }
    __builtin_amdgcn_s_setprio(0);
}

// Raw buffer access to an output of `bytes` bytes: one descriptor per
// workgroup (32-bit data, stride 0), so a store takes one per-lane byte
// offset and one wave-uniform one instead of a 64-bit address per lane; the
// hardware drops a store beyond the range instead of writing it.

MT_INLINE mt_u32x4 mt_raw_buffer(const void* p, unsigned bytes) {
    const unsigned long long a = mt_uniform_addr(static_cast<const float*>(p));
    return mt_u32x4{(unsigned)a, (unsigned)(a >> 32) & 0xffffu, (unsigned)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}

// 16 bytes to rs + voff + soff (POLICY 16: sc1, device scope, written
// through the L2; 0: default).  The store reads its data registers after
// it issues, so nothing may write them in the next cycles: on MI355X a
// v_mul writing the first data register right after a 128-bit buffer store
// (the compiler inserts no wait state for a buffer store with an SGPR
// soffset) let the store write the new value in lanes 12-15 of a 16-lane
// group -- the next row's score in C5 S, in 16-32 elements per run.  The
// store is therefore issued here with two wait states behind it.
template <int POLICY = 0>
MT_INLINE void mt_buffer_store4(mt_f32x4 v, mt_u32x4 rs, unsigned voff, unsigned soff) {
    const unsigned so = __builtin_amdgcn_readfirstlane(soff);
    if constexpr (POLICY == 16)
        asm volatile("buffer_store_dwordx4 %0, %1, %2, %3 offen sc1\n\ts_nop 1"
                     :
                     : "v"(v), "v"(voff), "s"(rs), "s"(so)
                     : "memory");
    else
        asm volatile("buffer_store_dwordx4 %0, %1, %2, %3 offen\n\ts_nop 1"
                     :
                     : "v"(v), "v"(voff), "s"(rs), "s"(so)
                     : "memory");
}

MT_INLINE void mt_zero(mt_f32x16& a) {
#pragma unroll
    for (int i = 0; i < 16; ++i) a[i] = 0.f;
}

// ---------------------------------------------------------------------------
// Stream-K schedule for a persistent matmul: T output tiles of C k-chunks on
// P workgroups.  The first DP = floor(T / P) * P tiles are data-parallel
// (workgroup w takes tiles w, w + P, ...).  The k-chunks of the remaining
// T - DP tiles -- U = (T - DP) * C units, tile-major -- are cut into P
// contiguous ranges of U / P units; range j goes to workgroup P - 1 - j.
// A workgroup walks its range first (at most a partial tile, whole tiles,
// a partial tile), then its data-parallel tiles.
//
// A tile split between ranges is finished by the workgroup whose range
// holds its chunk 0 (the owner).  The others (contributors) hold later
// chunks at the start of their ranges: they store their partial
// accumulators to the workspace, then raise their flag.  Ranges after the
// owner's belong to lower workgroup indices, so an owner only ever waits for
// workgroups dispatched before it, which did that work first.  The owner
// adds the partials in range order, so results are reproducible.
//
// Workspace: MT_WS_HEAD words of flags (one per workgroup, 0 = empty; word
// MT_WS_HEAD - 1 is the error word), then one partial tile per workgroup.
// Flags start at 0 and every owner clears the flags it consumed, so the
// next launch starts clean.  A wait gives up after MT_SK_SPIN_LIMIT polls
// and sets the error word instead of hanging; the host checks it.
// ---------------------------------------------------------------------------

#define MT_WS_HEAD 1024u
#define MT_SK_SPIN_LIMIT (1u << 22)
// The schedule is plain integer arithmetic, callable from host code too (the
// CPU test suite checks its coverage and wait order).

struct mt_stream_k {
    unsigned chunks, P, w, j, dp, sk0, nsk, ndp;
    unsigned long long U, lo, hi;

    MT_HD void init(unsigned tiles, unsigned chunks_, unsigned P_, unsigned w_) {
        chunks = chunks_, P = P_, w = w_;
        dp = (tiles / P) * P;
        U = (unsigned long long)(tiles - dp) * chunks;
        j = P - 1u - w;
        lo = U * j / P;
        hi = U * (j + 1u) / P;
        sk0 = (unsigned)(lo / chunks);
        nsk = hi > lo ? (unsigned)((hi - 1u) / chunks) - sk0 + 1u : 0u;
        ndp = dp > w ? (dp - w + P - 1u) / P : 0u;
    }
    MT_HD unsigned items() const { return nsk + ndp; }
    // Item `it`: output tile t, chunks [kb, ke).
    MT_HD void item(unsigned it, unsigned& t, unsigned& kb, unsigned& ke) const {
        if (it < nsk) {
            const unsigned st = sk0 + it;
            const unsigned long long ts = (unsigned long long)st * chunks;
            kb = (unsigned)((lo > ts ? lo : ts) - ts);
            ke = (unsigned)((hi < ts + chunks ? hi : ts + chunks) - ts);
            t = dp + st;
        } else {
            t = w + (it - nsk) * P;
            kb = 0u;
            ke = chunks;
        }
    }
    // Start unit of range jj (jj <= P).
    MT_HD unsigned long long range_lo(unsigned jj) const { return U * jj / P; }
    // The owner of the split tile whose units end at tend: the first range
    // at offset >= c (c >= 1) after its own that is non-empty and starts
    // before tend, as an offset (its workgroup is w - offset); 0 when none
    // is left.  (Ranges are empty when there are fewer units than ranges.)
    MT_HD unsigned contributor(unsigned c, unsigned long long tend) const {
        for (; j + c < P; ++c) {
            const unsigned long long a = range_lo(j + c);
            if (a >= tend) return 0u;
            if (range_lo(j + c + 1u) > a) return c;
        }
        return 0u;
    }
};

// The partial slot's base pointer passes through an empty asm statement, so
// the slot addresses are computed where they are used (the rare hand-over
// branches) and not hoisted out of the tile loop, where they would hold
// registers across the mainloop.
MT_INLINE float* mt_ws_slot_base(float* p) {
    asm volatile("" : "+s"(p));
    return p;
}
MT_INLINE unsigned* mt_ws_flag(float* ws, unsigned w) { return reinterpret_cast<unsigned*>(ws) + w; }
MT_INLINE unsigned* mt_ws_error(float* ws) { return reinterpret_cast<unsigned*>(ws) + (MT_WS_HEAD - 1u); }
MT_INLINE float* mt_ws_part(float* ws, unsigned w, unsigned tile_floats) {
    return mt_ws_slot_base(ws + MT_WS_HEAD + (size_t)w * tile_floats);
}

// Contributor: each wave waits for its own partial stores to complete
// (s_waitcnt on every counter), the workgroup meets at the barrier, then
// lane 0 alone publishes them with one agent-scope release store of the
// flag.  An agent-scope release writes back the XCD's L2; doing it once per
// hand-over instead of once per wave kept the C4 X @ W1 kernel at 2.7 ms
// instead of 3.0 ms.
MT_INLINE void mt_sk_signal(unsigned* flag) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0u) __hip_atomic_store(flag, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}

// Owner: lane 0 polls the contributor's flag with relaxed loads (bounded),
// then one agent-scope acquire fence (it invalidates the CU's L1 and the
// XCD's L2 once, not once per poll or per wave) and clears the flag for the
// next launch; the barrier orders every lane's partial loads after it.
MT_INLINE void mt_sk_wait(unsigned* flag, unsigned* error) {
    if (threadIdx.x == 0u) {
        unsigned n = 0u;
        while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u) {
            if (++n >= MT_SK_SPIN_LIMIT) {
                __hip_atomic_store(error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        __hip_atomic_store(flag, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// Row reduction of a matmul's output in its epilogue (the matmul -> reduction
// epilogue extension): the kernel that writes Y = A @ B (+ a register
// epilogue) also writes r[row] = op over Y[row][:], op one of sum (OP 0),
// max (1), min (2), product (3) with the row-reduction kernels' combines.
//
// 1. A wave holds WM x WN blocks of 32x32 values in the MFMA layout (lane l:
//    column l % 32 of each block, 16 rows per block, mt_acc_row).  Per lane,
//    the WN blocks of each row are combined in block order: 16 WM values.
// 2. Across the 32 lanes of each half-wave, halving exchanges over lane bits
//    0, 1, 2, 3, 4: a lane keeps the half of its values its bit selects,
//    sends the other half to the lane that differs in that bit and combines
//    what it receives into what it keeps; once a lane holds one value, the
//    remaining steps combine both lanes' values.  Lane l then holds
//    MT_RR_KEEP(WM) values, value k for wave row mt_rr_row<WM>(l, k).  The
//    low bits go first: their exchanges are the most numerous and DPP quad
//    permutes serve them within the VALU op; bits 2-4 go through ds_swizzle.
// 3. The waves that share rows combine through LDS in wave order, one value
//    per row of the tile (generated code).
// 4. Each tile publishes its row values in the workspace (after the
//    MT_WS_HEAD flag words); the workgroup that publishes a row block's last
//    tile combines the block's tiles in column order and writes r.
// Every step has a fixed order, so results are reproducible; max and min
// give the same values as the row-reduction kernel, sum and product round
// differently (another summation order).
// ---------------------------------------------------------------------------

#define MT_RR_KEEP(WM) ((16 * (WM)) >= 32 ? (16 * (WM)) / 32 : 1)

template <int OP>
MT_INLINE float mt_rr_op(float a, float b) {
    if constexpr (OP == 0) return a + b;
    else if constexpr (OP == 1) return fmaxf(a, b);
    else if constexpr (OP == 2) return fminf(a, b);
    else return a * b;
}

// v from the lane whose index differs from this lane's in the bits of M
// (M < 32): DPP quad permutes for 1 and 2, ds_swizzle in its bitmask mode
// (and 0x1F, xor M within each 32 lanes) for 4, 8 and 16.
template <unsigned M>
MT_INLINE float mt_xor_lanes(float v) {
    const int x = __float_as_int(v);
    int y;
    if constexpr (M == 1u)
        y = __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xF, 0xF, false);  // quad_perm [1, 0, 3, 2]
    else if constexpr (M == 2u)
        y = __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xF, 0xF, false);  // quad_perm [2, 3, 0, 1]
    else
        y = __builtin_amdgcn_ds_swizzle(x, (int)((M << 10) | 0x1Fu));
    return __int_as_float(y);
}

// Wave-tile row of value k that `lane` keeps after mt_wave_row_reduce<WM>.
template <int WM>
MT_HD unsigned mt_rr_row(unsigned lane, int k) {
    unsigned idx = 0u, n = 16u * (unsigned)WM;
    for (int b = 0; b <= 4; ++b) {
        if (n > 1u) {
            n >>= 1;
            if ((lane >> b) & 1u) idx += n;
        }
    }
    idx += (unsigned)k;
    const unsigned i = idx >> 4, r = idx & 15u;
    return 32u * i + 8u * (r >> 2) + 4u * (lane >> 5) + (r & 3u);
}

// One exchange step over lane bit M with N values per lane (N == 1: combine).
template <unsigned M, int N, int OP>
MT_INLINE void mt_rr_step(float* w, unsigned lane) {
    if constexpr (N > 1) {
        constexpr int H = N / 2;
        const bool hi = (lane & M) != 0u;
#pragma unroll
        for (int k = 0; k < H; ++k) {
            const float send = hi ? w[k] : w[k + H];
            const float keep = hi ? w[k + H] : w[k];
            w[k] = mt_rr_op<OP>(keep, mt_xor_lanes<M>(send));
        }
    } else {
        w[0] = mt_rr_op<OP>(w[0], mt_xor_lanes<M>(w[0]));
    }
}

template <int WM, int WN, int OP>
MT_INLINE void mt_wave_row_reduce(const mt_f32x16 (&val)[WM][WN], unsigned lane, float (&out)[MT_RR_KEEP(WM)]) {
    constexpr int V = 16 * WM;
    float w[V];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float x = val[i][0][r];
#pragma unroll
            for (int j = 1; j < WN; ++j) x = mt_rr_op<OP>(x, val[i][j][r]);
            w[16 * i + r] = x;
        }
    constexpr int N1 = V > 1 ? V / 2 : 1, N2 = N1 > 1 ? N1 / 2 : 1, N3 = N2 > 1 ? N2 / 2 : 1, N4 = N3 > 1 ? N3 / 2 : 1;
    mt_rr_step<1u, V, OP>(w, lane);
    mt_rr_step<2u, N1, OP>(w, lane);
    mt_rr_step<4u, N2, OP>(w, lane);
    mt_rr_step<8u, N3, OP>(w, lane);
    mt_rr_step<16u, N4, OP>(w, lane);
#pragma unroll
    for (int k = 0; k < MT_RR_KEEP(WM); ++k) out[k] = w[k];
}

// Publish this workgroup's tile values of a row block: every wave's stores
// complete, the workgroup meets, then lane 0 increments the block's counter
// with one agent-scope acquire-release add (the release writes back the
// XCD's L2; the acquire invalidates the caches before the combining loads).
// Returns true in every lane of the workgroup that published the block's
// last tile, which resets the counter to 0 for the next launch.
MT_INLINE bool mt_rr_publish(unsigned* counter, unsigned tiles, unsigned* flag_lds) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0u) {
        const unsigned old = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = old + 1u == tiles;
        if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag_lds = last ? 1u : 0u;
    }
    __syncthreads();
    return *flag_lds != 0u;
}

// Publish row block `blk`'s tile values written by this workgroup (a tile
// earlier: its stores completed long ago, so the publish's wait is short)
// and, in the workgroup that completes the block, combine the block's `tn`
// column tiles in order into out[m0 + t] for the rows below M.
template <int OP, unsigned TM, unsigned NT>
MT_INLINE void mt_rr_finish(float* ws, unsigned blk, unsigned tn, unsigned m0, unsigned M, float* out,
                            unsigned* flag_lds) {
    const float* part = ws + MT_WS_HEAD + (size_t)blk * tn * TM;
    if (mt_rr_publish(reinterpret_cast<unsigned*>(ws) + blk, tn, flag_lds)) {
        for (unsigned t = threadIdx.x; t < TM; t += NT) {
            if (m0 + t >= M) continue;
            float r = part[t];
            for (unsigned n = 1u; n < tn; ++n) r = mt_rr_op<OP>(r, part[(size_t)n * TM + t]);
            out[m0 + t] = r;
        }
    }
}
