// bf_passes.h -- what the propagation passes' kernels share: precision tags, pass
// flags and the launch arguments of the row, column, bounce and pair passes.
#pragma once
#include "bf_internal.h"
#include "bf_dftmm.h"

namespace bf {

// ---------------------------------------------------------------------------
// descriptors
// ---------------------------------------------------------------------------
enum : uint32_t { RF_INV = 1, RF_RTAB = 2, RF_MASK = 4, RF_FWD = 8 };
enum : uint32_t { CF_FWD = 1, CF_KMID = 2, CF_INV = 4, CF_KLOAD = 8, CF_INSHIFT = 16, CF_OUTSHIFT = 32 };
enum : uint32_t { DF_FWD = 1, DF_AMAX = 2, DF_EOUT_ASSIGN = 4 };
enum : int { FD_WHOLE = 1 };  // FieldDesc.pad: column pass stores every row of this field
constexpr int FD_PAIR_SHIFT = 8;  // FieldDesc.pad >> FD_PAIR_SHIFT: region pair of a cheerleader pair step

// Precision tags: `double` = FP64 storage and arithmetic; `float` = fields stored
// in FP32 in HBM, all in-register arithmetic (FFTs, phases, boundary updates) in
// FP64; `f32pure` = FP32 storage and FP32 arithmetic.
template <typename T> struct Storage { using type = T; };
template <> struct Storage<f32pure> { using type = float; };
template <typename T> struct Compute { using type = double; };
template <> struct Compute<f32pure> { using type = float; };
#define BF_TYPES(T)                           \
    using S = typename Storage<T>::type;      \
    using C = typename Compute<T>::type

// The matrix-core line transforms of a pass (bf_dftmm.h)
struct DftArgs {
    const double2* tab = nullptr;  // (cos, sin)(2 pi a b / n), [dft_tab_rows(n)][dft_ld(n)]
    int lo = 0;                    // smallest folded index inside the aperture along the line
    int smax = 1;                  // waves that may share an output tile (set by the launcher)
};

template <typename T>
struct RowArgs {
    cplx<typename Storage<T>::type>* base;
    const FieldDesc* fd;
    int nf, nx, ny;
    const cplx<typename Compute<T>::type>* tw;
    uint32_t flags;
    const cplx<typename Compute<T>::type>* rtab;
    const double* X;
    const double* Y;
    double R2;
    const int* active;
    // rows outside [ylo, yhi) are skipped (not read, not written) when yhi > ylo
    int ylo, yhi;
    DftArgs dft;  // transforms along x on the matrix cores (table null: not built)
};

template <typename T>
struct ColArgs {
    const cplx<typename Storage<T>::type>* src;
    cplx<typename Storage<T>::type>* dst;
    const FieldDesc* fd;
    int nf, nx, ny;
    const cplx<typename Compute<T>::type>* tw;
    uint32_t flags;
    const cplx<typename Compute<T>::type>* ktab;
    int tx;  // columns per block
    const int* active;
    // Row band: rows outside [ylo, yhi) are known to be zero on input (they are
    // not loaded) and are not needed on output (not stored), except for the
    // fields whose descriptor carries FD_WHOLE, stored whole.
    int ylo, yhi;
    int kq;  // 0: full k-space tables; else quarter tables of row width kq = nx/2 (dancer propagation)
    int all_whole;  // every field is stored whole (the band limits the loads only)
    DftArgs dft;
};

template <typename T>
__device__ __forceinline__ bool in_band(const ColArgs<T>& a, int y) {
    return (unsigned)(y - a.ylo) < (unsigned)(a.yhi - a.ylo);
}
__device__ __forceinline__ bool store_whole(const FieldDesc& d) { return (d.pad & FD_WHOLE) != 0; }

template <typename T>
struct DancerRowArgs {
    cplx<typename Storage<T>::type>* fields;  // [fb][R][2][ny][nx]
    int R, nx, ny;
    int rm;  // slot holding the right-moving fields this bounce
    const cplx<typename Compute<T>::type>* tw;
    const cplx<typename Compute<T>::type>* rtab;
    const int* rtab_idx;  // [fb][R], -1: none
    const zd* coef;       // boundary reflectivities r_b, b = 0..R (r_R = 0 appended)
    const double* X;
    const double* Y;
    double R2;
    const uint32_t* keep_tab;  // [ny][nx/16] aperture bits of the register path, or null
    int keep_band;             // band class of keep_tab: no bit outside [keep_band, 15 - keep_band]
    uint32_t flags;
    zd* Eout;  // [nslices][ny][nx] per frequency slot, stride eout_fstride
    size_t eout_fstride;
    int slice;
    double* amax;  // [fb]
    const int* active;
    int* count;  // [fb] bounce counters
    // Row band [ylo, yhi): outside it the next bounce's aperture zeroes every
    // row, so those rows are only needed for Eout at the exit boundary.  The
    // launcher fills the tile map from the band and its rows per block.
    int ylo, yhi;
    int tile0, nband, ntiles;
    DftArgs dft;
};

// Block -> (boundary b, row tile).  Blocks [0, nband (R+1)) cover the row tiles
// that meet the band at every boundary; the remaining ntiles - nband blocks
// cover the other row tiles at the exit boundary only (exit_only: Eout is
// accumulated, nothing is stored because the aperture zeroes those rows).
template <typename T>
__device__ __forceinline__ void dancer_block(const DancerRowArgs<T>& a, int i, int& b, int& tile, bool& exit_only) {
    const int nb = a.nband * (a.R + 1);
    if (i < nb) {
        b = i / a.nband;
        tile = a.tile0 + i % a.nband;
        exit_only = false;
    } else {
        const int j = i - nb;
        b = a.R;
        tile = j < a.tile0 ? j : j + a.nband;
        exit_only = true;
    }
}

__device__ __forceinline__ void atomic_max_pos(double* addr, double v) {
    // non-negative doubles order like their bit patterns
    atomicMax(reinterpret_cast<unsigned long long*>(addr), (unsigned long long)__double_as_longlong(v));
}

template <typename T>
struct ChPairArgs {
    cplx<typename Storage<T>::type>* F;  // [fb][Nd][K]
    // entry e (one frequency of one region pair (i, i+1)): fd[2e] field i,
    // fd[2e+1] field i+1; i = fd[2e].pad >> FD_PAIR_SHIFT
    const FieldDesc* fd;
    int ny, rows;
    const cplx<typename Compute<T>::type>* tw;
    const cplx<typename Compute<T>::type>* rtab;  // null: no tilt/surface tables
    const zd* coef;  // [i][4]: rl, tr, rr, tl of boundary i
    const int* active;
    int ylo, yhi;  // rows processed
    int xout;      // store the masked row transform of the updated fields
    const double* X;
    const double* Y;
    double R2;  // aperture radius squared
    DftArgs dft;
};

template <typename T>
inline unsigned dancer_tiles(DancerRowArgs<T>& a, int rows) {
    a.ntiles = (a.ny + rows - 1) / rows;
    if (a.yhi > a.ylo) {
        a.tile0 = a.ylo / rows;
        a.nband = (a.yhi + rows - 1) / rows - a.tile0;
    } else {
        a.tile0 = 0;
        a.nband = 0;
    }
    return (unsigned)(a.nband * (a.R + 1) + (a.ntiles - a.nband));
}

// matrix-core passes (bf_dft.hip), T = double or float (FP64 arithmetic)
std::shared_ptr<DevBuf> dft_table(bf_ctx* ctx, int n);
template <typename T> void launch_rows_dft(RowArgs<T> a, hipStream_t s);
template <typename T> void launch_cols_dft(ColArgs<T> a, hipStream_t s);
template <typename T> void launch_dancer_rows_dft(DancerRowArgs<T> a, int fb, hipStream_t s);
template <typename T> void launch_ch_pair_dft(ChPairArgs<T> a, int nx, int entries, hipStream_t s);

}  // namespace bf
