// erp_internal.h — shared declarations of the gfx950 HIP implementation of
// the per-shot raypath / phasor / range-compression path.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>
#include <string>
#include <vector>
#include <atomic>
#include <condition_variable>
#include <deque>
#include <memory>
#include <mutex>
#include <thread>

#include "../../include/erp.h"

// ---------------------------------------------------------------------------
// error plumbing: every failure is returned as a status, never exit()
// ---------------------------------------------------------------------------
struct ErpError {
    int code;
    std::string msg;
};

#define ERP_HIP_TRY(expr)                                                     \
    do {                                                                      \
        hipError_t _e = (expr);                                               \
        if (_e != hipSuccess)                                                 \
            throw ErpError{ERP_E_HIP, std::string(#expr) + ": " +             \
                                          hipGetErrorString(_e)};             \
    } while (0)

#define ERP_CHECK_LAUNCH(name)                                                \
    do {                                                                      \
        hipError_t _e = hipGetLastError();                                    \
        if (_e != hipSuccess)                                                 \
            throw ErpError{ERP_E_HIP, std::string("launch ") + (name) +       \
                                          ": " + hipGetErrorString(_e)};      \
    } while (0)

// ---------------------------------------------------------------------------
// constants shared by every kernel (the reference's literals)
// ---------------------------------------------------------------------------
// geometry_kernels.cu:45 `const float pi = 3.14159265f`
#define ERP_PI_F 3.14159265f
// geometry_kernels.cu:388,411 `pow(4 * 3.14159, 2)` evaluated in double
#define ERP_FOURPI5_SQ (4.0 * 3.14159 * 4.0 * 3.14159)

// FFT twiddle table size (largest supported transform)
#define ERP_TWN (1 << 18)

// ---------------------------------------------------------------------------
// device buffers
// ---------------------------------------------------------------------------
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
    // a region of memory the buffer does not own (see Arena): never freed,
    // never grown; asking for more than it holds is an error
    bool borrowed = false;
    void borrow(void* q, size_t n) {
        p = q;
        bytes = n;
        borrowed = true;
    }
    void ensure(size_t n) {
        if (n <= bytes) return;
        if (borrowed)
            throw ErpError{ERP_E_NOMEM, "a work buffer needs " + std::to_string(n) +
                                            " bytes, its scratch region holds " +
                                            std::to_string(bytes)};
        if (p) hipFree(p);
        p = nullptr;
        bytes = 0;
        if (n == 0) return;
        hipError_t e = hipMalloc(&p, n);
        if (e != hipSuccess) {
            p = nullptr;
            throw ErpError{ERP_E_NOMEM, "hipMalloc of " + std::to_string(n) +
                                            " bytes failed: " + hipGetErrorString(e)};
        }
        bytes = n;
    }
    // for sizes that vary from call to call: grow by up to a quarter more
    // than asked (never beyond cap, the caller's bound on n), so that a
    // slowly rising size does not free and reallocate (hipFree waits for the
    // device) on every call
    void ensure_grow(size_t n, size_t cap) {
        if (n > bytes) ensure(std::max(n, std::min(n + n / 4, cap)));
    }
    void release() {
        if (p && !borrowed) hipFree(p);
        p = nullptr;
        bytes = 0;
        borrowed = false;
    }
    template <class T> T* as() const { return static_cast<T*>(p); }
};

// Device memory of one run carved from a region the caller provides (the
// allocation-free entry point): 256-byte aligned bump allocation, nothing is
// freed before the run ends.
struct Arena {
    char* base = nullptr;
    size_t cap = 0;
    size_t used = 0;
    static size_t round(size_t n) { return (n + 255) & ~(size_t)255; }
    size_t left() const { return cap - used; }
    void* take(size_t n, const char* what) {
        const size_t r = round(std::max<size_t>(n, 1));
        if (r > left())
            throw ErpError{ERP_E_NOMEM, std::string("scratch exhausted: ") + what + " needs " +
                                            std::to_string(r) + " bytes, " +
                                            std::to_string(left()) + " of " +
                                            std::to_string(cap) + " left"};
        void* p = base + used;
        used += r;
        return p;
    }
    template <class T> T* take_n(size_t n, const char* what) {
        return static_cast<T*>(take(sizeof(T) * n, what));
    }
    void lend(DevBuf& b, size_t n, const char* what) { b.borrow(take(n, what), round(std::max<size_t>(n, 1))); }
};

struct erp_mesh {
    erp_ctx* ctx;
    int device;
    int64_t F;
    DevBuf soa;  // 12 x F float32 (stride Fpad)
    int64_t Fpad;
    // every facet normal equals +-(u x v) to 1e-5: kernels may derive n from
    // the tangents instead of loading it
    bool frame_ok = false;
    // facets in rows of tile_nx (a multiple of 64, row count a multiple of
    // 32): the surface kernels then take them in 64 x 32 tiles; 0 = in order
    int tile_nx = 0;
};

struct erp_targets {
    erp_ctx* ctx;
    int device;
    int64_t T;
    DevBuf xyzn;  // 6 x Tpad float32
    DevBuf type;  // T uint8
    int64_t Tpad;
    int64_t n0 = 0;  // targets of type 0
};

// FFT plan for one power-of-two size N (see erp_fft.hip)
struct FftPlan {
    int N = 0, log2N = 0;
    int N1 = 0, N2 = 0;  // two-pass split: N = N1 (row, contiguous) * N2 (rows)
    bool two_pass = false;
};

// A cached table: entries are shared between the context's cache and the runs
// that read them (TableHold), so a cache can drop an entry at any time.  Freed
// with the last reference; hipFree waits for the device, which covers work
// that a run has queued and not waited for.
struct Table {
    Table() = default;
    Table(const Table&) = delete;
    Table& operator=(const Table&) = delete;
};
using TableHold = std::vector<std::shared_ptr<void>>;

// Per-(nr, dr, res) chirp spectra
struct ChirpKey {
    int nr;
    float dr, res;
    int kind;  // 0 = padded (linear), 1 = circular (genChirp), rst in key2
    float rst;
    bool operator==(const ChirpKey& o) const {
        return nr == o.nr && dr == o.dr && res == o.res && kind == o.kind && rst == o.rst;
    }
};

struct ChirpSpec : Table {
    ChirpKey key;
    DevBuf spec;  // P complex64, permuted forward order, scaled by 1/P
    DevBuf nat;   // the same spectrum in natural order (filled on first use)
    DevBuf wl;    // the natural one in the layout of k_tpair_wl (first use)
    size_t bytes() const { return spec.bytes + nat.bytes + wl.bytes; }
    ~ChirpSpec() {
        spec.release();
        nat.release();
        wl.release();
    }
};

// Band crop and decimation of a shot's summed spectrum (convolveComplex's
// cropSpectrum + takeEveryOtherComplex, elementary_kernels.cu:187-194,
// 258-353).  DFT_L, crop to |freq| <= B, IDFT_L and keeping every second
// sample of the L = 2 nr - 1 samples c is a convolution with the band's real
// L-periodic kernel D:
//     out[i] = sum_j c[j] D[2 i - j],   i < nr,
// i.e. (j even and odd apart) two linear convolutions of nr points with
// D[2 d] and D[2 d - 1], which fit the P >= 2 nr - 1 point transforms.
// tab: the spectra of those two kernels (output i at P / 2 + i), P complex64
// each in fft_forward's order, scaled by 1 / P^2 (the two inverses).
struct BandTables : Table {
    int nr = 0, P = 0;
    float smpl = 0, B = 0;
    DevBuf tab;
    size_t bytes() const { return tab.bytes; }
    ~BandTables() { tab.release(); }
};

// Narrow-band chain of typed targets (erp_narrow.hip): band, decimation and
// tables of one (nr, dr, res, smpl, B)
struct NarrowPlan {
    int ok;                  // the chain takes this run
    int nr, K;               // kept frequencies |k| <= K
    int q, Tq, T;            // decimation, filter half length T = q Tq
    int iL0, nL, iR0, nR;    // first column and columns (multiples of 16) per part
    int Nu, nfb;             // all columns; blocks of 16 bins per filter tile
    double kappa;            // dr / res
    const float* tab;        // rows of e_k and M_k (k_narrow_table)
    const float* fir;        // filter operand of k_narrow_fir
};
struct NarrowTables : Table {
    int nr = 0;
    float dr = 0, res = 0, smpl = 0, B = 0;
    NarrowPlan plan{};
    DevBuf tab;
    size_t bytes() const { return tab.bytes; }
    ~NarrowTables() { tab.release(); }
};
constexpr int kNarrowSlice = 32;  // pairs per slice
// entries from one pair row to the next: 256 bytes past a power of two, so
// that the rows of a slice, read side by side, fall on different channels
inline int narrow_stride(int P) { return P / 2 + 32; }

// Pinned host words of a run, which the kernels write directly (a copy back
// is a launch of its own, 4.7 us): the counts of a batch (V per row, then U per
// block of two), the target counts, the window check, then target lists of up
// to kPinList entries.  Sizes for the rows of a multi-track batch.
constexpr int kPinCounts = 384;
constexpr int kPinTargets = 512;
constexpr size_t kPinList = 16384;
constexpr size_t kPinWords = kPinCounts + kPinTargets + 8 + kPinList;

struct WorkBufs {
    int* pin = nullptr;  // kPinWords pinned words, owned by the context or slot
    DevBuf cnt, off, V, Vd, tcnt, tlist, tcount;  // counts / offsets
    DevBuf rec;        // compacted facet records
    DevBuf bounds;     // per-shot bounds of illuminated facets
    DevBuf psurf;      // S x P complex: surface phasor trace (padded)
    DevBuf srow;       // S x nr FP64 / fixed-point surface bins + S per-shot maxima
    DevBuf refl;       // S x nr complex
    DevBuf shotS;      // S x P complex: per-shot spectral accumulator
    DevBuf blu;        // S x 2P complex: workspace of the band crop
    DevBuf tA, tB, tC; // per-target chunk buffers, C x P complex
    DevBuf pairs;      // chunk pair list
    DevBuf t0trace;    // S x P complex: summed type-0 target histograms
    DevBuf dpart;      // S x splits x nr FP64 complex: partial direct sinc sums
    DevBuf shots;      // S erp_shot
    DevBuf prisms;
    DevBuf out;        // S x nr complex (device output staging)
    DevBuf nvalid;     // S int32
    DevBuf oow;        // count of target terms outside their pair's bin window
    // shot-pair target kernel: union masks, counts and offsets per block of
    // two shots; block records; work items with their slices and segments
    DevBuf umask, ucnt, uoff, ubase, brec, items;
    DevBuf bbox;       // per (shot, facet block) box of the lit facets
};

// stage timers: events recorded on the run stream, resolved after it syncs
struct StageTimer {
    bool on = false;
    double ms[ERP_NSTAGES] = {};
    int64_t launches[ERP_NSTAGES] = {};
    double units[ERP_NSTAGES] = {};
    struct Pending {
        int stage;
        hipEvent_t a, b;
        double units;
    };
    std::vector<Pending> pending;
    std::vector<hipEvent_t> pool;
    hipEvent_t get();
    void begin(int stage, hipStream_t s, double units);
    void end(hipStream_t s);
    void resolve();  // after a stream sync
    void reset();
    int cur = -1;
};

struct ErpSlot;  // asynchronous job worker (erp_api.hip)

struct MtState;
void mt_state_free(MtState* m);

struct erp_ctx {
    int device = 0;
    StageTimer prof;
    hipStream_t stream = nullptr;
    std::string last_error;
    DevBuf twiddle;  // ladder table of the LDS FFT stages (65536 complex64)
    std::vector<std::pair<int, DevBuf*>> inter;  // inter-pass twiddles per size
    std::vector<std::shared_ptr<ChirpSpec>> chirps;
    std::vector<std::shared_ptr<BandTables>> bands;
    std::vector<std::shared_ptr<NarrowTables>> narrows;
    WorkBufs work;
    std::mutex mu;        // serialises the synchronous entry points
    // guards inter / chirps / bands / narrows (shared by all streams); recursive because
    // building a chirp or band table runs FFTs that look up inter tables
    std::recursive_mutex cache_mu;
    int num_cu = 0;
    // asynchronous jobs: worker slots, each with its own thread, stream and
    // work buffers, fed from one FIFO
    std::vector<ErpSlot*> slots;
    std::deque<erp_job*> queue;
    std::mutex qmu;
    std::condition_variable qcv;
    bool stopping = false;
    // caps on the batch shapes (erp_set_tuning; 0 = default)
    std::atomic<int64_t> tune_shots{0}, tune_pairs{0};
    // multi-track batches: rows per batch (0 = default), launch directly
    // instead of replaying captured graphs (> 0)
    std::atomic<int64_t> tune_rows{0}, tune_direct{0};
    // > 0 only in tests: shift every pair's bin window up by this many bins
    std::atomic<int64_t> tune_shift{0};
    // > 0: the plain target kernel one (shot, target) pair at a time
    std::atomic<int64_t> tune_single{0};
    MtState* mt = nullptr;  // buffers and graphs of erp_run_tracks
};

// ---------------------------------------------------------------------------
// FFT interface (erp_fft.hip)
// ---------------------------------------------------------------------------
FftPlan fft_plan(int N);
// Forward transform of `batch` rows of length N (row stride N), in place.
// Output in the plan's permuted order (natural order for single-pass sizes).
void fft_forward(erp_ctx* ctx, const FftPlan& p, float2* data, int batch, hipStream_t s);
// Inverse (unnormalised) of a permuted-order spectrum, in place, natural output.
void fft_inverse(erp_ctx* ctx, const FftPlan& p, float2* data, int batch, hipStream_t s);
void fft_init_twiddles(erp_ctx* ctx);
// Fused per-target spectral chain (erp_fft.hip): for n pairs with windowed
// inward traces in A (rows of P), accumulates scale * sum_p FFT(A_p) *
// FFT(window(IFFT(FFT(A_p) G))) into S[shot] for each shot segment.  Groups
// [gbeg, gend) partition the pairs without crossing shots; segment k sums
// groups (two-pass sizes) or pairs (single-pass sizes) [gseg_beg, gseg_end).
// one workgroup per (shot, target) pair, whole chain in LDS: P = 2n, n the
// next power of two of nr, from 1024 to 16384 (nr < n: the cropped variant)
bool target_half_supported(const FftPlan& p, int nr);
int target_half_slice();
// the chain runs with the wave-local transforms (k_tpair_wl): its range
// kernel spectra are then in that kernel's layout (wl_perm_table) and its
// rows are summed with target_sum_half(..., wl = true)
bool target_wl(const FftPlan& p);
// Gwl = Gnat in the layout of k_tpair_wl (P complex64 each)
void wl_perm_table(const float2* Gnat, float2* Gwl, int P, hipStream_t st);
// Gpair / npairs_dev (multi-track batches): per-pair range kernel spectra
// and the pair count on the device, n then being the grid's bound
void target_pairs_half(erp_ctx* ctx, const FftPlan& p, const float2* A, const int* pbase,
                       const int* pwin, int nr, int n, const float2* Gnat, float2* work,
                       hipStream_t st, const float4* const* Gpair = nullptr,
                       const int* npairs_dev = nullptr);
// seg_scale (multi-track batches): per-segment scale instead of `scale`;
// seq: each slice added to S on its own, in order, so that S does not
// depend on how launches group the slices (deterministic mode)
void target_sum_half(const FftPlan& p, const float2* work, float2* partial, const int* sl_beg,
                     const int* sl_end, int nslices, const int* seg_shot, const int* seg_beg,
                     const int* seg_end, int nseg, float2* S, float scale, hipStream_t st,
                     const float* seg_scale = nullptr, bool seq = false, bool wl = false);
// natural-order copy of a forward spectrum produced by fft_forward
void fft_natural_order(const FftPlan& p, const float2* src, float2* dst, hipStream_t st);
// Surface range compression of `rows` rows: FP64 bins srow (nr per row; det:
// fixed point, scaled by its row's V and smax) -> out (nr per row), by the
// spectrum G, or each row's track's (trk, rk; a track without one gets
// zeros).  work: rows x P, unused by single-pass sizes.
struct TrackK;
struct RowK;
struct FinalOut;
void surface_conv_rows(erp_ctx* ctx, const FftPlan& p, const double2* srow, int nr, int rows,
                       bool det, const unsigned* smax, const int* Vs, const float2* G,
                       float2* work, float2* out, const TrackK* trk, const RowK* rk,
                       hipStream_t st);
// spectra of the band kernels of (nr, smpl, B) into tab (2 P complex64)
void build_band(erp_ctx* ctx, const FftPlan& p, float2* tab, int nr, float smpl, float B,
                hipStream_t st);
// Last stage of typed targets: each row's summed spectrum S (P, overwritten)
// -> c = IFFT(S), cropped to the band and decimated, written as fo says.
// work: rows x 2P, unused by single-pass sizes.
void shot_final_rows(erp_ctx* ctx, const FftPlan& p, float2* S, float2* work, int nr, int rows,
                     const float2* tab, const FinalOut& fo, hipStream_t st);
// Specular typed targets of single-pass sizes: prod[p] = FFT(B_p) FFT(z_p),
// z_p the range-compressed window of A_p, summed per segment into S
void target_spectra_small(erp_ctx* ctx, const FftPlan& p, const float2* A, const float2* B, int nr,
                          int n, const float2* G, float2* prod, const int* seg_shot,
                          const int* seg_beg, const int* seg_end, int nseg, float2* S,
                          hipStream_t st);
void target_spectra_fused(erp_ctx* ctx, const FftPlan& p, float2* A, float2* Y,
                          const int* pbase, const int* pwin, int nr, int n, const float2* G,
                          float2* work, int ngroups, const int* gbeg, const int* gend,
                          const int* gseg_shot, const int* gseg_beg, const int* gseg_end,
                          int nseg, float2* S, float scale, hipStream_t st);

// ---------------------------------------------------------------------------
// pipeline (erp_pipeline.hip)
// ---------------------------------------------------------------------------
// timer: stage timers to record into, or nullptr (asynchronous jobs).
// arena: nullptr, or the region every work buffer and table of the run is
// carved from (then `work` must be empty and nothing is allocated; batch
// shapes shrink to fit and a job that cannot fit fails with ERP_E_NOMEM).
void erp_run_impl(erp_ctx* ctx, const erp_params* par, const erp_mesh* mesh,
                  const erp_targets* targets, const erp_shot* shots, int64_t ns,
                  const erp_prism* prisms, int64_t nprisms, float2* out_dev,
                  int32_t* nvalid_dev, uint32_t flags, hipStream_t stream,
                  WorkBufs& work, StageTimer* timer, Arena* arena = nullptr);
int64_t erp_footprint_impl(const erp_params* par, int64_t F, int64_t T, int64_t ns);
// multi-track batches of the eligible tracks, every other track alone
void erp_run_tracks_impl(erp_ctx* ctx, const erp_track* tracks, int64_t ntracks, uint32_t flags,
                         hipStream_t stream);
// focused rows row0 .. row0 + nrows - 1 of an Nr x Na radargram (erp_focus.hip)
void focus_rows(const float2* rdr, int Nr, int Na, int row0, int nrows, const int* row_hs,
                const int* row_nsx, const int64_t* row_off, const int* rows, const float2* filt,
                float2* out, hipStream_t st);
// 12 x Fpad SoA of a height grid (see erp_mesh_from_heights)
void mesh_from_heights(const double* heights, int64_t nx, int64_t ny, double fs, double ox,
                       double oy, float* soa, int64_t Fpad, hipStream_t st);
// ny x nx FP64 heights of a synthetic terrain into device memory h (see
// erp_mesh_from_terrain; erp_terrain.hip); synchronous on st
void terrain_heights(erp_ctx* ctx, const erp_terrain& t, double* h, hipStream_t st);

// Kernel-side parameter block (derived once per run on the host).
struct KPar {
    float lam, fs, P, ks, eps1, eps2, nu1, nu2, alpha1, alpha2, rng_res, dr;
    float c, c1, c2;
    float piLlam;      // PI_F*fs/lam (facet_G's sinc argument scale)
    float Dmax;        // 4*PI_F*fs^2/lam^2
    float fs_lam;      // fs/lam (facetReradiation)
    float fs2_lam;     // fs*fs/lam
    float nf;          // sqrt(eps_2) in float (accumulateTarget's n)
    int ortho;         // every facet frame (u, v, n) orthonormal (see sc_angles)
    float sqrtP;
    float invK;        // 1/(4*3.14159)^2
    float sqrt_e1e2;   // sqrt(eps_1/eps_2)
    float sqrt_e2e1;   // sqrt(eps_2/eps_1)
    double drd, inv_dr, cos_ap, n_d, inv_cyc, lam_d;
    // c1/c2 and c/c2 (genRefrPhasor, refrRadarSignal) divided in FP64: a
    // float quotient is off by up to 6e-8, i.e. 5e-5 rad of phase over a
    // 300 m refracted leg at 60 MHz
    double c1c2, cc2;
    // second subsurface medium below z = zi (has3 = 0: none): dn = n3 - n2,
    // tsq = sqrt(1 - rho23^2) (amplitude factor of a crossing path),
    // n_lo / n_hi = min / max(n2, n3) (window bounds)
    int has3;
    double zi, dn, n_lo, n_hi;
    float tsq;
    double B, smpl;
    int nr, P_fft, rerad;
    int row_live;      // entries of a pair row the spectral chain reads: P_fft / 2
                       // for the per-pair LDS chain, nr for the narrow-band one,
                       // P_fft otherwise
    int row_stride;    // entries from one pair row to the next
    uint32_t mode;
    uint64_t seed;
    int win_shift;     // 0; > 0 only to test the target kernel's window check
};

// Multi-track batches (erp_run_tracks): the rows of a batch are shots of
// several tracks of one range length; every kernel that reads a track's
// data takes it from that track's descriptor instead of its arguments.
struct TrackK {
    KPar kp;
    const float* mesh;             // 12 x Fpad SoA
    int64_t Fpad, F;
    int nblk, tile_nx, frame_ok;
    const float* tg;               // 6 x Tpad targets
    int64_t Tpad;
    int T;
    const unsigned char* ttype;
    const float2* g_surf;          // surface range kernel spectrum (fft order)
    const float2* g_targ_nat;      // target range kernel spectrum (natural order, or
                                   // in the layout of k_tpair_wl where it runs)
    const float2* band;            // band tables of the track (BandTables::tab)
    float2* out;                   // the track's radargram, ns x nr (device)
    int32_t* nvalid;               // its illuminated counts (device) or null
    float tscale;                  // -1 / sqrt(P): outward trace of a target
    NarrowPlan narrow;             // groups of the narrow-band chain
};
struct RowK {
    int trk;   // track of the row
    int shot;  // the row's shot index within its track
};

// Where a row's samples go (the combine step of combineRadarSignals,
// radar_kernels.cu:302-311): plus refl and add (either may be null), zero
// where Vs is 0, into a run's out and nvalid or its track's radargram (trk)
struct FinalOut {
    const float2* refl;
    const float2* add;
    const int* Vs;
    float2* out;
    int32_t* nvalid;
    const TrackK* trk;
    const RowK* rk;
};
// false: a padding row of a multi-track batch
__device__ __forceinline__ bool final_row(const FinalOut& fo, int r, int nr, float2** o,
                                          const float2** tab) {
    if (fo.trk) {
        const RowK row = fo.rk[r];
        if (row.shot < 0) return false;
        const TrackK& t = fo.trk[row.trk];
        *o = t.out + (size_t)row.shot * nr;
        *tab = t.band;
        if (t.nvalid && blockIdx.x == 0 && threadIdx.x == 0) t.nvalid[row.shot] = fo.Vs[r];
    } else {
        *o = fo.out + (size_t)r * nr;
        if (fo.nvalid && blockIdx.x == 0 && threadIdx.x == 0) fo.nvalid[r] = fo.Vs[r];
    }
    return true;
}
__device__ __forceinline__ float2 final_value(const FinalOut& fo, size_t i, bool live, float2 v) {
    if (!live) return make_float2(0.f, 0.f);
    if (fo.refl) v = make_float2(fo.refl[i].x + v.x, fo.refl[i].y + v.y);
    if (fo.add) v = make_float2(v.x + fo.add[i].x, v.y + fo.add[i].y);
    return v;
}


// rows of a multi-track batch (trk null: one run)
struct NarrowMt {
    const TrackK* trk;
    const RowK* rk;
    const int* pshot;  // row of each pair
};
// the largest kept frequency index of cropSpectrum (elementary_kernels.cu:
// 258-278): freq = k smpl / L, kept unless |freq| > B; -1: none
int band_limit(int nr, float smpl, float B);
void zero_words(float2* p, size_t n, hipStream_t st);
// plan of a run (p.ok: the narrow-band chain takes it), its table size, its
// tables (synchronous on st)
NarrowPlan narrow_plan(int nr, float dr, float res, float smpl, float B);
size_t narrow_table_floats(const NarrowPlan& p);
void narrow_build(NarrowPlan& p, float* tab, hipStream_t st);
// X_k Z_k summed per slice: part (nslices rows of K + 1 float4) from the
// pairs' rows of A; Ad: nslices x Nu x 64 floats
void narrow_pairs(const NarrowPlan& p, const NarrowMt& mt, const float2* A, int P,
                  const int* pbase, const int* pwin, const int* gb, const int* ge, int nslices,
                  float* Ad, float4* part, hipStream_t st);
// each segment's slices into its shot's row of S (rows of K + 1 float4)
void narrow_sum(const NarrowPlan& p, const NarrowMt& mt, const float4* part, const int* seg_shot,
                const int* seg_beg, const int* seg_end, int nseg, const float* seg_scale,
                float scale, float4* S, hipStream_t st);
// shot_final_rows for these sums
void narrow_final_rows(const NarrowPlan& p, const float4* S, int rows, const FinalOut& fo,
                       hipStream_t st);

// Deterministic accumulation: every term is rounded once to a signed 64-bit
// fixed-point value v * 2^E and summed with integer atomics, which are exact
// and so independent of the order in which threads and workgroups arrive.
// E is chosen from a bound M >= |component| of every term and the number of
// terms n that can reach one bin: |sum| * 2^E <= 2 n M 2^E <= 2^61.
__device__ __forceinline__ double det_scale(double n, double M) {
    if (!(M > 0.0)) return 0.0;
    int e;
    frexp(2.0 * n * M, &e);  // 2 n M < 2^e
    return ldexp(1.0, 61 - e);
}
__device__ __forceinline__ double det_unfix(unsigned long long u, double inv_scale) {
    return (double)(long long)u * inv_scale;
}

inline int next_pow2(int64_t n) {
    int p = 1;
    while (p < n) p <<= 1;
    return p;
}
inline int ilog2(int n) {
    int l = 0;
    while ((1 << l) < n) ++l;
    return l;
}
