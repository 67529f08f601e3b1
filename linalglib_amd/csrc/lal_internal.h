// Internal helpers shared by the gfx950 kernels and the C ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <memory>
#include <mutex>
#include <vector>

#include "../../include/lal.h"

// Deterministic two-stage reductions use a fixed grid of this many blocks.
#define LAL_RED_BLOCKS 1024
#define LAL_RED_THREADS 256
// Pinned scalars in the context (solver flags and norms).
#define LAL_NUM_SLOTS 64

struct lal_hierarchy_t;

namespace lal
{
    // Chunks of device memory that a context's arenas have given back, for its
    // next ones.  The driver takes freed memory back at a bounded rate: programs
    // that build hierarchies one after the other (121^3: 2.9 GB each) run dry
    // after about a second and then wait for it, in steps of 10 ms (500 builds
    // took 78 ms each on average, of which 12.5 are work; now 11.2).  At most 1/32
    // of the device's memory in all contexts' pools together; given back with the
    // context, and by every pool of the device when an allocation of this library
    // fails (device_malloc); nothing large is taken in while less than an eighth
    // of the device's memory is free.
    struct chunk_pool
    {
        struct chunk
        {
            char*  p;
            size_t cap;
        };
        chunk_pool(int device, size_t total);
        ~chunk_pool();
        chunk_pool(const chunk_pool&) = delete;
        chunk_pool& operator=(const chunk_pool&) = delete;
        // a chunk of `want` bytes or up to four times as many; cap 0: none
        chunk take(size_t want);
        // after every kernel that uses it has ended (any thread)
        void give(const chunk& k);
        // true: something went back to the driver
        bool clear();
        void close(); // the context is gone: what is given from now on is freed
        // Waits for the device's work, as a hipFree would; false: the `bytes` to
        // be given are better freed, the device is short of memory.
        bool settle(size_t bytes);
        // 64 bytes of zeroed mapped host memory (a solver's note); false: none left
        bool take_note(void** host, void** dev);
        void give_note(void* host);
        // clear() for every pool of the device
        static bool clear_all(int device);

    private:
        static constexpr int NOTES = 64;
        // arenas of less are given without a look at the device's free memory
        // (5 us; the build of a 25^3 hierarchy takes 1.7 ms)
        static constexpr size_t LARGE = (size_t)64 << 20;
        std::mutex           mu_;
        std::vector<chunk>   spare_; // oldest first
        size_t               held_ = 0;
        int                  device_;
        size_t               limit_; // of all the device's pools together
        char *               notes_ = nullptr, *notes_dev_ = nullptr;
        unsigned long long   noted_ = 0; // a bit per note in use
    };

    // hipMalloc, and hipMallocAsync on a stream; when the device is out of
    // memory, its pools are emptied and the allocation is tried once more.
    int device_malloc(void** p, size_t bytes);
    int device_malloc(void** p, size_t bytes, hipStream_t stream);

    // Device memory handed out from a few large allocations and freed with
    // the object, or kept by the pool it uses.  A hierarchy build makes several
    // hundred arrays; one hipMalloc and hipFree each cost more than the build's
    // kernels.
    struct arena
    {
        struct mark_t
        {
            size_t chunk = 0, used = 0;
        };
        arena() = default;
        arena(const arena&) = delete;
        arena& operator=(const arena&) = delete;
        ~arena();
        void use(const std::shared_ptr<chunk_pool>& pool)
        {
            pool_ = pool;
        }
        // `first` bytes for the first allocation (rounded up as needed)
        void reserve(size_t first)
        {
            next_ = first;
        }
        // no allocation beyond what is asked for (of 1 MiB at least)
        void tight()
        {
            tight_ = true;
        }
        int get_bytes(void** p, size_t bytes);
        template <typename T>
        int get(T** p, size_t n)
        {
            return get_bytes(reinterpret_cast<void**>(p), sizeof(T) * (n > 0 ? n : 1));
        }
        // release(mark()) gives back what was taken since, for later work on
        // the same stream
        mark_t mark() const;
        void   release(const mark_t& m);

    private:
        struct chunk
        {
            char*  p;
            size_t cap, used;
        };
        std::vector<chunk>          chunks_;
        size_t                      cur_ = 0, next_ = 0, total_ = 0;
        bool                        tight_ = false;
        std::shared_ptr<chunk_pool> pool_;
    };
}

// Flag words of a context, and integers one read_ints hands back at most.
#define LAL_FLAGS 32
#define LAL_NOTE_INTS 192

// Devices the per-device static scratch table covers.
#define LAL_MAX_DEVICES 64

struct lal_context
{
    hipStream_t stream     = nullptr; // where the work goes: `side` or the caller's
    hipStream_t side       = nullptr; // the context's own, non-blocking; graphs are
                                      // captured on it
    int         device     = 0;
    int         num_cu     = 0;
    // reduction workspace: partials and the ticket of the block that adds them up
    double*   d_part   = nullptr; // LAL_RED_BLOCKS * 2
    unsigned* d_ticket = nullptr;
    double*   h_slots  = nullptr; // LAL_NUM_SLOTS pinned scalars
    // flag words of the checks and setup passes: zero between calls (whoever
    // raises one reads it back with read_ints, which clears it)
    int*      d_flag   = nullptr;
    // small results reach the host through mapped pinned memory: LAL_NOTE_INTS
    // values and, after them, a sequence number that the host polls
    int*      h_note   = nullptr;
    int*      d_note   = nullptr;
    unsigned  note_seq = 0;
    std::shared_ptr<lal::chunk_pool> pool;
    // hierarchies built on this context: lal_destroy detaches them, so that
    // one destroyed after its context no longer touches it
    std::vector<lal_hierarchy_t*> hierarchies;
};

namespace lal
{
    int  hip_status(hipError_t e, const char* what, const char* file, int line);
    void set_last_error(const char* msg);
}

#define LAL_HIP(call)                                                                  \
    do                                                                                 \
    {                                                                                  \
        hipError_t lal_e_ = (call);                                                    \
        if(lal_e_ != hipSuccess)                                                       \
            return lal::hip_status(lal_e_, #call, __FILE__, __LINE__);                 \
    } while(0)

#define LAL_LAUNCHED()                                                                 \
    do                                                                                 \
    {                                                                                  \
        hipError_t lal_e_ = hipGetLastError();                                         \
        if(lal_e_ != hipSuccess)                                                       \
            return lal::hip_status(lal_e_, "kernel launch", __FILE__, __LINE__);       \
    } while(0)

#define LAL_TRY(...)                                                                   \
    do                                                                                 \
    {                                                                                  \
        int lal_s_ = (__VA_ARGS__);                                                    \
        if(lal_s_ != LAL_OK)                                                           \
            return lal_s_;                                                             \
    } while(0)

#define LAL_REQUIRE(cond)                                                              \
    do                                                                                 \
    {                                                                                  \
        if(!(cond))                                                                    \
        {                                                                              \
            lal::set_last_error("invalid argument: " #cond);                           \
            return LAL_ERR_INVALID;                                                    \
        }                                                                              \
    } while(0)

namespace lal
{
    inline int grid_for(long long n, int threads, int cap = 1 << 30)
    {
        long long g = (n + threads - 1) / threads;
        if(g < 1)
            g = 1;
        if(g > cap)
            g = cap;
        return (int)g;
    }

    // Blocks are dispatched round-robin over the 8 XCDs of an MI355X (block b
    // runs on XCD b % 8).  This maps the blocks of one XCD onto one
    // contiguous range of logical tiles so that neighbouring rows (and the x
    // entries they share) stay in that XCD's L2.
    __device__ __forceinline__ int xcd_tile(int bid, int nb)
    {
        const int nx  = 8;
        int       per = nb / nx;
        int       rem = nb % nx;
        int       x   = bid % nx;
        int       k   = bid / nx;
        return x * per + (x < rem ? x : rem) + k;
    }

    // By a whole wavefront: lane i < n's v into the note, then its sequence
    // number.  The system-scope release waits for the wave's stores before it.
    __device__ __forceinline__ void put_note(int* note, int n, int v, unsigned seq)
    {
        const int lane = (int)threadIdx.x & 63;
        if(lane < n)
            __hip_atomic_store(note + lane, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
        if(lane == 0)
            __hip_atomic_store(reinterpret_cast<unsigned*>(note + LAL_NOTE_INTS), seq,
                               __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }

    // v + the value of v in another lane of the same quad, half row or row
    // (DPP control CTRL: quad_perm, row_half_mirror 0x141, row_mirror 0x140).
    template <int CTRL>
    __device__ __forceinline__ double dpp_add(double v)
    {
        const long long b  = __builtin_bit_cast(long long, v);
        const int       lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, false);
        const int       hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, false);
        return v + __builtin_bit_cast(double, (long long)(unsigned)lo | ((long long)hi << 32));
    }
    template <int CTRL>
    __device__ __forceinline__ float dpp_add(float v)
    {
        const int o = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false);
        return v + __builtin_bit_cast(float, o);
    }

    // v of the partner lane in step STEP of a reduction over an aligned lane
    // group: lane ^ 1, lane ^ 2, the half row's mirror image, the row's.  (A DPP
    // move is an instruction or two; the shuffles they stand for go through LDS.)
    template <int STEP>
    __device__ __forceinline__ int partner(int v)
    {
        constexpr int CTRL = STEP == 0 ? 0xB1 : STEP == 1 ? 0x4E : STEP == 2 ? 0x141 : 0x140;
        return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
    }

    // Reduction of an int over aligned groups of G = 8, 16 or 64 lanes, left in
    // every lane; f is commutative, associative and f(a, a) = a.
    template <int G, typename F>
    __device__ __forceinline__ int group_fold(int v, F f)
    {
        v = f(v, partner<0>(v));
        v = f(v, partner<1>(v));
        v = f(v, partner<2>(v));
        if(G >= 16)
            v = f(v, partner<3>(v));
        if(G == 64)
            v = f(f(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
                  f(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
        return v;
    }

    // Sum over aligned groups of LANES (a power of two <= 64) lanes, left in
    // every lane of the group: lane ^ 1 and lane ^ 2 (quad permutations), the
    // half-row and row mirrors (each adds the other half's partial sum), then
    // exchanges with the lanes 16 and 32 away.
    template <int LANES, typename T>
    __device__ __forceinline__ T lane_sum(T v)
    {
        if(LANES >= 2)
            v = dpp_add<0xB1>(v); // quad_perm [1, 0, 3, 2]
        if(LANES >= 4)
            v = dpp_add<0x4E>(v); // quad_perm [2, 3, 0, 1]
        if(LANES >= 8)
            v = dpp_add<0x141>(v);
        if(LANES >= 16)
            v = dpp_add<0x140>(v);
        if(LANES >= 32)
            v += __shfl_xor(v, 16, 64);
        if(LANES >= 64)
            v += __shfl_xor(v, 32, 64);
        return v;
    }

    template <typename T>
    __device__ __forceinline__ T wave_sum(T v)
    {
#pragma unroll
        for(int o = 32; o > 0; o >>= 1)
            v += __shfl_xor(v, o, 64);
        return v;
    }

    template <typename T>
    __device__ __forceinline__ T wave_max(T v)
    {
#pragma unroll
        for(int o = 32; o > 0; o >>= 1)
        {
            T w = __shfl_xor(v, o, 64);
            v   = (w < v) ? v : w;
        }
        return v;
    }

    // v of lane t (the same t in every lane of the wavefront)
    __device__ __forceinline__ int wave_lane(int v, int t)
    {
        return __builtin_amdgcn_readlane(v, t);
    }
    __device__ __forceinline__ double wave_lane(double v, int t)
    {
        const long long b  = __builtin_bit_cast(long long, v);
        const unsigned  lo = (unsigned)__builtin_amdgcn_readlane((int)b, t);
        const unsigned  hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), t);
        return __builtin_bit_cast(double, (long long)(((unsigned long long)hi << 32) | lo));
    }

    // Workgroup barrier that orders LDS accesses only: global loads issued
    // before it stay in flight (__syncthreads() waits for them).
    __device__ __forceinline__ void lds_barrier()
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    }

    // Wavefront maximum that returns NaN when any lane holds one.
    template <typename T>
    __device__ __forceinline__ T wave_max_nan(T v)
    {
#pragma unroll
        for(int o = 32; o > 0; o >>= 1)
        {
            T w = __shfl_xor(v, o, 64);
            v   = (v != v || w < v) ? v : w;
        }
        return v;
    }

    // Temporary device arrays of one call: from `a` when given (marked and
    // released by whoever owns it), else stream-ordered allocations freed at
    // the end of the scope.
    struct temps
    {
        temps(lal_context* c, arena* a) : c_(c), a_(a) {}
        temps(const temps&) = delete;
        ~temps()
        {
            for(void* p : own_)
                (void)hipFreeAsync(p, c_->stream);
        }
        template <typename T>
        int get(T** p, size_t n)
        {
            if(a_)
                return a_->get(p, n);
            *p = nullptr;
            LAL_TRY(device_malloc(reinterpret_cast<void**>(p), sizeof(T) * (n > 0 ? n : 1),
                                  c_->stream));
            own_.push_back(*p);
            return LAL_OK;
        }

    private:
        lal_context*       c_;
        arena*             a_;
        std::vector<void*> own_;
    };

    // Internal launchers shared across translation units (device-resident
    // results; nothing is copied to the host).
    int dot_f64_dev(lal_context* c, int n, const double* x, const double* y, double* d_out,
                    int slot);
    int dot_f32_dev(lal_context* c, int n, const float* x, const float* y, double* d_out,
                    int slot);
    int norm_inf_f64_dev(lal_context* c, int n, const double* x, double* d_out, int slot);
    int scan_i32_dev(lal_context* c, int n, int32_t* x, arena* a = nullptr);
    int scan_i64_dev(lal_context* c, int n, int64_t* x, arena* a = nullptr);
    // Device address of the allocation-free scan's static scratch for
    // `device` (which must be current), looked up once per device.
    int noalloc_scratch_init(int device);
    // Polls a mapped host word until it is `seq`; *there false: the stream has
    // drained without it.
    int poll_word(lal_context* c, const unsigned* word, unsigned seq, bool* there);
    // Blocks until the context's note carries `seq`.
    int wait_note(lal_context* c, unsigned seq);
    // The first n ints of the note carrying `seq` (blocks), for a kernel that
    // was handed c->d_note and ++c->note_seq (put_note).
    int take_note(lal_context* c, unsigned seq, int n, int* out);
    // The n ints at src once the stream has come to them (blocks); clear: they
    // are zeroed behind the read.
    int read_ints(lal_context* c, int* src, int n, int* out, bool clear);
    // Clears the context pointer of every hierarchy built on c (lal_destroy).
    void detach_hierarchies(lal_context* c);
    // Sets *flag (on the device) unless every ci[0..nnz) lies in [0, n).
    int raise_bad_columns(lal_context* c, int nnz, int n, const int* ci, int* flag);
}
