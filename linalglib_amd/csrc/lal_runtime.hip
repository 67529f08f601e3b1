// Context, memory and elementwise utilities of the C ABI.
#include "lal_internal.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <mutex>
#include <string>

namespace lal
{
    static thread_local std::string g_last_error;

    void set_last_error(const char* msg)
    {
        g_last_error = msg;
    }

    namespace
    {
        // The process's pools, and what those of a device hold together.
        struct pool_list
        {
            std::mutex               mu;
            std::vector<chunk_pool*> pools;
            std::atomic<size_t>      held[LAL_MAX_DEVICES] = {};
        };
        pool_list& all_pools()
        {
            static pool_list* l = new pool_list; // (outlives every context)
            return *l;
        }
    }

    chunk_pool::chunk_pool(int device, size_t total)
        : device_(device), limit_(device < LAL_MAX_DEVICES ? total / 32 : 0)
    {
        std::lock_guard<std::mutex> lock(all_pools().mu);
        all_pools().pools.push_back(this);
    }

    chunk_pool::~chunk_pool()
    {
        {
            std::lock_guard<std::mutex> lock(all_pools().mu);
            auto&                       v = all_pools().pools;
            v.erase(std::remove(v.begin(), v.end(), this), v.end());
        }
        clear();
        if(notes_)
            (void)hipHostFree(notes_);
    }

    bool chunk_pool::take_note(void** host, void** dev)
    {
        std::lock_guard<std::mutex> lock(mu_);
        if(notes_ == nullptr)
        {
            void *h = nullptr, *d = nullptr;
            if(hipHostMalloc(&h, 64 * NOTES, hipHostMallocMapped | hipHostMallocCoherent) !=
               hipSuccess)
            {
                (void)hipGetLastError();
                return false;
            }
            if(hipHostGetDevicePointer(&d, h, 0) != hipSuccess)
            {
                (void)hipGetLastError();
                (void)hipHostFree(h);
                return false;
            }
            notes_     = static_cast<char*>(h);
            notes_dev_ = static_cast<char*>(d);
        }
        if(~noted_ == 0)
            return false;
        const int k = __builtin_ctzll(~noted_);
        noted_ |= 1ull << k;
        *host = notes_ + 64 * k;
        *dev  = notes_dev_ + 64 * k;
        std::memset(*host, 0, 64);
        return true;
    }

    void chunk_pool::give_note(void* host)
    {
        std::lock_guard<std::mutex> lock(mu_);
        noted_ &= ~(1ull << ((static_cast<char*>(host) - notes_) / 64));
    }

    chunk_pool::chunk chunk_pool::take(size_t want)
    {
        std::lock_guard<std::mutex> lock(mu_);
        size_t best = spare_.size();
        for(size_t k = 0; k < spare_.size(); k++)
            if(spare_[k].cap >= want && spare_[k].cap / 4 <= want &&
               (best == spare_.size() || spare_[k].cap < spare_[best].cap))
                best = k;
        if(best == spare_.size())
            return {nullptr, 0};
        const chunk k = spare_[best];
        spare_.erase(spare_.begin() + best);
        held_ -= k.cap;
        all_pools().held[device_] -= k.cap;
        return k;
    }

    void chunk_pool::give(const chunk& k)
    {
        std::lock_guard<std::mutex> lock(mu_);
        size_t                      drop = 0; // the oldest make room
        const auto                  room = [&] {
            if(k.cap > limit_)
                return false;
            std::atomic<size_t>& held = all_pools().held[device_];
            for(size_t now = held;;)
                if(now + k.cap <= limit_)
                {
                    if(held.compare_exchange_weak(now, now + k.cap))
                        return true;
                }
                else if(drop == spare_.size())
                    return false;
                else
                {
                    const chunk& old = spare_[drop++];
                    (void)hipFree(old.p);
                    held_ -= old.cap;
                    held -= old.cap;
                    now = held;
                }
        };
        const bool kept = room();
        spare_.erase(spare_.begin(), spare_.begin() + drop);
        if(kept)
        {
            spare_.push_back(k);
            held_ += k.cap;
        }
        else
            (void)hipFree(k.p);
    }

    bool chunk_pool::clear()
    {
        std::lock_guard<std::mutex> lock(mu_);
        for(const chunk& k : spare_)
            (void)hipFree(k.p);
        spare_.clear();
        const bool any = held_ > 0;
        if(any)
            all_pools().held[device_] -= held_;
        held_ = 0;
        return any;
    }

    bool chunk_pool::clear_all(int device)
    {
        std::lock_guard<std::mutex> lock(all_pools().mu);
        bool                        any = false;
        for(chunk_pool* p : all_pools().pools)
            if(p->device_ == device)
                any |= p->clear();
        return any;
    }

    void chunk_pool::close()
    {
        {
            std::lock_guard<std::mutex> lock(mu_);
            limit_ = 0;
        }
        clear();
    }

    bool chunk_pool::settle(size_t bytes)
    {
        int now = device_;
        (void)hipGetDevice(&now);
        if(now != device_)
            (void)hipSetDevice(device_);
        (void)hipDeviceSynchronize();
        size_t free = 0, total = 0;
        bool   ample = true;
        if(bytes >= LARGE)
            ample = hipMemGetInfo(&free, &total) == hipSuccess && free >= total / 8;
        if(now != device_)
            (void)hipSetDevice(now);
        return ample;
    }

    namespace
    {
        template <typename F>
        int with_room(F&& alloc, const char* what, int line)
        {
            hipError_t e   = alloc();
            int        dev = 0;
            if(e == hipErrorOutOfMemory)
            {
                (void)hipGetLastError();
                if(hipGetDevice(&dev) == hipSuccess && chunk_pool::clear_all(dev))
                    e = alloc();
            }
            if(e == hipSuccess)
                return LAL_OK;
            (void)hipGetLastError();
            return hip_status(e, what, __FILE__, line);
        }
    }

    int device_malloc(void** p, size_t bytes)
    {
        return with_room([&] { return hipMalloc(p, bytes); }, "hipMalloc", __LINE__);
    }

    int device_malloc(void** p, size_t bytes, hipStream_t stream)
    {
        return with_room([&] { return hipMallocAsync(p, bytes, stream); }, "hipMallocAsync",
                         __LINE__);
    }

    arena::~arena()
    {
        const bool keep = pool_ && !chunks_.empty() && pool_->settle(total_);
        for(chunk& k : chunks_)
            if(keep)
                pool_->give({k.p, k.cap});
            else
                (void)hipFree(k.p);
    }

    int arena::get_bytes(void** p, size_t bytes)
    {
        *p    = nullptr;
        bytes = (bytes + 255) & ~(size_t)255;
        for(; cur_ < chunks_.size(); cur_++)
        {
            chunk& k = chunks_[cur_];
            if(k.cap - k.used >= bytes)
            {
                *p = k.p + k.used;
                k.used += bytes;
                return LAL_OK;
            }
        }
        // a new chunk: half of what there is, within 1 MiB .. 512 MiB
        const size_t half = tight_ ? 0 : total_ / 2;
        size_t cap = std::max(next_, std::min(std::max(half, (size_t)1 << 20), (size_t)512 << 20));
        cap        = std::max((cap + 255) & ~(size_t)255, bytes);
        next_      = 0;
        char* q    = nullptr;
        if(pool_)
        {
            const chunk_pool::chunk k = pool_->take(cap);
            q                         = k.p;
            cap                       = q ? k.cap : cap;
        }
        if(q == nullptr && hipMalloc(&q, cap) != hipSuccess)
        {
            (void)hipGetLastError(); // no room to spare: just this array
            q   = nullptr;
            cap = bytes;
        }
        if(q == nullptr)
            LAL_TRY(device_malloc(reinterpret_cast<void**>(&q), cap));
        chunks_.push_back({q, cap, bytes});
        total_ += cap;
        *p = q;
        return LAL_OK;
    }

    arena::mark_t arena::mark() const
    {
        return {cur_, cur_ < chunks_.size() ? chunks_[cur_].used : 0};
    }

    void arena::release(const mark_t& m)
    {
        for(size_t k = m.chunk; k < chunks_.size(); k++)
            chunks_[k].used = k == m.chunk ? m.used : 0;
        cur_ = m.chunk;
    }

    int hip_status(hipError_t e, const char* what, const char* file, int line)
    {
        char buf[512];
        snprintf(buf, sizeof(buf), "%s failed: %s (%s:%d)", what, hipGetErrorString(e), file,
                 line);
        g_last_error = buf;
        if(e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation)
            return LAL_ERR_OOM;
        if(e == hipErrorNoDevice || e == hipErrorInvalidDevice)
            return LAL_ERR_NO_DEVICE;
        return LAL_ERR_HIP;
    }
}

namespace
{
    // One wavefront: n ints to mapped host memory, then the sequence number.
    // The system-scope release waits for the wave's stores before it.
    __global__ void __launch_bounds__(64)
        note_kernel(int* __restrict__ src, int n, int clear, int* note, unsigned seq)
    {
        for(int i = threadIdx.x; i < n; i += 64)
        {
            __hip_atomic_store(note + i, src[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if(clear)
                src[i] = 0;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
        if(threadIdx.x == 0)
            __hip_atomic_store(reinterpret_cast<unsigned*>(note + LAL_NOTE_INTS), seq,
                               __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

namespace lal
{
    int poll_word(lal_context* c, const unsigned* word, unsigned seq, bool* there)
    {
        // A query puts a marker into the stream, which the kernels behind it
        // then wait for: it is for a failed kernel to turn into an error instead
        // of a hang, every two milliseconds.
        using clock = std::chrono::steady_clock;
        const auto every = std::chrono::milliseconds(2);
        auto       next  = clock::now() + every;
        *there           = true;
        for(unsigned spins = 1; __atomic_load_n(word, __ATOMIC_ACQUIRE) != seq; spins++)
            if((spins & 255) == 0 && clock::now() >= next)
            {
                const hipError_t e = hipStreamQuery(c->stream);
                if(e == hipSuccess) // drained: the word is there, or never will be
                {
                    *there = __atomic_load_n(word, __ATOMIC_ACQUIRE) == seq;
                    return LAL_OK;
                }
                if(e != hipErrorNotReady)
                    LAL_HIP(e);
                next = clock::now() + every;
            }
        return LAL_OK;
    }

    int wait_note(lal_context* c, unsigned seq)
    {
        bool there = false;
        LAL_TRY(poll_word(c, reinterpret_cast<const unsigned*>(c->h_note + LAL_NOTE_INTS), seq,
                          &there));
        if(!there)
        {
            set_last_error("a result did not reach the host");
            return LAL_ERR_HIP;
        }
        return LAL_OK;
    }

    int take_note(lal_context* c, unsigned seq, int n, int* out)
    {
        LAL_TRY(wait_note(c, seq));
        for(int i = 0; i < n; i++)
            out[i] = __atomic_load_n(c->h_note + i, __ATOMIC_RELAXED);
        return LAL_OK;
    }

    int read_ints(lal_context* c, int* src, int n, int* out, bool clear)
    {
        LAL_REQUIRE(n >= 0 && n <= LAL_NOTE_INTS);
        const unsigned seq = ++c->note_seq;
        note_kernel<<<1, 64, 0, c->stream>>>(src, n, clear ? 1 : 0, c->d_note, seq);
        LAL_LAUNCHED();
        return take_note(c, seq, n, out);
    }
}

extern "C" const char* lal_last_error(void)
{
    return lal::g_last_error.c_str();
}

extern "C" const char* lal_status_string(int s)
{
    switch(s)
    {
    case LAL_OK: return "ok";
    case LAL_ERR_INVALID: return "invalid argument";
    case LAL_ERR_OOM: return "out of device memory";
    case LAL_ERR_HIP: return "HIP runtime error";
    case LAL_ERR_NOT_CONVERGED: return "not converged";
    case LAL_ERR_NAN: return "NaN in residual";
    case LAL_ERR_NO_DEVICE: return "no usable device";
    case LAL_ERR_UNSUPPORTED: return "unsupported input";
    default: return "unknown status";
    }
}

extern "C" int lal_create(lal_handle* handle)
{
    LAL_REQUIRE(handle != nullptr);
    *handle = nullptr;
    int ndev = 0;
    if(hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
    {
        lal::set_last_error("no HIP device");
        return LAL_ERR_NO_DEVICE;
    }
    lal_context* c = new lal_context;
    LAL_HIP(hipGetDevice(&c->device));
    hipDeviceProp_t prop;
    LAL_HIP(hipGetDeviceProperties(&prop, c->device));
    if(std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    {
        char buf[256];
        snprintf(buf, sizeof(buf), "device is %s, this library is built for gfx950",
                 prop.gcnArchName);
        lal::set_last_error(buf);
        delete c;
        return LAL_ERR_NO_DEVICE;
    }
    c->num_cu = prop.multiProcessorCount;
    {
        const int st = lal::noalloc_scratch_init(c->device);
        if(st != LAL_OK)
        {
            delete c;
            return st;
        }
    }
    LAL_HIP(hipStreamCreateWithFlags(&c->side, hipStreamNonBlocking));
    c->stream = c->side;
    LAL_TRY(lal::device_malloc((void**)&c->d_part, sizeof(double) * LAL_RED_BLOCKS * 2));
    LAL_TRY(lal::device_malloc((void**)&c->d_ticket, sizeof(unsigned)));
    LAL_TRY(lal::device_malloc((void**)&c->d_flag, sizeof(int) * LAL_FLAGS));
    LAL_HIP(hipHostMalloc(&c->h_slots, sizeof(double) * LAL_NUM_SLOTS, hipHostMallocDefault));
    LAL_HIP(hipHostMalloc(&c->h_note, sizeof(int) * (LAL_NOTE_INTS + 1),
                          hipHostMallocMapped | hipHostMallocCoherent));
    std::memset(c->h_note, 0, sizeof(int) * (LAL_NOTE_INTS + 1));
    LAL_HIP(hipHostGetDevicePointer((void**)&c->d_note, c->h_note, 0));
    LAL_HIP(hipMemsetAsync(c->d_ticket, 0, sizeof(unsigned), c->stream));
    LAL_HIP(hipMemsetAsync(c->d_flag, 0, sizeof(int) * LAL_FLAGS, c->stream));
    LAL_HIP(hipStreamSynchronize(c->stream));
    c->pool = std::make_shared<lal::chunk_pool>(c->device, prop.totalGlobalMem);
    *handle = c;
    return LAL_OK;
}

extern "C" int lal_destroy(lal_handle c)
{
    if(!c)
        return LAL_OK;
    (void)hipStreamSynchronize(c->stream);
    lal::detach_hierarchies(c);
    c->pool->close();
    (void)hipFree(c->d_part);
    (void)hipFree(c->d_ticket);
    (void)hipFree(c->d_flag);
    (void)hipHostFree(c->h_slots);
    (void)hipHostFree(c->h_note);
    (void)hipStreamDestroy(c->side);
    delete c;
    return LAL_OK;
}

extern "C" int lal_set_stream(lal_handle c, void* stream)
{
    LAL_REQUIRE(c != nullptr);
    LAL_HIP(hipStreamSynchronize(c->stream));
    c->stream = static_cast<hipStream_t>(stream);
    return LAL_OK;
}

extern "C" int lal_get_stream(lal_handle c, void** stream)
{
    LAL_REQUIRE(c != nullptr && stream != nullptr);
    *stream = c->stream;
    return LAL_OK;
}

extern "C" int lal_sync(lal_handle c)
{
    LAL_REQUIRE(c != nullptr);
    LAL_HIP(hipStreamSynchronize(c->stream));
    return LAL_OK;
}

extern "C" int lal_alloc(void** ptr, size_t bytes)
{
    LAL_REQUIRE(ptr != nullptr);
    *ptr = nullptr;
    if(bytes == 0)
        return LAL_OK;
    return lal::device_malloc(ptr, bytes);
}

extern "C" int lal_free(void* ptr)
{
    if(ptr)
        LAL_HIP(hipFree(ptr));
    return LAL_OK;
}

extern "C" int lal_memcpy_h2d(lal_handle c, void* dst, const void* src, size_t bytes)
{
    LAL_REQUIRE(c != nullptr);
    if(bytes == 0)
        return LAL_OK;
    LAL_REQUIRE(dst != nullptr && src != nullptr);
    LAL_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream));
    LAL_HIP(hipStreamSynchronize(c->stream));
    return LAL_OK;
}

extern "C" int lal_memcpy_d2h(lal_handle c, void* dst, const void* src, size_t bytes)
{
    LAL_REQUIRE(c != nullptr);
    if(bytes == 0)
        return LAL_OK;
    LAL_REQUIRE(dst != nullptr && src != nullptr);
    LAL_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream));
    LAL_HIP(hipStreamSynchronize(c->stream));
    return LAL_OK;
}

extern "C" int lal_memcpy_d2d(lal_handle c, void* dst, const void* src, size_t bytes)
{
    LAL_REQUIRE(c != nullptr);
    if(bytes == 0)
        return LAL_OK;
    LAL_REQUIRE(dst != nullptr && src != nullptr);
    LAL_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, c->stream));
    return LAL_OK;
}

namespace
{
    template <typename T>
    __global__ void __launch_bounds__(256) fill_kernel(T* __restrict__ x, size_t n, T v)
    {
        size_t i      = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
        size_t stride = (size_t)gridDim.x * blockDim.x;
        for(; i < n; i += stride)
            x[i] = v;
    }

    template <typename S, typename D>
    __global__ void __launch_bounds__(256)
        convert_kernel(const S* __restrict__ x, D* __restrict__ y, size_t n)
    {
        size_t i      = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
        size_t stride = (size_t)gridDim.x * blockDim.x;
        for(; i < n; i += stride)
            y[i] = static_cast<D>(x[i]);
    }

    template <typename T>
    int fill(lal_context* c, T* x, size_t n, T v)
    {
        LAL_REQUIRE(c != nullptr);
        if(n == 0)
            return LAL_OK;
        LAL_REQUIRE(x != nullptr);
        int g = lal::grid_for((long long)n, 256, 8192);
        fill_kernel<T><<<g, 256, 0, c->stream>>>(x, n, v);
        LAL_LAUNCHED();
        return LAL_OK;
    }

    template <typename S, typename D>
    int convert(lal_context* c, const S* x, D* y, size_t n)
    {
        LAL_REQUIRE(c != nullptr);
        if(n == 0)
            return LAL_OK;
        LAL_REQUIRE(x != nullptr && y != nullptr);
        int g = lal::grid_for((long long)n, 256, 8192);
        convert_kernel<S, D><<<g, 256, 0, c->stream>>>(x, y, n);
        LAL_LAUNCHED();
        return LAL_OK;
    }
}

extern "C" int lal_fill_f64(lal_handle c, double* x, size_t n, double v)
{
    return fill(c, x, n, v);
}
extern "C" int lal_fill_f32(lal_handle c, float* x, size_t n, float v)
{
    return fill(c, x, n, v);
}
extern "C" int lal_fill_i32(lal_handle c, int32_t* x, size_t n, int32_t v)
{
    return fill(c, x, n, v);
}
extern "C" int lal_fill_i64(lal_handle c, int64_t* x, size_t n, int64_t v)
{
    return fill(c, x, n, v);
}
extern "C" int lal_convert_f64_f32(lal_handle c, const double* x, float* y, size_t n)
{
    return convert(c, x, y, n);
}
extern "C" int lal_convert_f32_f64(lal_handle c, const float* x, double* y, size_t n)
{
    return convert(c, x, y, n);
}
