// Recorded calls replayed by one call: the host side of a layer whose launches take microseconds each.
//
// A layer's forward or backward is a fixed sequence of this library's calls for given sizes; only the addresses differ from
// call to call.  Made one by one from an interpreter they cost 5-10 us each, more than most of the kernels of a block of
// ordinary size take, so the GPU waits for its host.  Here the sequence is an array of words - per call the number of the
// function and its arguments, an address being the number of a buffer and an offset into it - and this file makes the
// calls.  Nothing is kept between calls.
#include <tuple>
#include <utility>

#include "mi8_common.h"

namespace mi8 {
namespace {

constexpr int64_t kStream = -1;   // the word that stands for the stream
constexpr int64_t kIgnored = -2;  // ... and for where a call writes how many slots it used, which follows from the sizes
constexpr int kOffsetBits = 48;

struct Reader {
    const int64_t* at;
    const int64_t* end;
    const void* const* buffers;
    int32_t n_buffers;
    void* stream;
    bool bad = false;
    int32_t ignored = 0;
    mi8_cast_item casts[MI8_CAST_BATCH];
    mi8_two_cast_item two_casts[MI8_CAST_BATCH];
    mi8_gemm_product products[MI8_GEMM_BATCH];

    int64_t word()
    {
        if (at >= end) {
            bad = true;
            return 0;
        }
        return *at++;
    }
    void* address()
    {
        const int64_t v = word();
        if (v == 0) return nullptr;
        if (v == kStream) return stream;
        if (v == kIgnored) return &ignored;
        const int64_t b = (v >> kOffsetBits) - 1;
        if (b < 0 || b >= n_buffers) {
            bad = true;
            return nullptr;
        }
        return (char*)const_cast<void*>(buffers[b]) + (v & (((int64_t)1 << kOffsetBits) - 1));
    }
    int items(int most)
    {
        const int64_t n = word();
        if (n < 0 || n > most) bad = true;
        return bad ? 0 : (int)n;
    }
};

template <typename T>
struct Get {
    static T from(Reader& r)
    {
        if constexpr (std::is_pointer_v<T>)
            return (T)r.address();
        else
            return (T)r.word();
    }
};
template <typename T>
void get(Reader& r, T& to) { to = Get<T>::from(r); }

template <>
struct Get<const mi8_cast_item*> {
    static const mi8_cast_item* from(Reader& r)
    {
        const int n = r.items(MI8_CAST_BATCH);
        for (int i = 0; i < n; ++i) {
            mi8_cast_item& t = r.casts[i];
            get(r, t.x), get(r, t.rows), get(r, t.cols), get(r, t.slots), get(r, t.scale_in), get(r, t.amax_ws), get(r, t.out);
            get(r, t.ld_out), get(r, t.out_t), get(r, t.ld_t), get(r, t.scale_out), get(r, t.n_slots), get(r, t.hp_dtype), get(r, t.pad_t128);
        }
        return r.casts;
    }
};
template <>
struct Get<const mi8_two_cast_item*> {
    static const mi8_two_cast_item* from(Reader& r)
    {
        const int n = r.items(MI8_CAST_BATCH);
        for (int i = 0; i < n; ++i) {
            mi8_two_cast_item& t = r.two_casts[i];
            get(r, t.x), get(r, t.rows), get(r, t.cols), get(r, t.out_rows), get(r, t.ld_rows), get(r, t.row_scale), get(r, t.out_t);
            get(r, t.ld_t), get(r, t.col_scale), get(r, t.workspace), get(r, t.group_rows), get(r, t.hp_dtype);
        }
        return r.two_casts;
    }
};
template <>
struct Get<const mi8_gemm_product*> {
    static const mi8_gemm_product* from(Reader& r)
    {
        const int n = r.items(MI8_GEMM_BATCH);
        for (int i = 0; i < n; ++i) {
            mi8_gemm_product& t = r.products[i];
            get(r, t.a), get(r, t.lda), get(r, t.b), get(r, t.ldb), get(r, t.M), get(r, t.N), get(r, t.K), get(r, t.sa), get(r, t.sb);
            get(r, t.out), get(r, t.ldc), get(r, t.sa_is_vector), get(r, t.sb_is_vector), get(r, t.out_dtype), get(r, t.add_to_previous);
        }
        return r.products;
    }
};

template <typename... A>
int call(int (*f)(A...), Reader& r)
{
    std::tuple<A...> args{Get<A>::from(r)...};  // (braces: read in order)
    if (r.bad) {
        set_error("mi8_run_plan: not a plan of this library");
        return MI8_ERR_ARG;
    }
    return std::apply(f, args);
}

struct Function {
    const char* name;
    int (*run)(Reader&);
};
#define MI8_PLANNED(f) {#f, [](Reader& r) { return call(&f, r); }}
const Function kFunctions[] = {
    MI8_PLANNED(mi8_amax_partials), MI8_PLANNED(mi8_cast_tensorwise), MI8_PLANNED(mi8_cast_tensorwise_batch),
    MI8_PLANNED(mi8_cast_rowwise), MI8_PLANNED(mi8_cast_colwise_t), MI8_PLANNED(mi8_cast_rows_and_colwise_t_batch),
    MI8_PLANNED(mi8_gemm_fp8), MI8_PLANNED(mi8_gemm_fp8_accumulate), MI8_PLANNED(mi8_gemm_fp8_splitk),
    MI8_PLANNED(mi8_gemm_fp8_splitk_accumulate), MI8_PLANNED(mi8_gemm_fp8_batch), MI8_PLANNED(mi8_gemm_fp8_swiglu),
    MI8_PLANNED(mi8_gemm_fp8_codes), MI8_PLANNED(mi8_few_rows_swiglu), MI8_PLANNED(mi8_few_rows_cast_gemm),
    MI8_PLANNED(mi8_swiglu_fwd), MI8_PLANNED(mi8_swiglu_bwd), MI8_PLANNED(mi8_swiglu_bwd_cast),
    MI8_PLANNED(mi8_swiglu_bwd_amax_from_codes), MI8_PLANNED(mi8_moe_gather_cast_rows), MI8_PLANNED(mi8_swiglu_cast_rows),
    MI8_PLANNED(mi8_grouped_gemm_fp8), MI8_PLANNED(mi8_moe_scatter),
};
#undef MI8_PLANNED
constexpr int kNumFunctions = sizeof(kFunctions) / sizeof(kFunctions[0]);

}  // namespace
}  // namespace mi8

using namespace mi8;

extern "C" int mi8_plan_function(const char* name)
{
    for (int i = 0; name && i < kNumFunctions; ++i)
        if (__builtin_strcmp(kFunctions[i].name, name) == 0) return i;
    return -1;
}

extern "C" int mi8_run_plan(const int64_t* words, int64_t n_words, const void* const* buffers, int32_t n_buffers, void* stream)
{
    MI8_REQUIRE(words && n_words >= 0 && (buffers || n_buffers == 0) && n_buffers >= 0, MI8_ERR_ARG, "mi8_run_plan: null pointer");
    Reader r{words, words + n_words, buffers, n_buffers, stream};
    while (r.at < r.end) {
        const int64_t f = r.word();
        MI8_REQUIRE(f >= 0 && f < kNumFunctions, MI8_ERR_ARG, "mi8_run_plan: not a plan of this library");
        if (int rc = kFunctions[f].run(r)) return rc;
    }
    return MI8_OK;
}
