// A graph's launches as one call from the host language.
//
// Through a foreign-function interface a launch costs the conversion of its 7 to 25 arguments, most of the host's time for a graph of small
// launches. Here the arguments of all of them stand in one array of 64-bit words, converted once; a call copies it, writes the addresses
// of the caller's arrays where they belong, and issues the launches one after the other. Nothing is kept between calls here: any number of
// threads may run the same array at once. The launches themselves may overlap on the GPU only where the graph has no intermediate array, of
// which a compiled graph keeps one for all of its calls.
// Bound by the runtime's launches, 3 us each. A call of an encoder layer over 16 tokens (seven launches) 51 -> 45 us, of a dense classifier
// (four) 30.3 -> 26.6, of one quantised layer 15.3 -> 14.5; the host's part of an image classifier of 15 launches 118 -> 98.
#include "common.h"

#include <stdlib.h>
#include <string.h>

#include <type_traits>
#include <utility>

namespace mi355x {
namespace {

template <class T>
T from_word(int64_t word) {
    if constexpr (std::is_pointer_v<T>) {
        return reinterpret_cast<T>(word);
    } else if constexpr (std::is_same_v<T, float>) {
        const uint32_t bits = (uint32_t)word;
        float value;
        memcpy(&value, &bits, sizeof(value));
        return value;
    } else {
        return static_cast<T>(word);
    }
}

// A function of the interface whose last argument is the stream, called with its other arguments from an array of words.
template <auto F>
struct Call;
template <class... A, int (*F)(A...)>
struct Call<F> {
    static constexpr int words = sizeof...(A) - 1;
    template <size_t... I>
    static int unpack(const int64_t* word, void* stream, std::index_sequence<I...>) {
        const auto argument = [&](auto index, auto* type) {
            using T = std::remove_pointer_t<decltype(type)>;
            if constexpr (decltype(index)::value == words) return static_cast<T>(stream);
            else return from_word<T>(word[decltype(index)::value]);
        };
        return F(argument(std::integral_constant<int, (int)I>{}, static_cast<A*>(nullptr))...);
    }
    static int run(const int64_t* word, void* stream) { return unpack(word, stream, std::make_index_sequence<sizeof...(A)>{}); }
};

struct Function {
    const char* name;
    int words;
    int (*run)(const int64_t*, void*);
};
#define MI355X_FUNCTION(name) {#name, Call<&name>::words, &Call<&name>::run}
constexpr Function kFunctions[] = {
    MI355X_FUNCTION(mi355x_gemm_f32), MI355X_FUNCTION(mi355x_gemm_packed_f32), MI355X_FUNCTION(mi355x_conv2d_f32),
    MI355X_FUNCTION(mi355x_conv2d_res_f32), MI355X_FUNCTION(mi355x_pack_conv_f32), MI355X_FUNCTION(mi355x_pack_conv_pool_f32),
    MI355X_FUNCTION(mi355x_conv2d_packed_f32), MI355X_FUNCTION(mi355x_conv2d_pool_packed_f32), MI355X_FUNCTION(mi355x_conv2d_skip_f32), MI355X_FUNCTION(mi355x_conv2d_parts_f32), MI355X_FUNCTION(mi355x_matmul_integer),
    MI355X_FUNCTION(mi355x_matmul_integer_i8), MI355X_FUNCTION(mi355x_softmax_f32), MI355X_FUNCTION(mi355x_log_softmax_f32), MI355X_FUNCTION(mi355x_softmax_max_f32),
    MI355X_FUNCTION(mi355x_attention_f32), MI355X_FUNCTION(mi355x_attention_masked_f32), MI355X_FUNCTION(mi355x_layernorm_f32), MI355X_FUNCTION(mi355x_layernorm_parts_f32), MI355X_FUNCTION(mi355x_gemm_parts_f32), MI355X_FUNCTION(mi355x_gemm_softmax_f32),
    MI355X_FUNCTION(mi355x_reduce_mean_f32), MI355X_FUNCTION(mi355x_reduce_f32), MI355X_FUNCTION(mi355x_reduce_nd_f32),
    MI355X_FUNCTION(mi355x_maxpool2d_f32), MI355X_FUNCTION(mi355x_batchnorm_f32), MI355X_FUNCTION(mi355x_eltwise_f32),
    MI355X_FUNCTION(mi355x_eltwise_program_f32), MI355X_FUNCTION(mi355x_permute_b32), MI355X_FUNCTION(mi355x_cast)};
#undef MI355X_FUNCTION
constexpr int kNumFunctions = sizeof(kFunctions) / sizeof(kFunctions[0]);

}  // namespace
}  // namespace mi355x

extern "C" int mi355x_program_function(const char* name) {
    using namespace mi355x;
    for (int i = 0; name && i < kNumFunctions; ++i)
        if (strcmp(name, kFunctions[i].name) == 0) return i;
    return -1;
}

extern "C" int64_t mi355x_program_run(const int64_t* program, int64_t words, int64_t calls, const int64_t* patches, int64_t num_patches,
                                      const int64_t* addresses, void* stream) {
    using namespace mi355x;
    constexpr int64_t ON_STACK = 2048;   // words: 80 launches of 25 arguments
    int64_t local[ON_STACK];
    int64_t* copy = local;
    if ((words && !program) || words < 0 || calls < 0 || num_patches < 0 || (num_patches && !patches))
        return set_error(MI355X_ERR_INVALID_ARGUMENT, "program: null pointer or negative size");
    if (words > ON_STACK && !(copy = static_cast<int64_t*>(malloc((size_t)words * sizeof(int64_t)))))
        return set_error(MI355X_ERR_INVALID_ARGUMENT, "program: no memory for %lld words", (long long)words);
    if (words) memcpy(copy, program, (size_t)words * sizeof(int64_t));
    int64_t result = MI355X_OK;
    for (int64_t i = 0; i < num_patches && result == MI355X_OK; ++i) {
        const int64_t slot = patches[3 * i], source = patches[3 * i + 1], offset = patches[3 * i + 2];
        if (slot < 0 || slot >= words || (source < 0 ? offset < 0 || offset >= words : !addresses))
            result = set_error(MI355X_ERR_INVALID_ARGUMENT, "program: patch %lld is outside the program", (long long)i);
        else
            copy[slot] = source < 0 ? (int64_t)reinterpret_cast<uintptr_t>(copy + offset) : addresses[source] + offset;
    }
    for (int64_t call = 0, at = 0; call < calls && result == MI355X_OK; ++call) {
        if (at >= words || copy[at] < 0 || copy[at] >= kNumFunctions || at + kFunctions[copy[at]].words >= words) {
            result = set_error(MI355X_ERR_INVALID_ARGUMENT, "program: call %lld is no function with all its arguments", (long long)call);
            break;
        }
        const Function& f = kFunctions[copy[at]];
        const int status = f.run(copy + at + 1, stream);
        if (status != MI355X_OK) result = (call << 8) | status;
        at += 1 + f.words;
    }
    if (copy != local) free(copy);
    return result;
}
