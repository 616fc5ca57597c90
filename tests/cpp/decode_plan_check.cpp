// CPU check of the decode split plan (api.hip: decode_plan), over batches of sequences of up to 256 keys, and of the order
// of a launch's sequences (decode_order).
#include "../../dooms_amd/csrc/api.hip"

#include <cstdlib>
#include <numeric>
#include <random>
#include <vector>

static int allocations = 0;
void * operator new(size_t n) {
    allocations++;
    return std::malloc(n);
}
void * operator new(size_t n, const std::nothrow_t &) noexcept { return operator new(n); }
void operator delete(void * p) noexcept { std::free(p); }
void operator delete(void * p, size_t) noexcept { std::free(p); }

// The longest first, equal lengths as they come, and nothing taken from the heap; on the XCD-mapped grid as they come.
static bool order_ok(const std::vector<int32_t> & lens, bool xcd) {
    std::vector<int> want(lens.size());
    std::iota(want.begin(), want.end(), 0);
    if (!xcd) std::stable_sort(want.begin(), want.end(), [&](int a, int b) { return lens[a] > lens[b]; });
    int got[mx::kMaxSeqPerLaunch];
    const int before = allocations;
    decode_order(lens.data(), (int)lens.size(), xcd, got);
    return allocations == before && std::equal(want.begin(), want.end(), got);
}

int main() {
    std::mt19937 rng(1);
    for (int t = 0; t < 4000; t++) {
        std::vector<int32_t> lens(1 + rng() % mx::kMaxSeqPerLaunch);
        for (int32_t & n : lens) n = 1 + rng() % (t % 2 ? 9000 : 5);
        if (!order_ok(lens, t % 4 >= 2)) {
            std::printf("the order of %zu sequences\n", lens.size());
            return 1;
        }
    }
    // Whole sequences run on workgroups of 8 waves, of which a CU holds one on f32 rows (two waves per SIMD): at head dim 64
    // they are taken only where every workgroup has a CU of its own, else a second round costs more than the merge. Where
    // splits of 128 keys pass the workgroup cap, the sequences are whole on 4 waves.
    for (int heads = 1; heads <= 48; heads++)
        for (int n_seq = 1; n_seq <= mx::kMaxSeqPerLaunch; n_seq++)
            for (int len : {129, 160, 256})
                for (bool f32 : {false, true}) {
                    mx_attn_desc d{};
                    d.n_head = d.n_head_kv = heads;
                    d.head_dim = 64;
                    d.n_q = 1;
                    const std::vector<int32_t> lens(n_seq, len);
                    const DecodePlan plan = decode_plan(d, lens.data(), n_seq, DecodeShape{1, 4, 1}, f32);
                    const bool capped = 2 * heads * n_seq > workgroup_cap(nullptr);
                    const bool whole = !capped && (!f32 || heads * n_seq <= 256);
                    if (plan.chunk != (whole || capped ? 256 : 128) || plan.waves != (whole ? 8 : 4)) {
                        std::printf("%d sequences of %d keys, %d heads, f32 %d: %lld keys per split, %d waves\n", n_seq, len, heads, f32,
                                    (long long)plan.chunk, plan.waves);
                        return 1;
                    }
                }
    // f32 rows of head dim 64 take 16 splits of 8 waves up to one workgroup per CU, in a ragged batch up to half of that
    for (int n_seq = 2; n_seq <= mx::kMaxSeqPerLaunch; n_seq++)
        for (int heads : {1, 2, 3, 4, 8, 20})
            for (int last : {4000, 1700}) {
                mx_attn_desc d{};
                d.n_head = d.n_head_kv = heads;
                d.head_dim = 64;
                d.n_q = 1;
                std::vector<int32_t> lens(n_seq, 4000);
                lens.back() = last;
                const DecodePlan plan = decode_plan(d, lens.data(), n_seq, DecodeShape{1, 4, 1}, true);
                const int wgs = heads * ((n_seq - 1) * 16 + (last + 255) / 256);
                if (wgs <= 512 && plan.waves != (wgs <= (last == 4000 ? 256 : 128) ? 8 : 4)) {
                    std::printf("%d sequences of 4000 and %d keys, %d heads: %lld keys per split, %d waves\n", n_seq, last, heads,
                                (long long)plan.chunk, plan.waves);
                    return 1;
                }
            }
    return 0;
}
