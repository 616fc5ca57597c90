// CPU check of the decode split plan (api.hip: decode_plan), over batches of sequences of up to 256 keys.
#include "../../dooms_amd/csrc/api.hip"

#include <vector>

int main() {
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
    return 0;
}
