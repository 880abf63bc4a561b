// The one upload of a described decoder's prompt call, as an array of 32-bit words: tokens, then per row its sequence and position, per segment its bounds (two orders), the last rows,
// first retention chunks, the rows asked for, the chunks, key plans.  Host code alone: nothing here needs a HIP header, so that it can be compiled and run with address checks by itself.
// Every place is an offset: the array grows while it is filled, and pointers into it do not outlive that.
#pragma once
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <vector>

struct PromptSeg { int row0, S, pos0, seq, key0; };      // first row of the call, rows, first position, cache slot, first key row

// Where the keys sit for layers of one chunk size: per sequence its cached rows of the chunk the portion goes on in, then the portion; pieces are the chunks (causal segments
// {first row, rows, place of the first row in its chunk, key row of the chunk's start}).
struct PromptKeys {
    int ring, n_pieces, longest, n_pre; size_t Mk;
    size_t row_key, row_slot, pieces, pre_key, pre_slot;
};

struct PromptUpload {
    std::vector<int32_t> words;                          // tokens first (64 bits each)
    size_t row_seq, row_pos, seg, rseg, last, snap0, want, chunks;
    std::vector<PromptKeys> keys;                        // one per distinct chunk size
    int snaps, longest;                                  // retention chunks in all, rows of the longest segment
    bool want_is_last;                                   // the rows asked for are the segments' last rows, in their order
};

inline PromptKeys prompt_keys(const std::vector<PromptSeg>& segs, int chunk, int max_tokens, std::vector<int32_t>& words) {
    PromptKeys o{};
    o.ring = std::min(chunk, max_tokens);
    std::vector<int32_t> key, slot, pieces, pk, ps;
    int base = 0;
    for (const PromptSeg& g : segs) {
        const int pre = g.pos0 % chunk, last_chunk = (g.pos0 + g.S - 1) / chunk;
        for (int i = 0; i < pre; i++) { pk.push_back(base + i); ps.push_back(g.seq * o.ring + i); }
        for (int t = 0; t < g.S; t++) {
            const int pos = g.pos0 + t;
            key.push_back(base + pre + t);
            slot.push_back(pos / chunk == last_chunk ? g.seq * o.ring + pos % chunk : -1);
        }
        for (int t = 0; t < g.S;) {
            const int at = (g.pos0 + t) % chunk, n = std::min(g.S - t, chunk - at);
            for (int32_t v : {g.row0 + t, n, at, base + pre + t - at}) pieces.push_back(v);
            o.longest = std::max(o.longest, n);
            t += n;
        }
        base += pre + g.S;
    }
    o.Mk = base; o.n_pieces = (int)pieces.size() / 4; o.n_pre = (int)pk.size();
    auto put = [&](const std::vector<int32_t>& v) { const size_t at = words.size(); words.insert(words.end(), v.begin(), v.end()); return at; };
    o.row_key = put(key); o.row_slot = put(slot); o.pieces = put(pieces); o.pre_key = put(pk); o.pre_slot = put(ps);
    return o;
}

// segs: the call's segments, rows 0 .. M in order; chunk_sizes: of attention's layers; ret_chunk: tokens of a retention chunk
inline PromptUpload prompt_upload(const std::vector<PromptSeg>& segs, int M, const int64_t* tokens, const int32_t* want, int n_want, const std::vector<int>& chunk_sizes, int max_tokens, int ret_chunk) {
    PromptUpload u{};
    const size_t n = segs.size();
    u.row_seq = 2 * (size_t)M; u.row_pos = u.row_seq + M; u.seg = u.row_pos + M; u.rseg = u.seg + 4 * n; u.last = u.rseg + 4 * n; u.snap0 = u.last + n; u.want = u.snap0 + n;
    u.chunks = u.want + n_want;
    std::vector<int32_t>& w = u.words;
    w.resize(u.chunks);
    memcpy(w.data(), tokens, (size_t)M * 8);
    u.want_is_last = n_want == (int)n;
    for (size_t i = 0; i < n; i++) {
        const PromptSeg& g = segs[i];
        for (int r = 0; r < g.S; r++) { w[u.row_seq + g.row0 + r] = g.seq; w[u.row_pos + g.row0 + r] = g.pos0 + r; }
        const int32_t b0[4] = {g.row0, g.S, g.pos0, g.key0}, b1[4] = {g.row0, g.S, g.pos0, g.seq};
        memcpy(&w[u.seg + 4 * i], b0, 16);
        memcpy(&w[u.rseg + 4 * i], b1, 16);
        w[u.last + i] = g.row0 + g.S - 1;
        w[u.snap0 + i] = u.snaps;
        u.snaps += (g.S + ret_chunk - 1) / ret_chunk;
        u.longest = std::max(u.longest, g.S);
        u.want_is_last = u.want_is_last && want[i] == g.row0 + g.S - 1;
    }
    if (n_want) memcpy(&w[u.want], want, (size_t)n_want * 4);
    for (const PromptSeg& g : segs)
        for (int t = 0; t < g.S; t += ret_chunk) { w.push_back(g.row0 + t); w.push_back(std::min(ret_chunk, g.S - t)); }
    for (int chunk : chunk_sizes) u.keys.push_back(prompt_keys(segs, chunk, max_tokens, w));
    return u;
}
