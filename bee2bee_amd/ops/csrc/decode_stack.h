// What a decode step's layers in one launch (decode_stack.hip) are told.
#pragma once

constexpr int DS_WGS = 256;                    // workgroups, a CU each
constexpr int DS_CLAIMS = DS_WGS + 8 * 32;     // words: a number's, 8 counters
constexpr int DS_STATE = 64;                   // words: progress; at 32: given up
constexpr int DS_PATIENCE = 1 << 22;           // polls, of half a microsecond or
                                               // more
constexpr int DS_LAYERS = 31;                  // of a launch: arguments of 4 KB
constexpr int DS_LAYER_NORM = 1024;            // layer norm: columns at most
constexpr int DS_ROWS = 8;
constexpr int DS_SPLITS = 32;                  // of a context, at most

// products of a layer
enum { DS_QKV = 0, DS_O = 1, DS_UP = 2, DS_DOWN = 3 };

struct StackLayer {
    const unsigned short* w[4];     // [rows, K]
    const unsigned short* bias[4];  // or null
    const unsigned short* norm[2];  // before q|k|v, before the feed-forward
    const unsigned short* norm_bias[2];
    void* k_cache;                  // [nb, nkv, bs, hd]
    void* v_cache;
};

struct StackHead {
    int K[4], octets[4];            // of the products; octets of 8 rows of w
    int half[4];                    // rows of w from an octet's first 4 to its
                                    // other 4
    int lo, hi, all;                // layers of this launch, of the stack
    int M, gelu, streamed;          // streamed: weights and pages past L2
    int nq, nkv, G, bs, W, Z;       // G: nq / nkv; W: pages a sequence; Z: splits
    int items;                      // M * nkv * Z
    float eps, scale;
    // words that pass between workgroups: [layers] of `stride`, and in each
    int stride, new_kv, att, o, up, down;    // (queries at 0)
    int turns, pages, area;         // in LDS (launch_decode_stack)
    int turn_rows;                  // of cos_t and sin_t
    int patience;                   // 2^n - 1: a wait looks for progress every 2^n
                                    // polls, and is given up if there is none
    unsigned* words;
    unsigned* parts;                // [M * nkv, Z, G, hd / 16, 18]
    unsigned* claims;               // [DS_CLAIMS]
    unsigned* state;                // [DS_STATE]
    int* status;                    // on the host: 1 if a wait was given up; null
    const unsigned short* x;        // [M, H] bf16: the first layer's input
    float* x32;                     // [M, H]: the residual between
    unsigned* out;                  // [M, H] bf16: the last layer's result
    const int* pos;
    const float* cos_t;             // [turn_rows, hd / 2]; null: no rotation
    const float* sin_t;
    const int* slots;               // null: where the table has the positions
    const int* table;               // [M, W]
    const int* seq_lens;
};
struct StackArgs : StackHead {
    StackLayer layer[DS_LAYERS + 1];         // and the next launch's first
};
static_assert(sizeof(StackArgs) <= 4096, "kernel arguments");
