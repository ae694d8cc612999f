// Plans GEMM batches on the host (gemm_plan, no GPU): one batch a line of stdin,
//   epi ws_bytes split_waves counters nprob, then per problem: M N K taps w_half y_pair
// (K counts the columns of A: a paired operand's hi and lo parts both), one answer a line of stdout:
//   status kernel hl2 sk splits tiles
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>

#include "kernels.h"

using namespace tsn;

int main() {
    int epi, split_waves, counters, nprob;
    unsigned long long ws;
    void *const at = (void *)(1ull << 20);   // an aligned address; nothing is read
    while (scanf("%d %llu %d %d %d", &epi, &ws, &split_waves, &counters, &nprob) == 5) {
        GemmBatch b;
        b.nprob = nprob;
        for (int i = 0; i < nprob; ++i) {
            GemmProblem &p = b.p[i];
            int M, N, K, taps, half, pair;
            if (scanf("%d %d %d %d %d %d", &M, &N, &K, &taps, &half, &pair) != 6) return 1;
            gemm_problem_init(p);
            p.A = at; p.lda = K / taps; p.amap = rowmap_dense(M); p.taps = taps; p.Kc = K / taps; p.pad = taps / 2; p.a_T = M;
            p.W = (const half_t *)at; p.w_half = half; p.ldw = half ? K / 2 : K;
            p.M = M; p.N = N; p.K = K;
            p.Y = at; p.ymap = rowmap_dense(M); p.y_pair = pair;
            p.y_f16 = epi != EPI_STORE || pair;
            const bool paired = pair || epi == EPI_SNAKE || epi == EPI_RSNAKE;
            p.ldy = (epi == EPI_SWIGLU ? N / 2 : N) * (paired ? 2 : 1);
            p.R = (float *)at; p.ldr = N; p.rmap = rowmap_dense(M); p.r_add = 1;
            p.gate = (const float *)at; p.gate_ld = N; p.gate_L = M;
            if (epi == EPI_SNAKE || epi == EPI_RSNAKE) p.snake = (const float *)at;
            if (epi == EPI_QKV) {
                p.Q = p.Kd = p.Vt = (half_t *)at; p.qn = p.kn = (const float *)at;
                p.Hq = N / 3; p.nh = N / 192; p.q_L = M; p.q_soff = 0; p.S_att = M; p.Sp = (M + 63) / 64 * 64; p.rope_len = 0;
            }
        }
        b.ws = ws ? (float *)at : nullptr;
        b.ws_bytes = ws;
        b.split_waves = split_waves;
        b.sk_cnt = counters ? (unsigned *)at : nullptr;
        b.sk_cnt_n = counters;
        const int rc = gemm_plan(b, epi, false);
        printf("%d %s %d %d %d %d\n", rc, rc ? "-" : b.kname, b.hl2, b.sk, b.p[0].splits, b.total_tiles);
        fflush(stdout);
    }
    return 0;
}
