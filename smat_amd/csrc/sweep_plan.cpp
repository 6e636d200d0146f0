// Builds the op streams of the sweep kernel.  Layout of an op: spmm_kernels.h (SweepOp).
#include "sweep_plan.h"

#include <algorithm>
#include <climits>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <queue>
#include <stdexcept>
#include <utility>

#include "../../include/smat.h"
#include "errors.h"
#include "sweep_format.h"

namespace smat {

namespace {
constexpr int G = SWEEP_G, RW = SWEEP_RW, WAVES = SWEEP_WAVES, S = SWEEP_S, MIN_OPS = SWEEP_MIN_OPS;
constexpr int AHEAD = SWEEP_AHEAD, COPIES = SWEEP_COPIES;
constexpr int VM_MARK = MIN_OPS; // a chunk boundary waits until at most this many vector memory operations are under way
// Eight counters of 16 bits, by the compiler's vector types: a register wherever the host has one of 128 bits.
typedef int16_t Counters __attribute__((vector_size(16)));
inline Counters smaller(Counters a, Counters b) { return a < b ? a : b; }
inline Counters larger(Counters a, Counters b) { return a > b ? a : b; }

// Sum of the cheapest caps of the periods (see build_sweep_plan) for the assignment win, n periods, with rows ri of wavefront wi
// and rj of wavefront wj changed over (ri NULL: none); LONG_MAX as soon as it cannot be below `below`.  The eight wavefronts are the
// eight 16-bit lanes of a register: a plan tries thousands of such changes a row group and this is nearly all of its time
// (a plan of 8192^2, 10 %: 15.4 ms with counters of 32 bits one by one, 7.8 ms so; 35696 x 2832, 7 nonzeros a row 31.6 and 15.6).
long sum_of_caps(const int16_t *win, size_t n, const int16_t *ri, const int16_t *rj, int wi, int wj, long below, int32_t *caps_out)
{
    static_assert(WAVES == 8 && RW * 3 * S < 32768, "a wavefront's ops of three chunks, in a lane of 16 bits");
    const Counters zero = {0, 0, 0, 0, 0, 0, 0, 0}, halves = {4, 5, 6, 7, 0, 1, 2, 3}, pairs = {2, 3, 0, 1, 6, 7, 4, 5}, ones = {1, 0, 3, 2, 5, 4, 7, 6};
    Counters sign = zero;
    if (ri) sign[wi] = -1, sign[wj] = 1;
    Counters due = zero, next = zero; // pending ops with deadline p - at the start of period p - and p + 1
    long sum = 0, rest = (long)n * MIN_OPS; // what the periods to come cost at least
    for (size_t p = 0; p < n; p++) {
        Counters c[3];
        for (size_t len = 0; len < 3; len++) {
            const size_t x = p * 3 + len;
            memcpy(&c[len], win + x * WAVES, sizeof(Counters));
            if (ri) c[len] += sign * (int16_t)(ri[x] - rj[x]);
        }
        const Counters p0 = due + c[0], p1 = next + c[1], p2 = c[2];
        Counters cap = larger(p0, __builtin_shuffle(p0, halves)); // the largest of the eight, in all of them
        cap = larger(cap, __builtin_shuffle(cap, pairs));
        cap = larger(cap, __builtin_shuffle(cap, ones));
        cap = larger(cap, zero + (int16_t)MIN_OPS);
        const int32_t cap_p = cap[0];
        sum += cap_p;
        rest -= MIN_OPS;
        if (sum + rest >= below) return LONG_MAX;
        if (caps_out) caps_out[p] = cap_p;
        // the ops due now run; what is left of the cap goes to the next deadlines, but the last pending op stays for the next
        // period when it may (see the schedule in build_sweep_plan)
        Counters room = cap - p0;
        if (p + 1 < n) {
            const Counters pending = p1 + p2;
            room = (pending > zero) & (pending <= room) ? pending - (int16_t)1 : room;
        }
        const Counters r1 = smaller(room, p1);
        due = p1 - r1;
        next = p2 - smaller(room - r1, p2);
    }
    return sum;
}
} // namespace

void build_sweep_plan(const int32_t *row_ptr, const int32_t *col_idx, size_t mb, size_t kb, SweepPlanHost &out,
                      const int32_t *rows, size_t n_rows, size_t group_rows, double search, bool light)
{
    const int32_t lead = light ? 0 : 1; // chunks past the one being swept that an op may use
    if (!rows) n_rows = mb;
    const size_t GR = std::min<size_t>(std::max<size_t>(group_rows, 1), G); // block rows that share a group's 64 places
    const size_t n_rg = (n_rows + GR - 1) / GR;
    // Row groups: GR block rows of the list each, in list order - unless that leaves one group with far more blocks
    // than the average.  A workgroup multiplies one row group under several panels, so the launch takes as long as
    // the heaviest group; then the rows are dealt out instead: in descending block count, each to the group with the
    // fewest blocks so far that still has room (the group sizes stay what they were).  Which rows share a group
    // matters for nothing else: the rows of C are found through row_map, and a matrix dense enough for this kernel
    // touches every K chunk from any 64 of its rows.
    std::vector<int32_t> order;
    {
        std::vector<int64_t> blocks_of(n_rg, 0);
        int64_t total = 0, heaviest = 0;
        for (size_t i = 0; i < n_rows; i++) {
            const size_t br = rows ? (size_t)rows[i] : i;
            blocks_of[i / GR] += row_ptr[br + 1] - row_ptr[br];
        }
        for (size_t rg = 0; rg < n_rg; rg++) total += blocks_of[rg], heaviest = std::max(heaviest, blocks_of[rg]);
        if (n_rg > 1 && (double)heaviest * (double)n_rows > 1.08 * (double)total * (double)GR) {
            std::vector<int32_t> by_count(n_rows);
            for (size_t i = 0; i < n_rows; i++) by_count[i] = rows ? rows[i] : (int32_t)i;
            std::stable_sort(by_count.begin(), by_count.end(), [&](int32_t x, int32_t y) {
                return row_ptr[x + 1] - row_ptr[x] > row_ptr[y + 1] - row_ptr[y];
            });
            std::vector<std::vector<int32_t>> members(n_rg);
            typedef std::pair<int64_t, size_t> Load; // blocks so far, row group
            std::priority_queue<Load, std::vector<Load>, std::greater<Load>> lightest;
            for (size_t rg = 0; rg < n_rg; rg++) lightest.push(Load(0, rg));
            for (int32_t br : by_count) {
                const Load l = lightest.top();
                lightest.pop();
                const size_t rg = l.second;
                members[rg].push_back(br);
                if (members[rg].size() < std::min(n_rows, (rg + 1) * GR) - rg * GR)
                    lightest.push(Load(l.first + (row_ptr[br + 1] - row_ptr[br]), rg));
            }
            order.reserve(n_rows);
            for (size_t rg = 0; rg < n_rg; rg++) {
                std::sort(members[rg].begin(), members[rg].end());
                order.insert(order.end(), members[rg].begin(), members[rg].end());
            }
        }
    }
    auto row_at = [&](size_t i) { return !order.empty() ? (size_t)order[i] : rows ? (size_t)rows[i] : i; }; // i-th block row of the plan
    const size_t n_kchunks = (kb + S - 1) / S;
    const int32_t nnzb = row_ptr[mb];
    out = SweepPlanHost();
    out.light = light;
    out.rg_chunk_ptr.assign(n_rg + 1, 0);
    out.op_ptr.reserve(n_rg * WAVES + 1);
    out.row_map.assign(n_rg * G, -1);
    std::vector<int32_t> local(n_kchunks, -1); // K chunk -> position in the row group's chunk list
    struct RowOp { int32_t first, last, hi; SweepOpHost op; }; // the periods it may run in, its later chunk
    std::vector<RowOp> row_ops[G];
    struct Ranked { int rank; int row; int32_t hi; SweepOpHost op; };
    std::vector<std::vector<Ranked>> by_chunk;
    for (size_t rg = 0; rg < n_rg; rg++) {
        const size_t r_begin = rg * GR, r_end = std::min(n_rows, (rg + 1) * GR);
        // the chunks this row group touches, ascending
        const size_t first_chunk = out.chunk_ids.size();
        for (size_t i = r_begin; i < r_end; i++)
            for (int32_t q = row_ptr[row_at(i)]; q < row_ptr[row_at(i) + 1]; q++) local[(size_t)(col_idx[q] / 16) / S] = 0;
        for (size_t c = 0; c < n_kchunks; c++)
            if (local[c] == 0) {
                local[c] = (int32_t)(out.chunk_ids.size() - first_chunk);
                out.chunk_ids.push_back((int32_t)c);
            }
        const size_t n_chunks = out.chunk_ids.size() - first_chunk;
        out.rg_chunk_ptr[rg + 1] = (int32_t)out.chunk_ids.size();

        // ---- ops of every block row: neighbouring blocks in pairs; w3 gets the local row later ----
        for (int lr = 0; lr < G; lr++) {
            row_ops[lr].clear();
            if (r_begin + (size_t)lr >= r_end) continue;
            const size_t br = row_at(r_begin + (size_t)lr);
            int32_t q = row_ptr[br];
            const int32_t q_end = row_ptr[br + 1];
            while (q < q_end) {
                const int32_t bc0 = col_idx[q] / 16;
                const int32_t cl0 = local[(size_t)bc0 / S];
                const uint32_t off0 = sweep_lds_offset(cl0, bc0 % S);
                SweepOpHost op{0, off0, 0, 0};
                int32_t cl_hi = cl0;
                bool pair = false;
                if (q + 1 < q_end) {
                    const int32_t bc1 = col_idx[q + 1] / 16;
                    const int32_t cl1 = local[(size_t)bc1 / S];
                    if (cl1 - cl0 <= 1 + lead) { // three (light streams: two) consecutive listed chunks are resident while one is swept
                        op.w0 = (uint32_t)q * 512u;
                        op.w2 = sweep_lds_offset(cl1, bc1 % S) - off0;
                        cl_hi = cl1;
                        pair = true;
                    }
                }
                if (!pair) {
                    // The other half of the MFMA reads zeros instead of rows of B, but the load brings two
                    // neighbouring blocks: take the neighbour from the SAME block row where the row has one, so that
                    // an Inf or NaN in another row's values (times zero: NaN) cannot reach this row of C.
                    if (q + 1 < q_end) { // blocks (q, q + 1), the second multiplies zeros
                        op.w0 = (uint32_t)q * 512u;
                        op.w2 = SWEEP_ZERO_OFF - off0;
                    } else if (q > row_ptr[br]) { // last block of its row: blocks (q - 1, q), the first multiplies zeros
                        op.w0 = (uint32_t)(q - 1) * 512u;
                        op.w1 = SWEEP_ZERO_OFF;
                        op.w2 = off0 - SWEEP_ZERO_OFF;
                    } else if (q + 1 < nnzb) { // the only block of its row: the neighbour is another row's
                        op.w0 = (uint32_t)q * 512u;
                        op.w2 = SWEEP_ZERO_OFF - off0;
                    } else { // and the last block of the matrix: the read stays inside vals
                        op.w0 = (uint32_t)(q - 1) * 512u;
                        op.w1 = SWEEP_ZERO_OFF;
                        op.w2 = off0 - SWEEP_ZERO_OFF;
                    }
                }
                // While chunk p is swept, chunks p - 1, p and p + 1 are in LDS: the op may run in any period p with
                // p - 1 <= cl0 and cl_hi <= p + 1 (light streams: p - 1 and p, cl_hi <= p).
                const int32_t first = std::max(cl_hi - lead, 0), last = std::min<int32_t>(cl0 + 1, (int32_t)n_chunks - 1);
                (pair ? out.n_pairs : out.n_singles)++;
                row_ops[lr].push_back(RowOp{first, last, cl_hi, op});
                q += pair ? 2 : 1;
            }
        }

        // ---- block rows -> wavefronts, and which period every op runs in.  All wavefronts meet at a barrier once per
        // period, so a period costs the op count of its busiest wavefront, and an op may run in any period of its
        // window [first, last] (at most three periods).  For a given row assignment the cheapest common caps c_p
        // (every wavefront runs at most c_p ops in period p) are found by going through the periods once: a wavefront
        // that runs its pending ops earliest deadline first, as many as the caps allow, is left at period p with the
        // ops that HAVE to run now, and c_p is the largest such count over the wavefronts (capacity is added as late
        // as possible, where it serves the most windows; with unit jobs and interval windows no other caps have a
        // smaller sum).  Pending ops of a wavefront are three counters (deadline p, p + 1, p + 2), so the sum of the
        // caps of an assignment costs O(periods x wavefronts).  The assignment: rows in descending op count to the
        // wavefront with the fewest ops so far, then swaps of two rows between wavefronts while the sum of the caps
        // falls (deterministic, bounded work per row group). ----
        int wave_of[G];
        for (int lr = 0; lr < G; lr++) wave_of[lr] = lr / RW;
        std::vector<int32_t> caps(n_chunks, MIN_OPS);
        if (n_chunks > 0) {
            const size_t n = n_chunks;
            {
                int order[G], n_rows_of[WAVES] = {0};
                long total_of[WAVES] = {0};
                for (int lr = 0; lr < G; lr++) order[lr] = lr;
                std::stable_sort(order, order + G, [&](int x, int y) { return row_ops[x].size() > row_ops[y].size(); });
                for (int k = 0; k < G; k++) {
                    int best = -1;
                    for (int w = 0; w < WAVES; w++)
                        if (n_rows_of[w] < RW && (best < 0 || total_of[w] < total_of[best])) best = w;
                    wave_of[order[k]] = best;
                    n_rows_of[best]++;
                    total_of[best] += (long)row_ops[order[k]].size();
                }
            }
            // ops of row lr with window [first, first + len]: row_win[lr][first * 3 + len]; of wavefront w: win[(first * 3 + len) * WAVES + w]
            std::vector<int16_t> row_win((size_t)G * n * 3, 0), win((size_t)WAVES * n * 3, 0);
            for (int lr = 0; lr < G; lr++) {
                int16_t *rw = &row_win[(size_t)lr * n * 3];
                for (const RowOp &ro : row_ops[lr]) rw[(size_t)ro.first * 3 + (size_t)(ro.last - ro.first)]++;
                for (size_t x = 0; x < n * 3; x++) win[x * WAVES + (size_t)wave_of[lr]] += rw[x];
            }
            long best = sum_of_caps(win.data(), n, nullptr, nullptr, 0, 0, LONG_MAX, nullptr);
            // work bound: so many counter updates per plan, shared evenly by the row groups
            long budget = (long)(search / (double)(n * WAVES * 3) / (double)n_rg);
            for (int pass = 0; pass < 4 && budget > 0; pass++) {
                bool improved = false;
                for (int i = 0; i < G && budget > 0; i++)
                    for (int j = i + 1; j < G && budget > 0; j++) {
                        const int wi = wave_of[i], wj = wave_of[j];
                        if (wi == wj || (row_ops[i].empty() && row_ops[j].empty())) continue;
                        const int16_t *ri = &row_win[(size_t)i * n * 3], *rj = &row_win[(size_t)j * n * 3];
                        const long now = sum_of_caps(win.data(), n, ri, rj, wi, wj, best, nullptr);
                        budget--;
                        if (now < best) {
                            best = now;
                            for (size_t x = 0; x < n * 3; x++) {
                                win[x * WAVES + (size_t)wi] += (int16_t)(rj[x] - ri[x]);
                                win[x * WAVES + (size_t)wj] += (int16_t)(ri[x] - rj[x]);
                            }
                            std::swap(wave_of[i], wave_of[j]);
                            improved = true;
                        }
                    }
                if (!improved) break;
            }
            sum_of_caps(win.data(), n, nullptr, nullptr, 0, 0, LONG_MAX, caps.data());
        }

        // where the rows of C are: also those of a group without a block, which the kernel fills with zeros
        for (int w = 0; w < WAVES; w++)
            for (int lr = 0, r = 0; lr < G; lr++)
                if (wave_of[lr] == w) {
                    if (r_begin + (size_t)lr < r_end) out.row_map[(rg * WAVES + (size_t)w) * RW + (size_t)r] = (int32_t)row_at(r_begin + (size_t)lr);
                    r++;
                }

        struct Pending { int32_t last, first, seq, row, hi; SweepOpHost op; };
        std::vector<std::vector<std::vector<Ranked>>> schedule((size_t)WAVES, std::vector<std::vector<Ranked>>(n_chunks));
        if (n_chunks > 0) {
            for (int w = 0; w < WAVES; w++) {
                std::vector<Pending> todo;
                int r = 0;
                for (int lr = 0; lr < G; lr++) {
                    if (wave_of[lr] != w) continue;
                    for (const RowOp &ro : row_ops[lr]) todo.push_back(Pending{ro.last, ro.first, (int32_t)todo.size(), r, ro.hi, ro.op});
                    r++;
                }
                std::stable_sort(todo.begin(), todo.end(), [](const Pending &a, const Pending &b) { return a.first < b.first; });
                std::vector<Pending> ready;
                size_t next = 0;
                for (size_t c = 0; c < n_chunks; c++) {
                    while (next < todo.size() && todo[next].first <= (int32_t)c) ready.push_back(todo[next++]);
                    std::stable_sort(ready.begin(), ready.end(), [](const Pending &a, const Pending &b) {
                        if (a.last != b.last) return a.last < b.last;
                        return a.seq < b.seq;
                    });
                    // Up to the cap, earliest deadline first.  The op that opens the next period has to be one that is
                    // ready now (its LDS reads are issued before the boundary's barrier, so its chunks must be resident
                    // already): a wavefront that could run everything it has keeps its last op for that.
                    size_t musts = 0;
                    while (musts < ready.size() && ready[musts].last <= (int32_t)c) musts++;
                    size_t k = std::min(ready.size(), (size_t)caps[c]);
                    if (k == ready.size() && k > musts && c + 1 < n_chunks) k--;
                    k = std::max(k, musts);
                    std::vector<Ranked> &list = schedule[(size_t)w][c];
                    for (size_t x = 0; x < k; x++) {
                        const Pending &pe = ready[x];
                        // rank = how many ops of this block row the period already holds: ops of one block
                        // row (same accumulators) end up spread over the period
                        int rank = 0;
                        for (const Ranked &y : list) rank += y.row == pe.row;
                        list.push_back(Ranked{rank, pe.row, pe.hi, pe.op});
                    }
                    ready.erase(ready.begin(), ready.begin() + (long)k);
                    if (!ready.empty() && ready.front().last <= (int32_t)c) throw std::logic_error("sweep plan: an op missed its last period");
                }
                if (!ready.empty() || next != todo.size()) throw std::logic_error("sweep plan: ops left over by the period schedule");
            }
        }

        // ---- streams: ops of chunk 0, ops of chunk 1, ..., end; the first op of a chunk carries the chunk boundary ----
        for (int w = 0; w < WAVES; w++) {
            out.op_ptr.push_back((int32_t)out.ops.size());
            if (n_chunks == 0) continue; // the kernel does not enter the interpreter for an empty row group
            by_chunk = schedule[(size_t)w];
            struct Item { int kind, row; bool opens; SweepOpHost op; }; // kind: 0 op, 2 end; opens: first op of a chunk but the first
            std::vector<Item> items;
            const SweepOpHost idle{0, SWEEP_ZERO_OFF, 0, 0}; // the end: no blocks of its own
            // A filler op multiplies two blocks by zeros and adds the result to one of the wavefront's block rows:
            // two blocks of that very row (then an Inf or NaN in them is in that row of C anyway), blocks 0 and 1
            // of the matrix only when no row of the wavefront has two.
            Item filler{0, 0, false, idle};
            for (int r = 0; r < RW; r++) {
                const int32_t br = out.row_map[(rg * WAVES + (size_t)w) * RW + (size_t)r];
                if (br >= 0 && row_ptr[br + 1] - row_ptr[br] >= 2) {
                    filler.row = r;
                    filler.op.w0 = (uint32_t)row_ptr[br] * 512u;
                    break;
                }
            }
            for (size_t c = 0; c < n_chunks; c++) {
                std::vector<Ranked> &list = by_chunk[c];
                std::stable_sort(list.begin(), list.end(), [](const Ranked &a, const Ranked &b) {
                    if (a.rank != b.rank) return a.rank < b.rank;
                    return a.row < b.row;
                });
                const size_t first_of_chunk = items.size();
                size_t n_here = list.size();
                if (c > 0) {
                    // The LDS reads of the op that opens a chunk are issued by the op before it, before the barrier of
                    // the boundary, when the copies of chunk c + 1 may still be under way: it has to be an op whose
                    // chunks are c or c - 1 (light streams: when those of chunk c may be, an op of chunk c - 1).
                    size_t ok = 0;
                    while (ok < list.size() && list[ok].hi > (int32_t)c - 1 + lead) ok++;
                    if (ok == list.size()) {
                        items.push_back(filler);
                        out.n_fillers++;
                        n_here++;
                    } else if (ok > 0) {
                        std::rotate(list.begin(), list.begin() + (long)ok, list.begin() + (long)ok + 1);
                    }
                }
                for (const Ranked &x : list) items.push_back(Item{0, x.row, false, x.op});
                for (size_t k = n_here; k < (size_t)MIN_OPS; k++) { // filler ops keep the chunk boundaries AHEAD positions apart
                    items.push_back(filler);
                    out.n_fillers++;
                }
                if (c > 0) items[first_of_chunk].opens = true;
            }
            items.push_back(Item{2, 0, false, idle});
            // Which s_waitcnt vmcnt an op needs: vector memory operations complete in order, every position issues
            // one A load (for the op AHEAD positions later), the op that opens a chunk issues the copies of the
            // boundary before that load.
            std::vector<long> a_issue(items.size() + (size_t)AHEAD + 1, 0), copy_seq(n_chunks + 3, 0);
            long seq = 0;
            for (int k = 0; k < AHEAD; k++) a_issue[(size_t)k] = ++seq; // entry code, after the copies of chunks 0..2
            size_t cur = 0;
            for (size_t i = 0; i < items.size(); i++) {
                Item &it = items[i];
                if (it.kind == 2) {
                    it.op.w3 = SWEEP_END_OFF;
                    break;
                }
                if (it.opens) {
                    cur++;
                    // the copies of chunk cur + 1 were issued by the boundary before this one (or by the entry code): the
                    // boundary waits until at most VM_MARK younger operations are under way
                    if (cur + 1 < n_chunks && seq - copy_seq[cur + 1] < VM_MARK) throw std::logic_error("sweep plan: a chunk boundary would not wait for its copies");
                    if (cur + 2 < n_chunks) {
                        seq += COPIES;
                        copy_seq[cur + 2] = seq;
                    }
                }
                a_issue[i + (size_t)AHEAD] = ++seq;
                const long younger = seq - a_issue[i];
                if (younger != AHEAD && younger != AHEAD + COPIES) throw std::logic_error("sweep plan: chunk boundaries closer than the A read-ahead");
                const int v = younger == AHEAD ? 0 : 1;
                it.op.w3 = it.opens ? sweep_boundary_op_code((int)i, it.row, v) : sweep_op_code((int)i, it.row, v);
            }
            if (cur + 1 != n_chunks) throw std::logic_error("sweep plan: a stream does not pass every chunk boundary");
            for (const Item &it : items) out.ops.push_back(it.op);
        }
        for (size_t c = first_chunk; c < out.chunk_ids.size(); c++) local[(size_t)out.chunk_ids[c]] = -1;
    }
    out.op_ptr.push_back((int32_t)out.ops.size());
    // what the kernel reads ahead of the last op: fetched, never executed
    out.ops.resize(out.ops.size() + SWEEP_OP_PAD, SweepOpHost{0, SWEEP_ZERO_OFF, 0, SWEEP_END_OFF});
    out.chunk_ids.resize(out.chunk_ids.size() + SWEEP_CHUNK_PAD, 0);
}

void encode_sweep_streams(const std::vector<int32_t> &rg_chunk_ptr, const std::vector<int32_t> &op_ptr, const SweepOpHost *ops,
                          bool b_row_major, std::vector<SweepOpHost> &dev, bool light)
{
    const uint32_t block_bytes = sweep_block_bytes(b_row_major), tramp_base = sweep_tramp_base(b_row_major), light_base = sweep_light_base(b_row_major);
    constexpr int DEV_AHEAD = SWEEP_DEV_AHEAD, DEV_MIN = SWEEP_DEV_MIN_OPS, HEAD = SWEEP_DEV_HEAD;
    const size_t n_streams = op_ptr.size() - 1;
    dev.assign((size_t)op_ptr.back() + HEAD * n_streams + SWEEP_OP_PAD, SweepOpHost{0, SWEEP_ZERO_OFF, 0, sweep_end_off(b_row_major)});
    struct Op { SweepOpHost op; uint32_t row; bool opens; };
    std::vector<Op> kept;
    std::vector<long> a_issue;
    for (size_t s = 0; s < n_streams; s++) {
        const SweepOpHost *op = ops + op_ptr[s];
        SweepOpHost *out = dev.data() + op_ptr[s] + HEAD * s;
        const size_t len = (size_t)(op_ptr[s + 1] - op_ptr[s]), n_plan = len ? len - 1 : 0; // the end is no op
        const long n_chunks = rg_chunk_ptr[s / WAVES + 1] - rg_chunk_ptr[s / WAVES];
        // the fillers of the plan keep chunks at MIN_OPS ops: those past DEV_MIN go, but not the one that opens a chunk, which
        // stands there because no other op may
        kept.clear();
        for (size_t i = 0; i < n_plan;) {
            size_t end = i + 1;
            while (end < n_plan && op[end].w3 < SWEEP_TRAMP_BASE) end++;
            long work = 0, taken = 0;
            auto filler = [&](size_t k) { return op[k].w1 == SWEEP_ZERO_OFF && op[k].w2 == 0; };
            for (size_t k = i; k < end; k++) work += k == i || !filler(k);
            long fill = DEV_MIN - work;
            for (size_t k = i; k < end; k++) {
                if (k > i && filler(k) && fill-- <= 0) continue;
                const bool opens = op[k].w3 >= SWEEP_TRAMP_BASE;
                const uint32_t block = opens ? (op[k].w3 - SWEEP_TRAMP_BASE) / SWEEP_TRAMP_BYTES : op[k].w3 / SWEEP_BLOCK_BYTES;
                kept.push_back(Op{op[k], block / 2 % 8, opens});
                taken++;
            }
            if (taken < DEV_MIN) throw std::logic_error("sweep plan: chunk boundaries closer than the copies' wait allows");
            i = end;
        }
        const size_t n_ops = kept.size();
        auto a_offset = [&](size_t i) { return i < n_ops ? kept[i].op.w0 : 0u; };
        uint32_t head[4 * HEAD] = {0};
        for (int k = 0; k < DEV_AHEAD; k++) head[k] = a_offset((size_t)k);
        memcpy(out, head, sizeof head);
        out += HEAD;
        // vector memory operations in issue order: what is younger than the load of an op's A operand when the op needs it
        a_issue.assign(n_ops + DEV_AHEAD + 1, 0);
        long seq = 0, cur = 0, in_chunk = 0, in_chunk_before = 0;
        bool copies_before = false; // by the boundary before
        for (int k = 0; k < DEV_AHEAD; k++) a_issue[(size_t)k] = ++seq;
        for (size_t i = 0; i < n_ops; i++) {
            const bool opens = kept[i].opens;
            uint32_t tramp = tramp_base;
            if (opens) {
                const long loads = std::min<long>(in_chunk + (light ? in_chunk_before : 0), DEV_AHEAD);
                // (cur = 0: no boundary before this one, and no two chunks)
                tramp = light && copies_before ? light_base + (uint32_t)(loads - 2 * DEV_MIN) * SWEEP_N_BLOCKS * SWEEP_TRAMP_BYTES
                                               : tramp_base + (uint32_t)(loads - DEV_MIN) * SWEEP_N_BLOCKS * SWEEP_TRAMP_BYTES;
                in_chunk_before = in_chunk;
                in_chunk = 0;
                copies_before = ++cur + 2 < n_chunks;
                if (copies_before) seq += COPIES;
            }
            in_chunk++;
            a_issue[i + DEV_AHEAD] = ++seq;
            const uint32_t code = (uint32_t)((i % 8 * 8 + kept[i].row) * 2) + (seq - a_issue[i] > DEV_AHEAD ? 1u : 0u);
            const uint32_t lo = kept[i].op.w1, hi = lo + kept[i].op.w2;
            out[i].w0 = a_offset(i + DEV_AHEAD - 1);
            out[i].w1 = b_row_major ? sweep_lds_offset_row_major(lo) : lo;
            out[i].w2 = (b_row_major ? sweep_lds_offset_row_major(hi) : hi) - out[i].w1;
            out[i].w3 = opens ? tramp + code * SWEEP_TRAMP_BYTES : code * block_bytes;
        }
        // the end, and what the dropped fillers leave behind it, stay what dev was filled with
    }
}

} // namespace smat

// Test hook (not part of smat.h): the streams of a plan that smat_internal_sweep_plan handed out as the kernel runs them (b_row_major + 2: of a light plan), in
// out[0 .. op_ptr[8 n_rg] + 2 * 8 n_rg + 16).
extern "C" int smat_internal_sweep_encode(const int32_t *rg_chunk_ptr, int64_t n_rg, const int32_t *op_ptr, const uint32_t *ops, int b_row_major, uint32_t *out)
{
    return smat::guarded("smat_internal_sweep_encode", [&] {
        const std::vector<int32_t> chunk_ptr(rg_chunk_ptr, rg_chunk_ptr + n_rg + 1), ptr(op_ptr, op_ptr + n_rg * smat::SWEEP_WAVES + 1);
        std::vector<smat::SweepOpHost> dev;
        smat::encode_sweep_streams(chunk_ptr, ptr, reinterpret_cast<const smat::SweepOpHost *>(ops), (b_row_major & 1) != 0, dev, (b_row_major & 2) != 0);
        memcpy(out, dev.data(), dev.size() * sizeof(smat::SweepOpHost));
        return (int)SMAT_OK;
    });
}

// Test hook (not part of smat.h): builds the work list on the host (rows != NULL: of these block rows only) and hands it out.  Arrays are
// allocated with malloc; release each with smat_host_free.  row_map: n_rg * 64 block rows (-1 = none).  counts[0..5] = row groups, listed
// chunks, stream entries (ops, fillers, ends; without padding), pairs, singles, fillers.
static int smat_internal_sweep_plan_impl(const int32_t *row_ptr, const int32_t *col_idx, size_t M, size_t K,
                                         const int32_t *rows, size_t n_rows, size_t group_rows, bool light, int32_t **rg_chunk_ptr, int32_t **chunk_ids, int32_t **op_ptr,
                                         uint32_t **ops, int32_t **row_map, int64_t *counts)
{
    if (!row_ptr || !col_idx || !rg_chunk_ptr || !chunk_ids || !op_ptr || !ops || !row_map || !counts) return SMAT_ERR_INVALID;
    if (M == 0 || M % 16 || K % 16 || row_ptr[M / 16] < 2) return SMAT_ERR_INVALID;
    smat::SweepPlanHost p;
    try {
        smat::build_sweep_plan(row_ptr, col_idx, M / 16, K / 16, p, rows, n_rows, group_rows, 2e8, light);
    } catch (...) {
        return SMAT_ERR_NOMEM;
    }
    auto dup = [](const void *src, size_t bytes) -> void * {
        void *d = malloc(bytes ? bytes : 1);
        if (d && bytes) memcpy(d, src, bytes);
        return d;
    };
    *rg_chunk_ptr = (int32_t *)dup(p.rg_chunk_ptr.data(), p.rg_chunk_ptr.size() * 4);
    *chunk_ids = (int32_t *)dup(p.chunk_ids.data(), p.chunk_ids.size() * 4);
    *op_ptr = (int32_t *)dup(p.op_ptr.data(), p.op_ptr.size() * 4);
    *ops = (uint32_t *)dup(p.ops.data(), p.ops.size() * 16);
    *row_map = (int32_t *)dup(p.row_map.data(), p.row_map.size() * 4);
    if (!*rg_chunk_ptr || !*chunk_ids || !*op_ptr || !*ops || !*row_map) return SMAT_ERR_NOMEM;
    counts[0] = (int64_t)p.rg_chunk_ptr.size() - 1;
    counts[1] = (int64_t)p.chunk_ids.size() - smat::SWEEP_CHUNK_PAD;
    counts[2] = (int64_t)p.ops.size() - smat::SWEEP_OP_PAD;
    counts[3] = (int64_t)p.n_pairs;
    counts[4] = (int64_t)p.n_singles;
    counts[5] = (int64_t)p.n_fillers;
    return SMAT_OK;
}

// Test hook: the pipeline depths this build was compiled with {A read-ahead, LDS read-ahead, minimum ops per chunk, copies per chunk boundary}.
extern "C" void smat_internal_sweep_params(int32_t *out)
{
    out[0] = smat::SWEEP_AHEAD; out[1] = smat::SWEEP_LDS_AHEAD; out[2] = smat::SWEEP_MIN_OPS; out[3] = smat::SWEEP_COPIES;
}

extern "C" int smat_internal_sweep_plan(const int32_t *row_ptr, const int32_t *col_idx, size_t M, size_t K,
                                         const int32_t *rows, size_t n_rows, int32_t **rg_chunk_ptr, int32_t **chunk_ids, int32_t **op_ptr,
                                         uint32_t **ops, int32_t **row_map, int64_t *counts)
{
    return smat::guarded("smat_internal_sweep_plan", [&] {
        return smat_internal_sweep_plan_impl(row_ptr, col_idx, M, K, rows, n_rows, smat::SWEEP_G, false, rg_chunk_ptr, chunk_ids, op_ptr, ops, row_map, counts);
    });
}
// The same on row groups of group_rows (at most 64) block rows.
extern "C" int smat_internal_sweep_plan_groups(const int32_t *row_ptr, const int32_t *col_idx, size_t M, size_t K, size_t group_rows,
                                               int32_t **rg_chunk_ptr, int32_t **chunk_ids, int32_t **op_ptr, uint32_t **ops,
                                               int32_t **row_map, int64_t *counts)
{
    return smat::guarded("smat_internal_sweep_plan_groups", [&] {
        return smat_internal_sweep_plan_impl(row_ptr, col_idx, M, K, nullptr, 0, group_rows, false, rg_chunk_ptr, chunk_ids, op_ptr, ops, row_map, counts);
    });
}
// The same for light streams.
extern "C" int smat_internal_sweep_plan_light(const int32_t *row_ptr, const int32_t *col_idx, size_t M, size_t K, size_t group_rows,
                                              int32_t **rg_chunk_ptr, int32_t **chunk_ids, int32_t **op_ptr, uint32_t **ops,
                                              int32_t **row_map, int64_t *counts)
{
    return smat::guarded("smat_internal_sweep_plan_light", [&] {
        return smat_internal_sweep_plan_impl(row_ptr, col_idx, M, K, nullptr, 0, group_rows, true, rg_chunk_ptr, chunk_ids, op_ptr, ops, row_map, counts);
    });
}
