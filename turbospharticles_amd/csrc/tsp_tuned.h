// tsp_tuned.h -- build-time variant chosen by turbospharticles_amd/tune.py on MI355X
// (1M rigid cube drop: 3.662 ms per step; every candidate checked bit-identical). The halo cap
// 1064, lane sorting and u16 halo slots were then chosen on the window and the whole 500-step drop
// (the late steps of the drop have 5-12% of blocks with more than 1000 distinct FF neighbors).
#ifndef TSP_TUNE_GRAPHS
#define TSP_TUNE_GRAPHS 1
#endif
#ifndef TSP_TUNE_HALO_MAX
#define TSP_TUNE_HALO_MAX 1064
#endif
#ifndef TSP_TUNE_JACOBI_WAVES
#define TSP_TUNE_JACOBI_WAVES 6
#endif
#ifndef TSP_TUNE_PA_WAVES
#define TSP_TUNE_PA_WAVES 6
#endif
#ifndef TSP_TUNE_STEP_GRAPH
#define TSP_TUNE_STEP_GRAPH 0
#endif
#ifndef TSP_TUNE_SWEEP_AHEAD
#define TSP_TUNE_SWEEP_AHEAD 2
#endif
