// Launch shapes and frontier chunk sizes of the persistent label kernels. brook_amd/tune.py rewrites
// this file with the values it measures fastest on the device it runs on (a -D on the compiler
// line still overrides each one). Every value gives bit-identical results; only speed changes.
// Words in flight and threads against other values, whole calls in ms (512^3 trees, a 31 M voxel request, a
// 48-voxel crop, 300^3 trees by parent walks), each pair timed in turn:
//   BROOK_NB_BATCH 9 against 13        87.3 89.4   22.8 23.3   5.87 6.21   38.6 40.1
//                    against 26        85.6 96.6   19.7 23.3   6.48 7.98   38.8 45.3
//   BROOK_TRACE_BLOCK 1024 against 512 86.1 90.9   20.8 24.1   6.54 7.30   38.2 44.3
//   BROOK_FLOOD_NB_BATCH 9 against 13  87.0 87.3   19.3 19.4   6.39 6.38   37.4 37.4
//                          against 26  91.3 90.8   19.5 19.9   6.07 6.14   38.0 37.8
//   BROOK_FLOOD_BLOCK 1024 against 512 86.8 89.8   19.9 20.5   6.36 6.53   37.8 39.5
#pragma once
#ifndef BROOK_TRACE_BLOCK
#define BROOK_TRACE_BLOCK 1024  // threads per trace_labels workgroup (one label at a time)
#endif
#ifndef BROOK_NB_BATCH
#define BROOK_NB_BATCH 9  // neighbour words a trace lane keeps in flight in a long front (9, 13 or 26)
#endif
#ifndef BROOK_FLOOD_BLOCK
#define BROOK_FLOOD_BLOCK 1024  // threads per prepare_labels workgroup
#endif
#ifndef BROOK_FLOOD_NB_BATCH
#define BROOK_FLOOD_NB_BATCH 9  // neighbour words a flood lane keeps in flight in a long front (9, 13 or 26)
#endif
#ifndef BROOK_TRACE_GRID
#define BROOK_TRACE_GRID 0  // trace_labels workgroups resident at once (0: two per compute unit)
#endif
#ifndef BROOK_FLOOD_GRID
#define BROOK_FLOOD_GRID 0  // prepare_labels workgroups resident at once (0: two per compute unit)
#endif
