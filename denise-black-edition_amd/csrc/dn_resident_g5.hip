// Chip-resident time loop, FDORDER 10, acoustic, VTI, TTI and SH.
#define DN_F 5
#define DN_GROUP 1
#include "dn_resident_inst.inc"
